"""MFMA windows of a plan by what their tiles hold: dropped where that is less than a sixteenth of the entries and less
than 262,144 of them, on the host's and the device's lowering, and window by window where residual rows are long."""
import numpy as np
import pytest
import torch

from oracle import spmm as osp
from trspmm import graphs
import trspmm

pytestmark = pytest.mark.gpu


def blocks(windows, rows, per_row, last, seed, long_windows=0, extra=0):
    """`windows` windows with a full 16 x 16 block (256 tile entries each; the first `long_windows` also `extra` random
    entries in every row), then `rows` rows of `per_row` random entries (the last one `last`)."""
    rng = np.random.default_rng(seed)
    n = 400_000
    first = 16 * windows
    cols = []
    for w in range(windows):
        block = np.arange(16 * w, 16 * w + 16)
        for _ in range(16):
            more = first + rng.choice((n - first) // 64, extra, replace=False) * 64 if w < long_windows else block[:0]
            cols.append(np.sort(np.concatenate([block, more])))
    step = (n - first) // per_row if per_row else 1
    for r in range(rows):
        k = last if r == rows - 1 else per_row
        # distinct columns in row order, another phase in each row: no column is shared in a window
        cols.append(first + np.arange(k) * step + (r * 7919) % step)
    count = np.array([len(c) for c in cols])
    m = (len(cols) + 15) // 16 * 16
    rowptr = np.zeros(m + 1, np.int32)
    rowptr[1: len(cols) + 1] = np.cumsum(count)
    rowptr[len(cols) + 1:] = rowptr[len(cols)]
    col = np.concatenate(cols).astype(np.int32)
    val = rng.uniform(-1, 1, len(col)).astype(np.float16).astype(np.float32)
    return m, n, rowptr, col, val


def plans(m, n, rowptr, col, val, **opts):
    f = trspmm.build_format(rowptr, col, val)
    return [trspmm.Plan.from_format(f, m, n, host_lowering=h, **opts) for h in (False, True)]


@pytest.mark.parametrize("extra", [0, 1])
def test_share_of_a_sixteenth(extra):
    """64 blocks hold 16,384 entries: of 262,144 in all they stay, of 262,145 they go; an explicit window_row_cap
    keeps them."""
    print("window share", extra, flush=True)
    M = blocks(64, 3841, 64, extra, seed=1)
    assert M[2][-1] == 262_144 + extra
    Bh = graphs.dense_operand(M[1], 64, seed=2)
    R = osp.csr_spmm(M[2], M[3], M[4], Bh, m=M[0])
    for opts, kept in (({}, extra == 0), (dict(window_row_cap=128), True)):
        for p in plans(*M, **opts):
            s = p.stats()
            assert s["mfma_windows"] == (64 if kept else 0) and s["mfma_nnz"] + s["csr_nnz"] == M[2][-1], (opts, s)
            C = p.spmm(torch.from_numpy(Bh).cuda()).cpu().numpy()
            # rows of at most 64 products of fp16 values <= 1, 32-bit sums
            assert np.max(np.abs(C - R)) <= 1e-5 * max(1.0, float(np.max(np.abs(R))))


@pytest.mark.parametrize("windows", [1023, 1024])
def test_enough_tile_entries_stay_whatever_their_share(windows):
    print("windows", windows, flush=True)
    m, n, rowptr, col, val = blocks(windows, 65_536, 64, 64, seed=3)
    assert windows * 256 * 16 < rowptr[-1]
    f = trspmm.build_format_device(*(torch.from_numpy(a).cuda() for a in (rowptr, col, val)))
    assert trspmm.Plan.from_format(f, m, n).stats()["mfma_windows"] == (windows if windows == 1024 else 0)


def test_windows_of_long_rows_go_and_the_others_stay():
    """64 windows whose rows all carry 700 residual entries (more than 4 x 128) beside 256 of blocks alone."""
    print("long windows", flush=True)
    M = blocks(320, 0, 0, 0, seed=4, long_windows=64, extra=700)
    for p in plans(*M):
        assert p.stats()["mfma_windows"] == 256, p.stats()
    for p in plans(*M, window_row_cap=1 << 30):
        assert p.stats()["mfma_windows"] == 320, p.stats()
