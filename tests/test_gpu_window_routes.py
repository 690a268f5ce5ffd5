"""GPU format builder: windows at the edges of its routing rule (1024, 2048 and 8192 distinct columns; 9/8
entries a column), bit for bit against the host builder."""
import numpy as np
import pytest
import torch

from conftest import same_array
import trspmm

pytestmark = pytest.mark.gpu


def _window(U, extra, rng, n):
    """16 rows over U distinct columns of n: two rows share them out, a third repeats `extra` of them."""
    cols = np.sort(rng.choice(n, size=U, replace=False))
    first = rng.random(U) < 0.5
    return [cols[first], cols[~first], np.sort(rng.choice(cols, size=extra, replace=False))] + [cols[:0]] * 13


def _check(rows, rng):
    rowptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    col = np.concatenate(rows).astype(np.int32)
    val = rng.integers(1, 16, size=len(col)).astype(np.float32)
    hf = trspmm.build_format(rowptr, col, val)
    f = trspmm.build_format_device(*(torch.from_numpy(a).cuda() for a in (rowptr, col, val))).download()
    bad = [trspmm.ops.SLOT_NAMES[i] for i in range(32) if not same_array(f.slot(i), hf.slot(i))]
    assert not bad, bad


@pytest.mark.parametrize("U", [1024, 1025, 2048, 2049, 3001, 8192, 8193])
def test_windows_at_the_routing_edges(U):
    rng = np.random.default_rng(U)
    n = 20000
    rows = []
    for extra in (0, (U - 1) // 8, U // 8 + 1, U):   # below, just below, just above 9/8 entries a column; 2
        print("window of", U, "columns", U + extra, "entries", flush=True)
        rows += _window(U, extra, rng, n)
    _check(rows, rng)


@pytest.mark.parametrize("windows", [128, 129])
def test_few_and_many_wide_windows(windows):
    """Up to 128 windows of more than 1024 columns share one launch with those of more than 2048."""
    print("windows past 1024 columns:", windows, flush=True)
    rng = np.random.default_rng(windows)
    rows = _window(2049, 0, rng, 20000) + _window(100, 20, rng, 20000)
    for _ in range(windows - 1):
        rows += _window(1025, 0, rng, 20000)
    _check(rows, rng)
