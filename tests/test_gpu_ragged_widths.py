"""Feature widths and rows off every vector boundary: rows are read with whole vectors whatever their
alignment, the last lane of a row taking its last VEC features, and the staged hot rows of such widths
are padded.  Every operand is a view inside a wider buffer whose other elements are NaN, so a read past
a row's end shows in the result, and outputs are views whose surroundings must stay as they were."""
import numpy as np
import pytest
import torch

from oracle import spmm as osp
from trspmm import _native as nat
from trspmm import graphs
import trspmm

pytestmark = pytest.mark.gpu

_cache = {}


def graph(name):
    if name not in _cache:
        g = graphs.rmat(scale=12, edge_factor=16, seed=12) if name == "rmat" else graphs.sbm(communities=64, seed=5, val_seed=6)
        _cache[name] = (g, trspmm.build_format(g.rowptr, g.col, g.val))
    return _cache[name]


def inside(rows, K, off, pad, seed):
    """fp16 [rows, K] view starting `off` elements into a NaN buffer, `pad` NaNs after each row."""
    buf = torch.full((off + rows * (K + pad),), float("nan"), dtype=torch.float16, device="cuda")
    v = buf[off:].view(rows, K + pad)[:, :K]
    h = graphs.dense_operand(rows, K, seed)
    v.copy_(torch.from_numpy(h).cuda())
    return v, h


# edges of every load width (2 | 4 | 8 | 16 bytes), of the 4-, 8- and 16-lane groups, of the widths that
# stage hot rows, and of a second feature pass
WIDTHS = [4, 5, 7, 8, 9, 13, 16, 17, 23, 31, 33, 40, 47, 63, 65, 72, 96, 103, 104, 106, 119, 121, 127, 129, 130, 135, 136,
          200, 255]


@pytest.mark.parametrize("K", WIDTHS)
@pytest.mark.parametrize("off,pad", [(1, 0), (3, 2), (0, 1)])
def test_spmm_any_width_and_alignment(K, off, pad):
    print("ragged spmm", K, off, pad, flush=True)
    for name, opts in (("rmat", dict(piece_nnz=64, xcd_split=64, hot_rows=64)), ("sbm", {}), ("sbm", dict(mfma_tc=False, mfma_sptc=False))):
        g, f = graph(name)
        plan = trspmm.Plan.from_format(f, g.m, g.n, **opts)
        B, Bh = inside(g.n, K, off, pad, seed=K)
        full = torch.full((g.m, K + 3), 7.0, device="cuda")
        out = full[:, 1: 1 + K]
        plan.spmm(B, out=out)
        torch.cuda.synchronize()
        C, R = out.cpu().numpy(), osp.csr_spmm(g.rowptr, g.col, g.val, Bh, m=g.m)
        # 32-bit sums of fp16 products (exact in fp32): |error| <= entries * 2^-24 * sum |a b|, rows of
        # at most 4096 entries with |a|, |b| <= 1; the sums' own spread makes it far smaller
        assert np.max(np.abs(C - R)) <= 1e-5 * max(1.0, float(np.max(np.abs(R)))), (name, K)
        assert torch.all(full[:, :1] == 7.0) and torch.all(full[:, 1 + K:] == 7.0), (name, K)


@pytest.mark.parametrize("K", WIDTHS)
@pytest.mark.parametrize("off,pad", [(1, 0), (2, 3)])
def test_sddmm_any_width_and_alignment(K, off, pad):
    print("ragged sddmm", K, off, pad, flush=True)
    for name, opts in (("rmat", dict(piece_nnz=64, xcd_split=64, hot_rows=64)), ("sbm", {})):
        g, f = graph(name)
        plan = trspmm.Plan.for_sddmm(f, g.m, g.n, **opts)
        X, Xh = inside(g.m, K, off, pad, seed=K)
        Y, Yh = inside(g.n, K, off + 1, pad, seed=K + 1)
        # an Inf in one X row and one Y row: only their own entries are not finite, and they are +-Inf.  (In Y
        # among the features that lanes past K read, to no effect.)
        X[5, K - 1] = float("inf")
        Y[9, 0] = float("inf")
        Xh, Yh = X.cpu().numpy(), Y.cpu().numpy()
        S = plan.sddmm(X, Y)
        torch.cuda.synchronize()
        with np.errstate(invalid="ignore", over="ignore"):
            R = osp.csr_sddmm(g.rowptr[: g.m + 1], g.col, Xh, Yh)
        S = S.cpu().numpy()
        fin = np.isfinite(R)
        assert np.array_equal(fin, np.isfinite(S)), (name, K)
        assert np.array_equal(np.isnan(R), np.isnan(S)) and np.array_equal(R[~fin & ~np.isnan(R)], S[~fin & ~np.isnan(R)])
        tol = (1e-5 * np.sqrt(K) * 4 + 1e-6) * max(1.0, float(np.max(np.abs(R[fin]))))
        assert np.max(np.abs(S[fin] - R[fin])) <= tol, (name, K)


@pytest.mark.parametrize("K", [65, 106, 127, 130, 255])
def test_ragged_staging_is_optional_and_changes_nothing(K):
    """The staged rows of a ragged width are used where the workspace has room for them and left out where it
    only holds the partial slots: the same bits."""
    print("ragged staging", K, flush=True)
    g, f = graph("rmat")
    plan = trspmm.Plan.from_format(f, g.m, g.n, xcd_split=64, hot_rows=64)
    plain = trspmm.Plan.from_format(f, g.m, g.n, xcd_split=64, hot_rows=-1)
    need, least = plan.workspace_bytes(K), plain.workspace_bytes(K)
    stride = (K + 63) // 64 * 64
    assert need == (least + 255) // 256 * 256 + 64 * stride * 2 and least > 0
    B = torch.from_numpy(graphs.dense_operand(g.n, K, K)).cuda()
    want = plan.spmm(B)
    assert torch.equal(want, plain.spmm(B))
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    out = torch.full((g.m, K), float("nan"), device="cuda")
    s = int(torch.cuda.current_stream().cuda_stream)
    call = lambda nbytes: nat.lib().trs_spmm_f16(plan.handle, B.data_ptr(), K, K, out.data_ptr(), K, ws.data_ptr(), nbytes, s)
    assert call(least) == 0
    assert torch.equal(out, want)
    assert call(least - 1) == 1 and b"workspace" in nat.lib().trs_last_error()
    out.fill_(float("nan"))
    nat.check(nat.lib().trs_spmm_f16_noalloc(plan.handle, B.data_ptr(), K, K, out.data_ptr(), K, s), "trs_spmm_f16_noalloc")
    torch.cuda.synchronize()
    assert torch.equal(out, want)
    # SDDMM: staged, unstaged plan, no workspace
    ph = trspmm.Plan.for_sddmm(f, g.m, g.n, xcd_split=64, hot_rows=64)
    pp = trspmm.Plan.for_sddmm(f, g.m, g.n, xcd_split=64, hot_rows=-1)
    X = torch.from_numpy(graphs.dense_operand(g.m, K, K + 1)).cuda()
    S = ph.sddmm(X, B)
    assert torch.equal(S, pp.sddmm(X, B))
    S2 = torch.empty_like(S)
    nat.check(nat.lib().trs_sddmm_f16(ph.handle, X.data_ptr(), K, B.data_ptr(), K, K, S2.data_ptr(), s), "trs_sddmm_f16")
    torch.cuda.synchronize()
    assert torch.equal(S, S2)
