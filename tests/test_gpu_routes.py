"""Plans whose rows choose the route of a width (spmm_route, sddmm_route in csrc/kernels.hpp): even rows, short rows,
a mesh with a few long rows.  Operands and outputs lie inside NaN or marked buffers, so that a read or write past a row's
end shows."""
import numpy as np
import pytest
import torch

from oracle import spmm as osp
from trspmm import graphs
import trspmm

pytestmark = pytest.mark.gpu

GRAPHS = {
    # even rows of 17 entries, more than 786,432 of them
    "even": lambda: graphs.erdos_renyi_gcn(nodes=60_000, edges=480_000, seed=1),
    # even and short: 9 entries a row
    "short": lambda: graphs.erdos_renyi_gcn(nodes=90_000, edges=360_000, seed=2),
    # even, few entries
    "even_small": lambda: graphs.erdos_renyi_gcn(nodes=6_000, edges=48_000, seed=3),
    # a mesh with long rows: below and from 262,144 entries, and from 786,432 on
    "mesh_small": lambda: graphs.grid_hubs(side=100, hubs=8, hub_degree=900, seed=4, val_seed=4),
    "mesh": lambda: graphs.grid_hubs(side=250, hubs=16, hub_degree=3000, seed=5, val_seed=5),
    "mesh_large": lambda: graphs.grid_hubs(side=400, hubs=16, hub_degree=12_000, seed=6, val_seed=6),
    # power law, few entries
    "rmat_tiny": lambda: graphs.rmat(scale=13, edge_factor=8, seed=7),
}
WIDTHS = [5, 9, 15, 16, 17, 24, 31, 32, 36, 41, 48, 64, 100, 124, 132, 180, 252, 300]
_cache = {}


def graph(name):
    if name not in _cache:
        _cache.clear()
        g = GRAPHS[name]()
        _cache[name] = (g, trspmm.build_format_device(*(torch.from_numpy(a).cuda() for a in (g.rowptr, g.col, g.val))))
    return _cache[name]


def inside(rows, K, off, pad, seed):
    buf = torch.full((off + rows * (K + pad),), float("nan"), dtype=torch.float16, device="cuda")
    v = buf[off:].view(rows, K + pad)[:, :K]
    h = graphs.dense_operand(rows, K, seed)
    v.copy_(torch.from_numpy(h).cuda())
    return v, h


@pytest.mark.parametrize("off,pad", [(0, 0), (1, 1)])
@pytest.mark.parametrize("name", list(GRAPHS))
def test_spmm_routes(name, off, pad):
    g, f = graph(name)
    plan = trspmm.Plan.from_format(f, g.m, g.n)
    for K in WIDTHS:
        print("spmm route", name, K, off, pad, flush=True)
        B, Bh = inside(g.n, K, off, pad, seed=K)
        full = torch.full((g.m, K + 3), 7.0, device="cuda")
        out = full[:, 1: 1 + K]
        plan.spmm(B, out=out)
        torch.cuda.synchronize()
        C, R = out.cpu().numpy(), osp.csr_spmm(g.rowptr, g.col, g.val, Bh, m=g.m)
        # 32-bit sums of fp16 products (exact in fp32), |a|, |b| <= 1, rows of at most 12,004 entries: 1e-5 of the largest
        # sum is many times their spread
        assert np.max(np.abs(C - R)) <= 1e-5 * max(1.0, float(np.max(np.abs(R)))), (name, K)
        assert torch.all(full[:, :1] == 7.0) and torch.all(full[:, 1 + K:] == 7.0), (name, K)


SDDMM_GRAPHS = {
    # even rows, Y past the lines of the narrow routes
    "even_wide_y": lambda: graphs.erdos_renyi_gcn(nodes=700_000, edges=700_000, seed=8),
    "even": GRAPHS["even"],
    # blocks: tiles whose widths 16 and 32 do not divide
    "sbm": lambda: graphs.sbm(communities=64, seed=5, val_seed=6),
}


@pytest.mark.parametrize("off,pad", [(0, 0), (1, 1)])
@pytest.mark.parametrize("name", list(SDDMM_GRAPHS))
def test_sddmm_routes(name, off, pad):
    g = SDDMM_GRAPHS[name]()
    plan = trspmm.Plan.for_sddmm(trspmm.build_format_device(*(torch.from_numpy(a).cuda() for a in (g.rowptr, g.col, g.val))), g.m, g.n)
    for K in (9, 12, 15, 16, 17, 24, 31, 32, 100, 124, 244):
        print("sddmm route", name, K, off, pad, flush=True)
        X, Xh = inside(g.m, K, off, pad, seed=K)
        Y, Yh = inside(g.n, K, off, pad, seed=K + 1)
        S = plan.sddmm(X, Y)
        torch.cuda.synchronize()
        R = osp.csr_sddmm(g.rowptr[: g.m + 1], g.col, Xh, Yh)
        # per-entry dot of K fp16 products, fp32 accumulation
        assert np.max(np.abs(S.cpu().numpy() - R)) <= (1e-5 * np.sqrt(K) * 4 + 1e-6) * max(1.0, float(np.max(np.abs(R)))), (name, K)
