"""SDDMM of more than one feature pass whose last pass is narrow: it adds to where the earlier passes
wrote, also where the plan holds a split part (merged from a buffer of its own) and a task list for
narrow lane groups."""
import numpy as np
import pytest
import torch

from oracle import spmm as osp
from trspmm import graphs
import trspmm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [130, 136, 160, 192, 193, 264])
def test_narrow_last_pass_adds_to_the_merged_outputs(K):
    print("sddmm narrow last pass", K, flush=True)
    g = graphs.rmat(scale=13, edge_factor=16, seed=9)
    f = trspmm.build_format(g.rowptr, g.col, g.val)
    plan = trspmm.Plan.for_sddmm(f, g.m, g.n, mfma_tc=False, mfma_sptc=False, xcd_split=64, task_nnz=16)
    assert plan.stats()["split_rows"] > 0 and plan.sddmm_workspace_bytes(K) > 0
    Xh = graphs.dense_operand(g.m, K, seed=K)
    Yh = graphs.dense_operand(g.n, K, seed=K + 1)
    S = plan.sddmm(torch.from_numpy(Xh).cuda(), torch.from_numpy(Yh).cuda())
    torch.cuda.synchronize()
    R = osp.csr_sddmm(g.rowptr[: g.m + 1], g.col, Xh, Yh)
    # per-entry dot of K fp16 products, fp32 accumulation
    tol = (1e-5 * np.sqrt(K) * 4 + 1e-6) * max(1.0, float(np.max(np.abs(R))))
    assert np.max(np.abs(S.cpu().numpy() - R)) <= tol
