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


# 2^13 columns: one pass of 32 lanes to K = 256, passes of 128 above.  2^16 and 2^18 columns: Y beyond the
# size to which one pass is taken (odd widths 16 MB, even ones 64 MB), so passes of 128 from K = 129 on.
@pytest.mark.parametrize("K, scale", [(130, 13), (136, 13), (160, 13), (192, 13), (193, 13), (256, 13), (257, 13),
                                      (264, 13), (145, 16), (129, 16), (130, 18)])
def test_narrow_last_pass_adds_to_the_merged_outputs(K, scale):
    print("sddmm narrow last pass", K, scale, flush=True)
    g = graphs.rmat(scale=scale, edge_factor=16 if scale == 13 else 1, seed=9)
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
