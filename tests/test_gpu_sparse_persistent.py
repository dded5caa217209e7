"""The 2:4 kernel with the activations in registers (17..32 rows on more than two tiles per CU): every number of waves, one
and two K stages a wave, whole and ragged last tiles, workgroups of two tiles and more; against the oracle and the
kernel of one workgroup per tile."""
import numpy as np
import pytest
import torch

from gpu_util import GEMM_TOL, bits, dev, scale_tensor, sparse_reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(17, 8194, 2048), (32, 8210, 2560), (31, 8194, 3072), (20, 8206, 3584), (32, 16386, 4096),
                                   (18, 8194, 5120), (32, 8194, 6144), (29, 8200, 7168), (32, 8194, 8192)])
def test_against_the_oracle(oracle, m, n, k):
    import rocm_dev_amd as sg
    a8, vals, meta, _, scale = oracle.make_sparse24_operands(m, n, k, seed=m + k)
    room = torch.full((m + 8, n), 7.0, dtype=torch.bfloat16, device="cuda")     # guard rows around the output
    D = room[4:4 + m]
    A, V, M, S = dev(a8), dev(vals), dev(meta), scale_tensor(scale)
    D.fill_(float("nan"))
    assert sg.sparse24_gemm(A, V, M, D, S) == 0
    first = D.clone()
    assert sg.sparse24_gemm(A, V, M, D, S) == 0
    torch.cuda.synchronize()
    assert (room[:4] == 7).all() and (room[4 + m:] == 7).all()
    assert torch.equal(first, D)
    assert oracle.max_rel_err_bf16(bits(D), sparse_reference(oracle, a8, vals, meta, scale)) <= GEMM_TOL
    # one workgroup per tile, its K in another order: one bf16 rounding apart (1.6e-3 is a rounding's 2-norm, four times that)
    E = torch.empty_like(first)
    one = sg.SgTuning(2, 1, 1, 1, 2, 2, 8, 1, 0, 0)
    assert sg.sparse24_gemm(A, V, M, E, S, tuning=one) == 0
    assert float((E.float() - first.float()).norm() / first.float().norm()) < 7e-3


def test_a_nan_code_poisons_its_row_only(oracle):
    import rocm_dev_amd as sg
    m, n, k = 32, 8194, 2048
    a8, vals, meta, _, scale = oracle.make_sparse24_operands(m, n, k, seed=5)
    vals = vals.copy()
    vals[8193, 17] = 0x7f
    D = torch.zeros((m, n), dtype=torch.bfloat16, device="cuda")
    assert sg.sparse24_gemm(dev(a8), dev(vals), dev(meta), D, scale_tensor(scale)) == 0
    bad = torch.isnan(D).cpu().numpy()
    assert bad[:, 8193].all() and not bad[:, :8193].any()
