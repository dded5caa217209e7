"""K splits of the mid-batch kernel and of the skinny ring over several activation tiles beyond their records'."""
import numpy as np
import pytest
import torch

from gpu_util import GEMM_TOL, bits, dev, rowcol_reference, scale_tensor

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sg():
    import rocm_dev_amd
    rocm_dev_amd.tuning_clear()
    yield rocm_dev_amd
    rocm_dev_amd.tuning_clear()


# unsplit records and split ones, whole lines and part of a block at the end of K, an n that four does not divide, padded rows
@pytest.mark.parametrize("m,n,k,pad", [(1061, 128, 6144, 0), (316, 230, 3584, 16), (915, 188, 8640, 0), (1500, 134, 4048, 128),
                                       (268, 164, 6656, 0), (130, 160, 11904, 0), (33, 650, 4944, 16), (256, 130, 5792, 0),
                                       (92, 314, 12416, 128)])
@pytest.mark.parametrize("factors", [False, True])
def test_the_choice_against_the_oracle_eagerly_and_in_a_graph(sg, oracle, m, n, k, pad, factors):
    """The library's own launch, with and without row and column factors; recorded, where an unsplit record stays what it was,
    and replayed."""
    t, _ = sg.skinny_gemm_choice(m, n, k)
    assert t.engine in (2, 4) and t.split_k > 1, "not a shape of these rules"
    a8, b8, scale = oracle.make_gemm_operands(m, n, k, seed=n)
    rs, cs = (np.random.default_rng(m + i).uniform(0.5, 1.5, c).astype(np.float32) if factors else None for i, c in enumerate((m, n)))
    # (the model of the instruction's summation: a sum near zero, at the metric's floor of 1e-2 rms, is 1e-4 rms off the sequential one)
    ref = rowcol_reference(oracle, a8, b8, scale, rs, cs, model=True)
    A, S = dev(a8), scale_tensor(scale)
    B = torch.full((n, k + pad), 0x7f, dtype=torch.uint8, device="cuda")[:, :k]
    B.copy_(dev(b8))
    R, Cs = (None if x is None else torch.from_numpy(x).cuda() for x in (rs, cs))
    D = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    call = (lambda: sg.skinny_gemm_rowcol(A, B, D, S, R, Cs, check=True)) if factors else (lambda: sg.skinny_gemm_fastpath(A, B, D, S, check=True))
    call()
    assert oracle.max_rel_err_bf16(bits(D), ref) <= GEMM_TOL
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for _ in range(3):
        D.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert oracle.max_rel_err_bf16(bits(D), ref) <= GEMM_TOL
        call()
