"""Up to 16 rows with fewer workgroups than CUs and a long K: two waves of six ring slots in place of one of eight."""
import numpy as np
import pytest

# m, n, k -> waves, ring slots, K splits; either side of each limit of the rule
EDGES = [((1, 560, 4352), (2, 6, 1)), ((1, 560, 4096), (1, 8, 1)),             # seventeen blocks of K
         ((8, 3200, 4352), (2, 6, 1)), ((8, 3216, 4352), (1, 8, 1)),           # 200 workgroups
         ((8, 3216, 7680), (2, 6, 1)), ((8, 3856, 7680), (1, 8, 1)),           # 240 with thirty blocks each
         ((9, 1600, 4352), (2, 6, 1)), ((9, 1616, 4352), (1, 8, 1)),           # 100 at 9..16 rows
         ((16, 130, 17408), (2, 6, 4)), ((2, 130, 4368), (1, 8, 1))]           # split; off the 128-byte lines


@pytest.fixture(scope="module")
def sg():
    import rocm_dev_amd
    rocm_dev_amd.tuning_clear()
    yield rocm_dev_amd
    rocm_dev_amd.tuning_clear()


@pytest.mark.parametrize("shape,want", EDGES)
def test_the_choice_on_either_side_of_its_limits(sg, shape, want):
    t, _ = sg.skinny_gemm_choice(*shape)
    assert (t.engine, t.row_tiles, t.waves, t.depth, t.split_k) == (2, 1) + want


@pytest.mark.gpu
@pytest.mark.parametrize("shape,want", EDGES)
def test_the_choice_against_the_oracle(sg, oracle, shape, want):
    from gpu_util import GEMM_TOL, bits, dev, rowcol_reference, scale_tensor
    import torch
    m, n, k = shape
    a8, b8, scale = oracle.make_gemm_operands(m, n, k, seed=n)
    D = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    sg.skinny_gemm_fastpath(dev(a8), dev(b8), D, scale_tensor(scale), check=True)
    assert oracle.max_rel_err_bf16(bits(D), rowcol_reference(oracle, a8, b8, scale, model=True)) <= GEMM_TOL
