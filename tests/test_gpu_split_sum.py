"""The launch that adds a K split's partials: every build of it against the sum inside the GEMM."""
import pytest
import torch

from gpu_util import scale_tensor

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sg():
    import rocm_dev_amd
    rocm_dev_amd.tuning_clear()
    yield rocm_dev_amd
    rocm_dev_amd.tuning_clear()


@pytest.mark.parametrize("split", [2, 3, 4, 5, 8, 9, 16, 17])
@pytest.mark.parametrize("m,n,k", [(130, 70, 2176), (100, 1346, 2192), (600, 4098, 2176)])   # 6, 44 and 650 workgroups that add
def test_the_sum_in_a_launch_of_its_own_has_the_bits_of_the_sum_in_the_gemm(sg, m, n, k, split):
    """Both add the partials in split order, whatever the build of the launch and however the splits fill its batches."""
    g = torch.Generator().manual_seed(split)
    A, B = (torch.randn((rows, k), generator=g).to(torch.float8_e4m3fn).view(torch.uint8).cuda() for rows in (m, n))
    S = scale_tensor(0.5)
    D = [torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    for deferred in (0, 1):
        assert sg.skinny_gemm_tuned(A, B, D[deferred], S, engine=4, split_k=split, waves=4, row_tiles=2, m_blocks=2, depth=4, k_chunks=0,
                                    wave_tiles=deferred) == 0
    assert torch.equal(D[0], D[1])
