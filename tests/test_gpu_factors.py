"""Row and column factors in every epilogue but the wide tile's (test_gpu_wide.py), and outputs whose rows are off their 8-byte pieces.

Factors that are powers of two commute with every rounding on the way (no output here is subnormal), so the product with
factors must be, bit for bit, the product without them times the factors."""
import numpy as np
import pytest
import torch

from gpu_util import bits, scale_tensor

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sg():
    import rocm_dev_amd
    return rocm_dev_amd


# m, n, k, pad: n = 2 mod 4 (the last fragment ends inside a lane's four columns) except where a kernel wants whole tiles
SHAPES = [
    (1, 2, 512, 0), (8, 4098, 4096, 0), (13, 6146, 4112, 16), (30, 4098, 14336, 0), (32, 1026, 8192, 0),   # per-tile ring, K splits
    (17, 14338, 2816, 0), (32, 14338, 5120, 0),                                                            # ... on 64-row tiles
    (8, 28674, 4096, 0), (16, 9218, 4096, 0), (5, 12290, 3072, 128),                                       # persistent, activations in LDS
    (32, 28674, 4096, 0), (16, 14338, 8192, 0),                                                            # persistent, in registers
    (12, 14338, 9472, 0),                                                                                  # persistent, in the ring
    (8, 16386, 512, 0), (32, 28674, 1040, 0), (32, 40962, 1792, 0),                                        # whole tiles per wave
    (9, 302, 208, 0),                                                                                      # register streaming
    (64, 6146, 4096, 0), (40, 1026, 28672, 0),                                                             # several activation tiles
    (40, 130, 144, 16), (128, 8194, 8192, 0), (33, 57346, 640, 0),                                         # mid-batch, with and without a K split
    (100, 2374, 5440, 16), (100, 10946, 3696, 16), (100, 3698, 10944, 16),                                 # rows off their lines, the same
]


@pytest.mark.parametrize("m,n,k,pad", SHAPES)
def test_factors_of_two_scale_every_output_exactly(sg, m, n, k, pad):
    g = torch.Generator().manual_seed(m + n + k)
    W = torch.zeros((n, k + pad), dtype=torch.uint8)
    W[:, :k] = torch.randn((n, k), generator=g).to(torch.float8_e4m3fn).view(torch.uint8)
    A = torch.randn((m, k), generator=g).to(torch.float8_e4m3fn).view(torch.uint8).cuda()
    W = W.cuda()[:, :k]
    S = scale_tensor(0.25)
    # views one float into their buffers: 4-byte alignment is all that the library asks for
    row = torch.pow(2.0, torch.randint(-3, 4, (m + 1,), generator=g).float()).cuda()[1:]
    col = torch.pow(2.0, torch.randint(-3, 4, (n + 1,), generator=g).float()).cuda()[1:]
    guard = 5

    def run(r, c):
        D = torch.full((m + 2 * guard, n), 77.0, dtype=torch.bfloat16, device="cuda")
        assert sg.skinny_gemm_rowcol(A, W, D[guard:guard + m], S, r, c) == 0
        torch.cuda.synchronize()
        assert (D[:guard] == 77).all() and (D[guard + m:] == 77).all(), "wrote outside its rows"
        return D[guard:guard + m]

    if (guard * n * 2) % 8:
        guard = 4       # the output is 8-byte aligned
    plain = run(None, None).float()
    assert float(plain.abs().max()) > 0
    for r, c in ((row, None), (None, col), (row, col)):
        want = plain.clone()
        if r is not None:
            want *= r[:, None]
        if c is not None:
            want *= c[None, :]
        assert np.array_equal(bits(run(r, c)), bits(want.bfloat16())), (r is not None, c is not None)
