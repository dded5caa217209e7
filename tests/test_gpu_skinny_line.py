"""The skinny kernels for rows off their 128-byte lines (sg_skinny_line_kernel.h): every compiled build at the sizes where its
edges can go wrong, every place a row can start on its line, and the library's own choice of them."""
import numpy as np
import pytest
import torch

from gpu_util import GEMM_TOL, bits, dev, rowcol_reference, scale_tensor
from test_gpu_line import _in_nans

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sg():
    import rocm_dev_amd
    rocm_dev_amd.tuning_clear()
    yield rocm_dev_amd
    rocm_dev_amd.tuning_clear()


def _builds(m, k):
    """(resident, waves, row tiles, depth, K split) of every compiled kernel that takes m rows, with rings that fit the LDS; one
    wave per workgroup as well, which then walks several tiles with one ring"""
    xu, blocks = 8 if m > 16 else 1 if m <= 4 else 2 if m <= 8 else 4, -(-k // 256)
    tiles = [(1, 4), (2, 4), (4, 3)] if m > 16 else [(1, 4), (2, 3), (2, 4)] + ([(4, 3)] if m > 8 else [])
    return ([(1, w, 1, d, 1) for w in (1, 4, 8) for d in (3, 4) if blocks * xu + w * d * 4 + 4 <= 159] +
            [(0, w, rg, d, sk) for rg, d in tiles for w in (1, 2, 3) for sk in (1, 2, 3)
             if w * d * (4 * rg + xu) + 4 <= 159 and sk <= k // 256])


def _run(A, B, D, S, rs, cs, build):
    from rocm_dev_amd._lib import lib
    resident, waves, rg, depth, sk = build
    return lib.sg_debug_skinny_line_gemm(A.data_ptr(), B.data_ptr(), D.data_ptr(), S.data_ptr(),
                                         rs.data_ptr() if rs is not None else None, cs.data_ptr() if cs is not None else None,
                                         A.shape[0], B.shape[0], A.shape[1], B.stride(0), resident, waves, rg, depth, sk,
                                         torch.cuda.current_stream().cuda_stream)


# a block and one piece; the last piece that needs no pair behind the last block's own (400, 656) and the first that does (416);
# whole blocks; more pairs than any ring has slots; one weight row pair, a tile's rows and two more, edges of 64-row tiles;
# 520 tiles, of which one-wave workgroups walk two or three and some waves of the others find none
@pytest.mark.parametrize("m,n,k,pad", [(1, 2, 272, 0), (4, 34, 400, 0), (5, 130, 656, 48), (8, 258, 416, 16), (9, 66, 2304, 16),
                                       (16, 190, 1680, 0), (17, 34, 400, 112), (32, 322, 2032, 0), (25, 66, 512, 80),
                                       (3, 8310, 784, 0), (32, 8310, 528, 0), (12, 8310, 400, 16)])
def test_every_build_at_its_edges(oracle, m, n, k, pad):
    a8, b8, scale = oracle.make_gemm_operands(m, n, k, seed=m + n)
    ref = rowcol_reference(oracle, a8, b8, scale, None, None, model=True)
    rs = np.random.default_rng(1).uniform(0.5, 2.0, size=m).astype(np.float32)
    cs = np.random.default_rng(2).uniform(0.5, 2.0, size=n).astype(np.float32)
    ref_rc = rowcol_reference(oracle, a8, b8, scale, rs, cs, model=True)
    A, B, S, R, C = _in_nans(a8, k, 16), _in_nans(b8, k + pad, 48), scale_tensor(scale), dev(rs), dev(cs)
    ran = 0
    for build in _builds(m, k):
        G = torch.full((m + 8, n), 9.0, dtype=torch.bfloat16, device="cuda")   # guard rows around the output
        D = G[4:4 + m]
        for r, c, want in ((None, None, ref), (R, C, ref_rc)):
            D.fill_(float("nan"))
            assert _run(A, B, D, S, r, c, build) == 0, build
            torch.cuda.synchronize()
            assert (G[:4] == 9).all() and (G[4 + m:] == 9).all(), build
            err = oracle.max_rel_err_bf16(bits(D), want)
            assert err <= GEMM_TOL, (build, err)
        ran += 1
    assert ran > 8


@pytest.mark.parametrize("pitch", range(16, 129, 16))
def test_every_place_on_the_line(oracle, pitch):
    """Weight rows `pitch` bytes further on their line each (eight pitches), both operands starting at each of its eight
    pieces, on a k of whole blocks and on two that end within a block."""
    n = 3 * 64 + 2
    for m, builds in ((7, [(1, 4, 1, 3, 1), (0, 2, 2, 4, 1), (0, 1, 1, 4, 2)]), (30, [(1, 4, 1, 4, 1), (0, 2, 4, 3, 1)])):
        for k in (1024, 1024 + 48, 1024 + 144):
            a8, b8, scale = oracle.make_gemm_operands(m, n, k, seed=pitch)
            ref = rowcol_reference(oracle, a8, b8, scale, None, None, model=True)
            S = scale_tensor(scale)
            for offset in range(0, 128, 16):
                A, B = _in_nans(a8, k, offset), _in_nans(b8, 1280 + pitch, 112 - offset)
                for build in builds:
                    D = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
                    assert _run(A, B, D, S, None, None, build) == 0
                    err = oracle.max_rel_err_bf16(bits(D), ref)
                    assert err <= GEMM_TOL, (k, offset, build, err)


@pytest.mark.parametrize("m", [11, 28])
def test_nan_codes_poison_their_row_and_column_only(oracle, m):
    """A NaN in the pieces of the last block, which pieces behind the end of a row repeat."""
    n, k = 200, 1040
    a8, b8, scale = oracle.make_gemm_operands(m, n, k, seed=3)
    a8[7, k - 1] = 0x7f
    b8[150, k - 16] = 0x7f
    A, B, S = dev(a8), dev(b8), scale_tensor(scale)
    want = np.zeros((m, n), bool)
    want[7] = True
    want[:, 150] = True
    for build in _builds(m, k):
        D = torch.zeros((m, n), dtype=torch.bfloat16, device="cuda")
        assert _run(A, B, D, S, None, None, build) == 0
        assert np.array_equal(torch.isnan(D).cpu().numpy(), want), build


# every launch the rule takes, up to 16 rows and above; a K split, and one off its lines by the stride only
@pytest.mark.parametrize("m,n,k,pad", [(3, 400, 26000, 0), (12, 1522, 23056, 0), (5, 2434, 21584, 16), (16, 8192, 4112, 0), (2, 8522, 2832, 0),
                                       (12, 14000, 9664, 0), (1, 20288, 1344, 16), (10, 18096, 8208, 0), (4, 27680, 1488, 16),
                                       (30, 698, 5488, 128), (27, 4112, 12352, 0), (20, 2538, 6112, 0), (24, 5042, 3984, 0), (24, 9314, 4320, 16),
                                       (29, 13116, 6960, 16), (32, 32768, 1040, 0), (31, 26412, 3648, 0)])
def test_the_choice_and_whose_workspace(sg, m, n, k, pad):
    """The library's own launch is the build that the choice names, bit for bit: eagerly, by engine 0, behind the encoder, on a
    workspace of the caller's of the size the query asks for and in a replayed graph."""
    from rocm_dev_amd import api
    choice = api.skinny_gemm_skinny_line_choice(m, n, k, k + pad)
    assert choice, "not a shape of these kernels"
    waves, rg, depth, sk, resident = choice
    g = torch.Generator(device="cuda").manual_seed(m)
    W = torch.zeros((n, k + pad), dtype=torch.uint8, device="cuda")
    W[:, :k] = torch.randn((n, k), generator=g, device="cuda").to(torch.float8_e4m3fn).view(torch.uint8)
    X = torch.randn((m, k), generator=g, device="cuda").bfloat16()
    A, W, S = X.float().to(torch.float8_e4m3fn).view(torch.uint8), W[:, :k], scale_tensor(0.5)
    want, D = (torch.empty((m, n), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    assert _run(A, W, want, S, None, None, (resident, waves, rg, depth, sk)) == 0
    assert sg.skinny_gemm_fastpath(A, W, D, S) == 0
    assert torch.equal(D, want)
    D.zero_()
    assert sg.skinny_gemm_tuned(A, W, D, S, engine=0) == 0
    assert torch.equal(D, want)
    ws = torch.empty(max(sg.workspace_query(m, n, k), 1 << 17), dtype=torch.uint8, device="cuda")
    sg.workspace_init(ws)
    D.zero_()
    assert sg.skinny_gemm_auto_ws(A, W, D, S, ws) == 0
    assert torch.equal(D, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        sg.skinny_gemm_auto_ws(A, W, D, S, ws, check=True)
    for _ in range(3):
        D.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(D, want)
    Q, s = torch.empty((m, k), dtype=torch.uint8, device="cuda"), torch.empty((m,), device="cuda")
    assert sg.fp8_encode_rows(X, Q, s) == 0 and sg.skinny_gemm_rowcol(Q, W, want, S, s) == 0
    assert sg.skinny_gemm_bf16act(X, W, D, S) == 0
    assert torch.equal(D, want)
