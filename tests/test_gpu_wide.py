"""The wide-tile GEMM (more than 128 activation rows): every compiled tile at the sizes where its edges can go wrong,
and the library's own choice of it."""
import numpy as np
import pytest
import torch

from gpu_util import GEMM_TOL, bits, dev, gemm_reference, rowcol_reference, scale_tensor

pytestmark = pytest.mark.gpu

TILES = [(4, 8), (5, 8), (6, 8), (7, 8), (8, 8), (8, 4), (4, 4)]     # weight rows / 32, activation rows / 32


def _wide(A, B, D, S, rs, cs, rg, mb, sk):
    from rocm_dev_amd._lib import lib
    m, k = A.shape
    return lib.sg_debug_wide_gemm(A.data_ptr(), B.data_ptr(), D.data_ptr(), S.data_ptr(), rs.data_ptr() if rs is not None else None,
                                  cs.data_ptr() if cs is not None else None, m, B.shape[0], k, B.stride(0), rg, mb, sk,
                                  torch.cuda.current_stream().cuda_stream)


# one row more and less than a tile, a single weight row pair, rows of D off their 16-byte pieces, K of one block and a bit,
# odd and even block counts shorter and longer than the rings, a last block of one 16-byte piece and of seven
@pytest.mark.parametrize("m,n,k,pad", [(129, 2, 144, 0), (256, 256, 256, 0), (257, 226, 384, 16), (255, 514, 640, 0),
                                       (300, 322, 1136, 16), (130, 1000, 2048, 0), (513, 160, 2064, 128)])
def test_every_tile_at_its_edges(oracle, m, n, k, pad):
    a8, b8, scale = oracle.make_gemm_operands(m, n, k, seed=m + n, b_stride=k + pad if pad else None)
    dense = np.ascontiguousarray(b8[:, :k])
    # The oracle's model of the instruction's own sum at every k: an aligned run of 8 products is cut about 14 binades
    # below its largest, so one of n outputs of a sum of k products leaves the sequential sum by up to about
    # sqrt(k) * 2^-14 of a product - 0.010056 of the metric, whose floor is 1e-2 rms, in one of the 82080 outputs of the
    # last shape, whichever kernel forms it.
    ref = rowcol_reference(oracle, a8, dense, scale, None, None, model=True)
    rs = np.random.default_rng(1).uniform(0.5, 2.0, size=m).astype(np.float32)
    cs = np.random.default_rng(2).uniform(0.5, 2.0, size=n).astype(np.float32)
    ref_rc = rowcol_reference(oracle, a8, dense, scale, rs, cs, model=True)
    A, B, S, R, Cc = dev(a8), dev(b8)[:, :k], scale_tensor(scale), dev(rs), dev(cs)
    for rg, mb in TILES:
        for sk in (1, 2, 3):
            # guard rows around the output
            room = torch.full((m + 16, n), 7.0, dtype=torch.bfloat16, device="cuda")
            D = room[8:m + 8]
            scaled = sk != 2
            rc = _wide(A, B, D, S, R if scaled else None, Cc if scaled else None, rg, mb, sk)
            torch.cuda.synchronize()
            if sk > k // 128:
                assert rc == 6
                continue
            assert rc == 0, (rg, mb, sk, rc)
            assert oracle.max_rel_err_bf16(bits(D), ref_rc if scaled else ref) <= GEMM_TOL, (rg, mb, sk)
            assert bool((room[:8] == 7.0).all()) and bool((room[m + 8:] == 7.0).all()), (rg, mb, sk)


# every remainder of n by the 8 outputs of a 16-byte store, on a D that is aligned to 16 bytes and to 8 only, and a tile
# whose last columns are all beyond n
@pytest.mark.parametrize("n", [260, 262, 264, 266, 390])
@pytest.mark.parametrize("off", [0, 4])
def test_rows_off_their_16_byte_pieces(oracle, n, off):
    m, k = 131, 256
    a8, b8, scale = oracle.make_gemm_operands(m, n, k, seed=n)
    ref = rowcol_reference(oracle, a8, b8, scale, None, None, model=True)
    A, B, S = dev(a8), dev(b8), scale_tensor(scale)
    for rg, mb in TILES:
        room = torch.full((m * n + 64,), 7.0, dtype=torch.bfloat16, device="cuda")
        D = room[8 + off:8 + off + m * n].view(m, n)
        assert D.data_ptr() % 16 == 2 * off
        assert _wide(A, B, D, S, None, None, rg, mb, 1) == 0
        torch.cuda.synchronize()
        assert oracle.max_rel_err_bf16(bits(D), ref) <= GEMM_TOL, (rg, mb)
        assert bool((room[:8 + off] == 7.0).all()) and bool((room[8 + off + m * n:] == 7.0).all()), (rg, mb)


# shapes the library itself runs on wide tiles, and on which: unsplit with whole K blocks, K split with its sum in a second
# launch, partial last block with padded rows, rows of D off their 16-byte pieces
CHOICES = [(512, 11008, 4096, 0, (4, 8, 1)), (640, 3584, 8192, 0, (8, 4, 3)), (1030, 4098, 3088, 16, (4, 8, 1)),
           (600, 8196, 8192, 0, (4, 8, 1))]
SPLIT = CHOICES[1]


def _operands(oracle, m, n, k, pad, seed):
    a8, b8, scale = oracle.make_gemm_operands(m, n, k, seed=seed, b_stride=k + pad if pad else None)
    return a8, np.ascontiguousarray(b8[:, :k]), scale, dev(a8), dev(b8)[:, :k], scale_tensor(scale)


@pytest.mark.parametrize("m,n,k,pad,tile", CHOICES)
def test_the_librarys_choice(oracle, m, n, k, pad, tile):
    import rocm_dev_amd as sg
    sg.tuning_clear()
    assert sg.api.skinny_gemm_wide_choice(m, n, k, k + pad) == tile
    a8, dense, scale, A, B, S = _operands(oracle, m, n, k, pad, k)
    D = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    assert sg.skinny_gemm_fastpath(A, B, D, S) == 0
    torch.cuda.synchronize()
    assert oracle.max_rel_err_bf16(bits(D), gemm_reference(oracle, a8, dense, scale)) <= GEMM_TOL
    # bit for bit what that tile computes
    again = torch.full_like(D, float("nan"))
    assert _wide(A, B, again, S, None, None, *tile) == 0
    torch.cuda.synchronize()
    assert torch.equal(D.view(torch.int16), again.view(torch.int16))


def test_caller_owned_workspace_of_a_split_wide_tile(oracle):
    """Exactly the bytes sg_workspace_query asks for hold a wide tile's K split, the result is the one with the library's own
    workspace, and nothing behind them is written; one byte less is refused."""
    import rocm_dev_amd as sg
    sg.tuning_clear()
    m, n, k, pad, tile = SPLIT
    _, _, _, A, B, S = _operands(oracle, m, n, k, pad, 1)
    want, D = (torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    assert sg.skinny_gemm_fastpath(A, B, want, S) == 0
    need = sg.workspace_query(m, n, k)
    assert need > 0
    room = torch.full((need + 4096,), 0xA5, dtype=torch.uint8, device="cuda")
    ws = room[:need]
    sg.workspace_init(ws)
    for _ in range(2):
        D.fill_(float("nan"))
        assert sg.skinny_gemm_auto_ws(A, B, D, S, ws) == 0
        torch.cuda.synchronize()
        assert torch.equal(D.view(torch.int16), want.view(torch.int16))
    assert bool((room[need:] == 0xA5).all())
    assert sg.skinny_gemm_auto_ws(A, B, D, S, room[:need - 1]) == 10
    # the library's fixed array is smaller: its own choice is made to fit
    assert sg.skinny_gemm_tuned_noalloc(A, B, D, S) == 0
    torch.cuda.synchronize()
    assert float((D.float() - want.float()).norm() / want.float().norm()) < 4e-3      # two bf16 roundings


def test_split_wide_tiles_in_graphs_and_on_two_streams(oracle):
    """The K split of wide tiles, whose partials live in the stream's workspace: two streams and two threads at once, and a
    graph replayed with eager work between, give the bits of one launch by itself."""
    import threading

    import rocm_dev_amd as sg
    sg.tuning_clear()
    m, n, k, pad, tile = SPLIT
    jobs = [_operands(oracle, m, n, k, pad, seed)[3:] for seed in (2, 3)]
    want = []
    for A, B, S in jobs:
        want.append(torch.empty((m, n), dtype=torch.bfloat16, device="cuda"))
        assert sg.skinny_gemm_fastpath(A, B, want[-1], S) == 0
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in jobs]
    outs = [[torch.empty_like(want[0]) for _ in range(8)] for _ in jobs]
    codes = []

    def work(j):
        with torch.cuda.stream(streams[j]):
            for D in outs[j]:
                codes.append(sg.skinny_gemm_fastpath(jobs[j][0], jobs[j][1], D, jobs[j][2]))

    threads = [threading.Thread(target=work, args=(j,)) for j in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert codes == [0] * 16
    for j, w in enumerate(want):
        assert all(torch.equal(D.view(torch.int16), w.view(torch.int16)) for D in outs[j])

    graph, D = torch.cuda.CUDAGraph(), torch.empty_like(want[0])
    A, B, S = jobs[0]
    with torch.cuda.stream(streams[0]):
        with torch.cuda.graph(graph, stream=streams[0]):
            assert sg.skinny_gemm_fastpath(A, B, D, S) == 0
    for _ in range(3):
        D.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(D.view(torch.int16), want[0].view(torch.int16))
        assert sg.skinny_gemm_fastpath(jobs[1][0], jobs[1][1], outs[1][0], jobs[1][2]) == 0     # eager, the same split, between replays
        torch.cuda.synchronize()
        assert torch.equal(outs[1][0].view(torch.int16), want[1].view(torch.int16))
    del graph


@pytest.mark.parametrize("k", [512, 1040])
def test_nan_codes_stay_in_their_rows_and_columns(oracle, k):
    """NaN codes of both signs in the first block, at the end of the row and in the part of the last window that the block
    before has already multiplied: exactly their rows (activations) and columns (weights) are NaN, no other bit changes."""
    m, n = 260, 300
    a8, b8, scale = oracle.make_gemm_operands(m, n, k, seed=k)
    rows, cols = {3: (0, 0x7F), 130: (k - 1, 0xFF), 259: (k - 130, 0x7F)}, {0: (k - 1, 0x7F), 131: (5, 0xFF), 299: (k - 100, 0x7F)}
    clean_a, clean_b = a8.copy(), b8.copy()
    for i, (at, code) in rows.items():
        a8[i, at], clean_a[i, at] = code, 0
    for j, (at, code) in cols.items():
        b8[j, at], clean_b[j, at] = code, 0
    S = scale_tensor(scale)
    for rg, mb in TILES:
        for sk in (1, 2):
            D, C = (torch.zeros((m, n), dtype=torch.bfloat16, device="cuda") for _ in range(2))
            assert _wide(dev(a8), dev(b8), D, S, None, None, rg, mb, sk) == 0
            assert _wide(dev(clean_a), dev(clean_b), C, S, None, None, rg, mb, sk) == 0
            torch.cuda.synchronize()
            want = torch.isnan(C)
            assert not bool(want.any())
            want[list(rows)] = True
            want[:, list(cols)] = True
            assert torch.equal(torch.isnan(D), want), (rg, mb, sk)
            assert torch.equal(D.view(torch.int16)[~want], C.view(torch.int16)[~want]), (rg, mb, sk)


def test_refused_tiles(oracle):
    a8, b8, scale = oracle.make_gemm_operands(129, 64, 256, seed=0)
    A, B, S = dev(a8), dev(b8), scale_tensor(scale)
    D = torch.zeros((129, 64), dtype=torch.bfloat16, device="cuda")
    for rg, mb, sk in ((3, 8, 1), (9, 8, 1), (5, 4, 1), (8, 2, 1), (8, 8, 0), (8, 8, 3)):
        assert _wide(A, B, D, S, None, None, rg, mb, sk) == 6, (rg, mb, sk)
