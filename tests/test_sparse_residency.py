"""17..32 rows of a 2:4 GEMM on more than two tiles per CU: 16-row tiles only where three of their workgroups fit a CU (no GPU: the
calls run on a stand-in for the runtime)."""
import random

import launch_recorder
import pytest

CU, LDS = 256, 160 * 1024


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return launch_recorder.build(tmp_path_factory.mktemp("fake"))


# timed with 16-row and with 32-row tiles, us: 6.80 / 5.20, 9.40 / 8.50, 24.6 / 22.1, 28.2 / 25.1, 30.0 / 24.6; K of no whole metadata lines
SHAPES = [(28, 10414, 1024), (23, 20232, 1024), (17, 8948, 9216), (25, 9984, 10240), (20, 8210, 12288), (24, 9988, 896)]


def launches(rec, count):
    r, out = random.Random(3), []
    for i in range(count):
        m, n, k = r.randint(17, 32), 2 * r.randint(4097, 16384), 128 * int(4 * 56 ** r.random())
        if i < len(SHAPES):
            m, n, k = SHAPES[i]
        rc, seen = rec.of("sg_sparse24_gemm", rec.A, rec.B, rec.WS, rec.D, rec.S, m, n, k, None)
        assert rc == 0 and len(seen) == 1
        out.append([(m, n, k), seen[0]])
    return out


def test_sixteen_row_tiles_only_where_three_workgroups_fit_a_cu(fake):
    tall = 0
    for (m, n, k), (kernel, grid, threads, lds) in launch_recorder.scenario(fake, "test_sparse_residency", "launches", 3000):
        if "sparse24_gemm_kernel<2, 1," in kernel:
            assert 3 * lds <= LDS and threads == 64, (m, n, k, kernel, lds)
        elif "sparse24_gemm_kernel<2, 2," in kernel:
            assert 2 * lds <= LDS or threads > 64, (m, n, k, kernel, lds)
            tall += 1
    assert tall > 100


# (m, n, k) -> (16-row tiles of a workgroup, waves).  Timed with these and with one wave on 16-row tiles (m > 16) or on the tile of the
# other line, us: 56.5 / 67.4, 40.6 / 42.9, 77.9 / 90.2; 86 / 117, 82.5 / 96, 41 / 48; 66.9 / 72.6, 78.7 / 100
WAVES = {(32, 20120, 13440): (2, 2), (23, 18202, 9600): (2, 2), (21, 18168, 25088): (2, 2), (32, 17646, 4352): (2, 1), (22, 21052, 7296): (1, 1), (21, 18294, 1280): (1, 1),
         (15, 27430, 23808): (2, 2), (11, 25888, 23808): (2, 2), (16, 14064, 21248): (2, 2), (12, 17654, 12928): (2, 1), (13, 11224, 25600): (1, 1),
         (15, 20000, 12288): (2, 2), (11, 26000, 12288): (2, 1), (12, 13200, 12288): (1, 1), (15, 15786, 7168): (2, 1), (15, 13732, 7168): (2, 1), (10, 14850, 11264): (1, 1), (12, 13200, 20480): (2, 2),
         (3, 25732, 24576): (2, 2), (6, 28004, 24576): (2, 2), (7, 28004, 24448): (2, 1), (6, 20480, 24576): (2, 1), (2, 26624, 7680): (2, 1)}


def builds(rec):
    return [rec.of("sg_sparse24_gemm", rec.A, rec.B, rec.WS, rec.D, rec.S, *shape, None) for shape in WAVES]


def test_two_waves_on_32_row_tiles_where_the_k_is_long(fake):
    for (shape, (rg, waves)), (rc, seen) in zip(WAVES.items(), launch_recorder.scenario(fake, "test_sparse_residency", "builds")):
        kernel, grid, threads, _ = seen[0]
        assert rc == 0 and "sparse24_gemm_kernel<%d, %d," % (1 if shape[0] <= 16 else 2, rg) in kernel and threads == 64 * waves, (shape, kernel, threads)
        assert grid == -(-shape[1] // (16 * rg)), (shape, grid)
