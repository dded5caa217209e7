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
