"""A recorded launch whose record splits no K takes no memory of its stream's, so that graphs recorded on one stream may replay side
by side (no GPU: the calls run on a stand-in for the runtime)."""
import ctypes as C
import random

import launch_recorder
import pytest


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return launch_recorder.build(tmp_path_factory.mktemp("fake"))


# 17..32 rows off their 128-byte lines, by k and by the row stride; 33..256 rows on the skinny ring; more on mid-batch tiles: each
# with K splits eagerly in place of a record without
SPLIT_EAGERLY = [(20, 460, 4960, 128), (32, 512, 5136, 0), (31, 676, 5536, 0), (24, 1024, 6160, 0), (18, 1824, 5408, 0), (18, 252, 5296, 0),
                 (25, 316, 6432, 0), (20, 1956, 6832, 0), (130, 160, 11904, 0), (256, 130, 5792, 0), (1061, 128, 6128, 0), (339, 432, 3840, 0)]


def _shapes(count):
    r = random.Random(11)
    yield from SPLIT_EAGERLY
    for _ in range(count):
        m = r.randint(1, 32) if r.random() < 0.6 else int(33 * 31 ** r.random())
        yield m, 2 * int(32 * 200 ** r.random()), 16 * int(16 * 100 ** r.random()), 16 * r.choice([0, 0, 0, 1, 3, 8])


def recorded(rec, count):
    """[shape, launches of the record alone, recorded launches, eager launches], and allocations of all the recorded calls"""
    own_choice, out, four = (C.c_int * 10)(), [], (C.c_int * 4)()
    for m, n, k, pad in _shapes(count):
        shape = (m, n, k, k + pad)
        assert rec.call("sg_debug_line_choice", *shape, 0, four) == 0
        rec.fake.rec_capturing(1)
        # a caller without a workspace is refused where the record needs one
        rc, alone = rec.of("sg_skinny_gemm_auto_ws", rec.A, rec.B, rec.D, rec.S, *shape, None, C.c_size_t(0), None)
        if rc == 0 and not four[0]:
            calls = [rec.of("sg_skinny_gemm_auto", rec.A, rec.B, rec.D, rec.S, *shape, None),
                     rec.of("sg_skinny_gemm_rowcol", rec.A, rec.B, rec.D, rec.S, None, None, *shape, None),
                     rec.of("sg_skinny_gemm_tuned", rec.A, rec.B, rec.D, rec.S, *shape, own_choice, None)]
            assert all(c[0] == 0 for c in calls), (shape, calls)
            out.append([shape, alone, [c[1] for c in calls]])
    allocations = rec.fake.rec_allocations()
    rec.fake.rec_capturing(0)
    for item in out:
        rc, eager = rec.of("sg_skinny_gemm_auto", rec.A, rec.B, rec.D, rec.S, *item[0], None)
        assert rc == 0
        item.append([x for x in eager if "fill_zero" not in x[0]])
    return out, allocations


def test_a_recorded_launch_is_the_record_where_that_needs_no_workspace(fake):
    seen, allocations = launch_recorder.scenario(fake, "test_capture_choice", "recorded", 4000)
    assert allocations == 0
    assert len(seen) > 2000
    for shape, alone, calls, _ in seen:
        assert all(c == alone for c in calls), (shape, alone, calls)
    split = [shape for shape, alone, _, eager in seen if eager != alone]
    assert [list(s) for s in split[:len(SPLIT_EAGERLY)]] == [[m, n, k, k + pad] for m, n, k, pad in SPLIT_EAGERLY]
    assert sum(s[0] <= 32 for s in split) > 30 and sum(s[0] > 32 for s in split) > 30


def recorded_sparse(rec, count):
    r = random.Random(12)
    rec.fake.rec_capturing(1)
    for _ in range(count):
        m, n, k = r.randint(1, 32), 2 * int(1 + 4000 ** r.random()), 128 * int(4 * 56 ** r.random())
        rc, launches = rec.of("sg_sparse24_gemm", rec.A, rec.B, rec.WS, rec.D, rec.S, m, n, k, None)
        assert rc == 0 and len(launches) == 1, (m, n, k)
    allocations = rec.fake.rec_allocations()
    rec.fake.rec_capturing(0)
    rc, _ = rec.of("sg_sparse24_gemm", rec.A, rec.B, rec.WS, rec.D, rec.S, 26, 1040, 12160, None)     # split eagerly
    assert rc == 0
    return allocations, rec.fake.rec_allocations()


def test_recorded_sparse_launches_take_none(fake):
    recorded, eager = launch_recorder.scenario(fake, "test_capture_choice", "recorded_sparse", 2000)
    assert recorded == 0 and eager == 2
