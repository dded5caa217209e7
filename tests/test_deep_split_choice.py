"""K splits of the mid-batch kernel and of the skinny ring over several activation tiles beyond their records', on few weight rows
(no GPU: the library's host code, its launches on a stand-in for the runtime)."""
import ctypes as C
import random
import re

import launch_recorder
import pytest


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return launch_recorder.build(tmp_path_factory.mktemp("fake"))


# shapes whose heuristic record has no K split where the rule takes one: whole lines, a part of a block at the end of K
UNSPLIT_RECORDS = [(1061, 128, 6128), (339, 432, 3840), (915, 188, 8640), (1257, 178, 30144), (1817, 1146, 18160)]


def chosen_and_launched(rec, count):
    """[shape, record, bytes asked for, launches] of random shapes that the mid-batch kernel takes with a K split above 128 rows"""
    r, out = random.Random(5), []
    record, four, three = (C.c_int * 10)(), (C.c_int * 4)(), (C.c_int * 3)()
    need = C.c_size_t()
    for i in range(count):
        m, n, k = int(129 * 20 ** r.random()), 2 * int(1 + 4000 ** r.random()), 16 * int(64 * 40 ** r.random())
        if r.random() < 0.5:
            k = max(1024, k // 128 * 128)
        pad = r.choice([0, 0, 16, 128])
        if i < len(UNSPLIT_RECORDS):
            (m, n, k), pad = UNSPLIT_RECORDS[i], 0
        assert rec.call("sg_skinny_gemm_choice", m, n, k, record, None) == 0
        assert rec.call("sg_debug_line_choice", m, n, k, k + pad, 0, four) == 0
        assert rec.call("sg_debug_wide_choice", m, n, k, k + pad, 0, three) == 0
        if record[0] != 4 or record[1] == 1 or four[0] or three[0]:
            continue
        assert rec.call("sg_workspace_query", m, n, k, C.byref(need)) == 0
        rc, launches = rec.of("sg_skinny_gemm_auto", rec.A, rec.B, rec.D, rec.S, m, n, k, k + pad, None)
        assert rc == 0
        out.append([(m, n, k, pad), list(record), need.value, [x for x in launches if "fill_zero" not in x[0]]])
    return out


def test_the_reported_record_is_what_runs_and_fits_the_workspace_asked_for(fake):
    seen = launch_recorder.scenario(fake, "test_deep_split_choice", "chosen_and_launched", 4000)
    assert len(seen) > 500 and sum(s[0][2] % 128 != 0 for s in seen) > 100
    assert [tuple(s[0][:3]) for s in seen[:len(UNSPLIT_RECORDS)]] == UNSPLIT_RECORDS
    for shape, record, need, launches in seen:
        m, n, k, _ = shape
        _, split, waves, rg, mb = record[:5]
        tiles = -(-n // (8 * waves * rg)) * -(-m // (32 * mb))
        assert len(launches) == 2 and "mid_gemm_kernel" in launches[0][0] and "mid_reduce_kernel" in launches[1][0], (shape, record, launches)
        assert launches[0][1:3] == [tiles * split, 64 * waves], (shape, record, launches)
        assert need >= 65536 + tiles * split * 8 * waves * rg * 32 * mb * 4, (shape, record, need)


TILES = [(4, 2, 2), (4, 2, 4), (4, 4, 4), (8, 2, 2), (8, 2, 4), (8, 2, 8), (8, 4, 2), (8, 4, 4), (8, 4, 8)]    # waves, rg, mt


def model_us(k, waves, rg, mt, of_m_n, split, cu=256):
    bn, bm, lines = 8 * waves * rg, 32 * mt, k % 128 == 0
    stage = (0.232 * bn + 0.247 * bm) / 128 + 0.12 * bn * bm / 16384 if lines else (0.458 * bn + 0.384 * bm) / 128 + 0.073 * bn * bm / 16384
    full, rest = divmod(of_m_n * split, cu)
    part = 0.87 if lines else 0.84
    rounds = full + (part + (1 - part) * rest / cu if rest else 0)
    us = rounds * -(-(-(-k // 128)) // split) * stage + (3.5 + full + (rest > 0) if lines else 4.2)
    return us + (3.1 if lines else 2.7) + (1.36e-6 if lines else 1.57e-6) * bn * bm * of_m_n * split if split > 1 else us


def records_and_choices(rec, count):
    """[shape, the heuristics' own kernel, the record reported] where the former is an unsplit mid-batch launch"""
    r, out, record, three = random.Random(7), [], (C.c_int * 10)(), (C.c_int * 3)()
    for _ in range(count):
        m, n, k = int(129 * 15.8 ** r.random()), 2 * int(1 + 6000 ** r.random()), 128 * int(8 * 32 ** r.random())
        if r.random() < 0.4:
            m, k = r.randint(769, 2048), k + 16 * r.randint(1, 7)
        if m * n * k > 2 ** 36 or k > 32768:
            continue
        rc, launches = rec.of("sg_skinny_gemm_auto_ws", rec.A, rec.B, rec.D, rec.S, m, n, k, k, None, C.c_size_t(0), None)
        assert rec.call("sg_skinny_gemm_choice", m, n, k, record, None) == 0
        assert rec.call("sg_debug_wide_choice", m, n, k, k, 0, three) == 0
        if rc == 0 and len(launches) == 1 and "mid_gemm_kernel" in launches[0][0] and not three[0]:
            out.append([(m, n, k), launches[0][0], list(record)])
    return out


def test_the_choice_is_what_the_model_puts_first_of_all_tiles_and_splits(fake):
    seen = launch_recorder.scenario(fake, "test_deep_split_choice", "records_and_choices", 3000)
    taken = 0
    for (m, n, k), kernel, record in seen:
        own_rg, own_mt, _, along_n = (int(x) for x in re.search(r"mid_gemm_kernel<(\d+), (\d+), (\d+), (\d+)", kernel).groups())
        if along_n == 7:
            continue

        def us(waves, rg, mt, split):
            return model_us(k, waves, rg, mt, -(-n // (8 * waves * rg)) * -(-m // (32 * mt)), split)
        best, pick = 0.95 * us(2 * along_n, own_rg, own_mt, 1), None
        for waves, rg, mt in TILES:
            of_m_n = -(-n // (8 * waves * rg)) * -(-m // (32 * mt))
            if k % 128 and (waves, rg) == (4, 4):
                continue
            for split in range(2, min(16, -(-k // 128) // 4, 512 // of_m_n) + 1):
                if us(waves, rg, mt, split) < best - 1e-9:
                    best, pick = us(waves, rg, mt, split), (split, waves, rg, mt)
        assert tuple(record[1:5]) == pick if pick else record[1] == 1, ((m, n, k), kernel, record, pick)
        taken += bool(pick)
    assert taken > 200 and len(seen) - taken > 200, (taken, len(seen))


RINGS = [(130, 160, 11904), (56, 302, 12288), (90, 464, 10144), (256, 130, 5792), (33, 4998, 2048)]


def rings_chosen_and_launched(rec, count):
    """The same of 33..256 rows on the skinny ring: [shape, record, bytes asked for, launches]"""
    r, out = random.Random(6), []
    record, four, need = (C.c_int * 10)(), (C.c_int * 4)(), C.c_size_t()
    for i in range(count):
        m, n, k = int(33 * 7.8 ** r.random()), 2 * int(1 + 2500 ** r.random()), 16 * int(64 * 32 ** r.random())
        if i < len(RINGS):
            m, n, k = RINGS[i]
        assert rec.call("sg_skinny_gemm_choice", m, n, k, record, None) == 0
        assert rec.call("sg_debug_line_choice", m, n, k, k, 0, four) == 0
        if record[0] != 2 or four[0]:
            continue
        assert rec.call("sg_workspace_query", m, n, k, C.byref(need)) == 0
        rc, launches = rec.of("sg_skinny_gemm_auto", rec.A, rec.B, rec.D, rec.S, m, n, k, k, None)
        assert rc == 0
        out.append([(m, n, k), list(record), need.value, [x for x in launches if "fill_zero" not in x[0]]])
    return out


def test_the_rings_reported_record_is_what_runs_and_fits_the_workspace_asked_for(fake):
    seen = launch_recorder.scenario(fake, "test_deep_split_choice", "rings_chosen_and_launched", 3000)
    assert sum(s[1][1] > 1 and s[0][2] < 16384 for s in seen) > 100
    for shape, record, need, launches in seen:
        m, n, k = shape
        _, split, waves, rg, mt = record[:5]
        tiles = -(-n // (16 * rg)) * -(-m // (16 * mt))
        assert len(launches) == 1 and "lds_gemm_kernel" in launches[0][0], (shape, record, launches)
        assert launches[0][1:3] == [tiles * split, 64 * waves], (shape, record, launches)
        assert need == (65536 + tiles * split * rg * mt * 1024 if split > 1 else 0), (shape, record, need)


def records_at_the_edges(rec):
    """K splits of the choice on either side of the ranges that were timed"""
    record, out = (C.c_int * 10)(), []
    for m, n, k in [(2048, 128, 6144), (2049, 128, 6144), (915, 188, 32768), (915, 188, 32784), (1024, 8192, 8192 + 128)]:
        assert rec.call("sg_skinny_gemm_choice", m, n, k, record, None) == 0
        out.append(record[1])
    return out


def test_nothing_beyond_the_timed_ranges(fake):
    at = launch_recorder.scenario(fake, "test_deep_split_choice", "records_at_the_edges")
    assert at[0] > 1 and at[1] == 1 and at[2] > 4 and at[3] == 2 and at[4] == 1, at    # (2: the record's own)


def without_room_for_partials(rec):
    out = []
    rec.fake.rec_largest_allocation(1 << 12)
    for m, n, k in UNSPLIT_RECORDS + [(130, 160, 11904), (92, 316, 12416)]:
        out.append(rec.of("sg_skinny_gemm_auto", rec.A, rec.B, rec.D, rec.S, m, n, k, k, None))
        out.append(rec.of("sg_skinny_gemm_auto_ws", rec.A, rec.B, rec.D, rec.S, m, n, k, k, None, C.c_size_t(0), None))
    return out


def test_the_record_runs_where_there_is_no_room_for_the_partials(fake):
    """... and a caller who brings no workspace, as the record without a K split let it, is not refused"""
    for rc, launches in launch_recorder.scenario(fake, "test_deep_split_choice", "without_room_for_partials"):
        assert rc == 0 and len(launches) == 1 and "_gemm_kernel" in launches[0][0] and "line" not in launches[0][0], (rc, launches)
