"""Entry points that promise the library's own choice launch the same kernels with the same grids (no GPU: the calls run on a
stand-in for the runtime)."""
import ctypes as C
import random

import launch_recorder
import pytest


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return launch_recorder.build(tmp_path_factory.mktemp("fake"))


def _shapes(count, seed):
    """Every row count the entry points take, half of the shapes off their 128-byte lines by k, by the row stride or by both."""
    r = random.Random(seed)
    for _ in range(count):
        m = int(33 * 31 ** r.random()) if r.random() < 0.75 else r.randint(1, 32)
        n, k = 2 * int(16 * 2000 ** r.random()), 16 * int(1 + 1500 ** r.random())
        if r.random() < 0.5:
            k = max(128, k // 128 * 128)
        yield m, n, k, k + r.choice([0, 0, 16, 112, 128])


def _gemms(launches):
    return [x for x in launches if "fill_zero" not in x[0]]


def engine_0_and_auto(rec, count):
    """[shape, launches of the one, of the other] where they differ, and what kernels there were"""
    own_choice, differ, kernels = (C.c_int * 10)(), [], {}
    for m, n, k, stride in _shapes(count, 1):
        rc, auto = rec.of("sg_skinny_gemm_auto", rec.A, rec.B, rec.D, rec.S, m, n, k, stride, None)
        rc2, own = rec.of("sg_skinny_gemm_tuned", rec.A, rec.B, rec.D, rec.S, m, n, k, stride, own_choice, None)
        assert rc == rc2 == 0, (m, n, k, stride, rc, rc2)
        if _gemms(auto) != _gemms(own):
            differ.append([(m, n, k, stride), _gemms(auto), _gemms(own)])
        name = _gemms(auto)[0][0].split("sg::")[1].split("<")[0]
        kernels[name] = kernels.get(name, 0) + 1
    return differ, kernels


def test_engine_0_of_the_tuned_entry_point_is_the_librarys_choice(fake):
    differ, kernels = launch_recorder.scenario(fake, "test_launch_choice", "engine_0_and_auto", 3000)
    assert not differ, (len(differ), differ[:3])
    assert all(kernels.get(name, 0) > 20 for name in ("line_gemm_kernel", "mid_gemm_kernel", "wide_gemm_kernel", "lds_gemm_kernel")), kernels


def noalloc_and_auto(rec, count):
    """The same of sg_skinny_gemm_tuned_noalloc with engine 0, on shapes whose partials fit its array; large weight matrices too"""
    own_choice, differ, seen, r = (C.c_int * 10)(), [], 0, random.Random(3)
    need = C.c_size_t()
    shapes = list(_shapes(count, 2))
    shapes += [(r.randint(33, 768), 2 * r.randint(15000, 400000), k, stride) for _, _, k, stride in _shapes(count, 4)]
    for m, n, k, stride in shapes:
        assert rec.call("sg_workspace_query", m, n, k, C.byref(need)) == 0
        if need.value > 65536 + (8 << 20):
            continue
        seen += 1
        rc, auto = rec.of("sg_skinny_gemm_auto", rec.A, rec.B, rec.D, rec.S, m, n, k, stride, None)
        rc2, own = rec.of("sg_skinny_gemm_tuned_noalloc", rec.A, rec.B, rec.D, rec.S, m, n, k, stride, own_choice, None)
        assert rc == rc2 == 0, (m, n, k, stride, rc, rc2)
        if _gemms(auto) != _gemms(own):
            differ.append([(m, n, k, stride), _gemms(auto), _gemms(own)])
    return differ, seen


def test_the_fixed_array_changes_no_launch_that_fits_it(fake):
    differ, seen = launch_recorder.scenario(fake, "test_launch_choice", "noalloc_and_auto", 3000)
    assert not differ, (len(differ), differ[:3])
    assert seen > 3000


def without_room_for_partials(rec):
    """Launches where the device has no memory left for a workspace, of both entry points that would allocate one"""
    own_choice, out = (C.c_int * 10)(), []
    rec.fake.rec_largest_allocation(1 << 20)
    for m, n, k in UNSPLIT_RECORDS:
        out.append(rec.of("sg_skinny_gemm_auto", rec.A, rec.B, rec.D, rec.S, m, n, k, k, None))
        out.append(rec.of("sg_skinny_gemm_tuned", rec.A, rec.B, rec.D, rec.S, m, n, k, k, own_choice, None))
    return out


# shapes whose heuristic record has no K split where the kernel for rows off their lines takes one
UNSPLIT_RECORDS = [(100, 2374, 5456), (190, 940, 7600), (468, 566, 9200)]


def test_a_split_that_stands_in_for_an_unsplit_launch_is_left_where_no_workspace_can_be_had(fake):
    for rc, launches in launch_recorder.scenario(fake, "test_launch_choice", "without_room_for_partials"):
        assert rc == 0 and len(launches) == 1 and "line_gemm" not in launches[0][0], (rc, launches)
