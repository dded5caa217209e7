"""Where sg_skinny_gemm_bf16act_choice says that the fused kernel runs, it runs, whatever the row stride, and takes no memory of its
stream's (no GPU: the calls run on a stand-in for the runtime)."""
import ctypes as C
import random

import launch_recorder
import pytest


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return launch_recorder.build(tmp_path_factory.mktemp("fake"))


def launches_of(rec, fused, count):
    """[shape, launches eagerly, recorded] where the choice says `fused`, and allocations of all the calls"""
    r, out, said, record = random.Random(7), [], C.c_int(), (C.c_int * 10)()
    shapes = [(8, 28672, 4096, 16), (4, 28672, 4096, 16), (8, 57344, 4096, 16), (8, 28672, 4096, 0), (8, 28672, 4096, 128), (16, 28672, 4096, 16)]
    for _ in range(count):
        shapes.append((r.randint(1, 9), 2 * int(3000 * 12 ** r.random()), 256 * r.randint(1, 33) + 16 * (r.random() < 0.2), 16 * r.randint(0, 8)))
    for m, n, k, pad in shapes:
        assert rec.call("sg_skinny_gemm_bf16act_choice", m, n, k, record, C.byref(said)) == 0
        if said.value != fused:
            continue
        calls = []
        for capturing in (0, 1):
            rec.fake.rec_capturing(capturing)
            rc, launches = rec.of("sg_skinny_gemm_bf16act", rec.A, rec.B, rec.D, rec.S, rec.COL, None, m, n, k, k + pad, None)
            assert rc == 0, (m, n, k, pad)
            calls.append([x for x in launches if "fill_zero" not in x[0]])
        out.append([(m, n, k, k + pad), *calls])
    return out, rec.fake.rec_allocations()


def test_the_fused_kernel_is_one_launch_without_memory_of_the_streams(fake):
    seen, allocations = launch_recorder.scenario(fake, "test_bf16act_choice", "launches_of", 1, 1500)
    assert len(seen) > 300 and sum(s[0][3] % 128 != 0 for s in seen) > 200
    for shape, eager, recorded in seen:
        assert eager == recorded and len(eager) == 1 and "lds_gemm_persistent_kernel" in eager[0][0], (shape, eager, recorded)
    assert allocations == 0


def test_elsewhere_the_encoder_goes_first(fake):
    seen, _ = launch_recorder.scenario(fake, "test_bf16act_choice", "launches_of", 0, 300)
    assert len(seen) > 100
    for shape, *calls in seen:
        assert all(len(c) >= 2 and "encode" in c[0][0] for c in calls), (shape, calls)
