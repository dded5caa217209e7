"""Host threads that call the library on one stream: the launches of one call that hand each other memory of the stream's -
a GEMM and the sum of its K split's partials, the row encoder and the GEMM on its codes - stay together (no GPU: the calls
run on a stand-in for the runtime, on which every launch takes long enough for another thread to get in between)."""
import ctypes as C
import threading

import launch_recorder
import pytest

THREADS, CALLS = 3, 6
# second launches that a first one has to be followed by, on the same thread
SECOND = {"line": "mid_reduce_kernel", "mid": "mid_reduce_kernel", "wide": "mid_reduce_kernel", "bf16act": "gemm"}
# m, n, k, row stride (the 2304 x 20864 one is a mid-batch record summed by a second launch, the 28672-column ones are too)
SHAPES = {"line": (96, 4828, 11984, 11984), "mid": (128, 8192, 28672, 28672), "wide": (640, 3584, 8192, 8192),
          "bf16act": (16, 4096, 4096, 4096), "one launch": (8, 1024, 14336, 14336)}


def _first(kind, kernel):
    return {"line": "line_gemm", "mid": "mid_gemm", "wide": "wide_gemm", "bf16act": "encode"}[kind] in kernel


def threads_on_one_stream(rec, kinds, entry):
    """kinds[i % len(kinds)] on thread i, through `entry`; [[kernel, thread]] in the order of the launches"""
    rec.fake.rec_pause(400)
    start = threading.Barrier(THREADS)
    own_choice = (C.c_int * 10)()
    codes = []

    def work(kind):
        m, n, k, stride = SHAPES[kind]
        start.wait()
        for _ in range(CALLS):
            if kind == "bf16act":
                codes.append(rec.call("sg_skinny_gemm_bf16act", rec.A, rec.B, rec.D, rec.S, None, None, m, n, k, stride, None))
            elif entry == "auto_ws":
                codes.append(rec.call("sg_skinny_gemm_auto_ws", rec.A, rec.B, rec.D, rec.S, m, n, k, stride, rec.WS, 1 << 30, None))
            elif entry == "noalloc":
                codes.append(rec.call("sg_skinny_gemm_tuned_noalloc", rec.A, rec.B, rec.D, rec.S, m, n, k, stride, own_choice, None))
            else:
                codes.append(rec.call("sg_skinny_gemm_auto", rec.A, rec.B, rec.D, rec.S, m, n, k, stride, None))

    threads = [threading.Thread(target=work, args=(kinds[i % len(kinds)],)) for i in range(THREADS)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert codes == [0] * (THREADS * CALLS), codes
    return [[x[0], x[4]] for x in rec.launches() if "fill_zero" not in x[0]]


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return launch_recorder.build(tmp_path_factory.mktemp("fake"))


@pytest.mark.parametrize("kinds,entry", [(["line"], "auto"), (["mid"], "auto"), (["wide"], "auto"), (["line", "mid", "wide"], "auto"),
                                         (["line", "one launch"], "auto"), (["bf16act"], "auto"), (["bf16act", "line"], "auto"),
                                         (["line", "mid"], "auto_ws"), (["line"], "noalloc")])
def test_the_launches_of_a_call_stay_together(fake, kinds, entry):
    launches = launch_recorder.scenario(fake, "test_launch_order", "threads_on_one_stream", kinds, entry)
    assert len({t for _, t in launches}) == THREADS
    pairs = 0
    for kind in kinds:
        if kind not in SECOND:
            continue
        for i, (kernel, thread) in enumerate(launches):
            if _first(kind, kernel):
                assert i + 1 < len(launches) and launches[i + 1][1] == thread and SECOND[kind] in launches[i + 1][0], launches[i:i + 2]
                pairs += 1
    assert pairs >= CALLS
