#!/usr/bin/env python3
"""Benchmark of the FP8 skinny-GEMM hot path on one MI355X.

A *step* is one decode layer's worth of projections at M = 8 on the Llama-3-8B shapes
(QKV 6144x4096, O 4096x4096, gate_up 28672x4096, down 4096x14336): four dense FP8 GEMMs
with E4M3 operands from N(0,1), per-tensor scales, fp32 accumulation and bf16 output.
Weights are COLD: every shape rotates through enough distinct weight buffers that more
than 2x the 256 MB memory-side cache passes between two uses of the same buffer.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-sweep] [--no-cpu]

prints one JSON line.  `value` is the achieved HBM throughput of the whole step
(algorithmic bytes of the four GEMMs / step time, inputs resident in HBM), in TB/s.
`roofline` is for the dominant kernel (the gate_up GEMM): back-to-back launches on cold
weights inside one HIP event pair on the launch stream; `cpu_baseline` is the CPU oracle (all cores) on the same step.
`sweep` lists us/GEMM and TB/s for every shape and M in {1,2,4,8,16,32}.
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

SHAPES = {"qkv": (6144, 4096), "o": (4096, 4096), "gate_up": (28672, 4096), "down": (4096, 14336)}
M_SWEEP = (1, 2, 4, 8, 16, 32)
HBM_PEAK_GBS = 8000.0
COLD_BYTES = 640e6          # per shape: distinct weight bytes cycled through (> 2x the 256 MB cache)
# HBM bytes per launch of the dominant kernel (gate_up, M = 8), measured off-line with two
# rocprofv3 --pmc runs (FETCH_SIZE x 1.9998, WRITE_SIZE x 1.0, factors from a 256 MiB copy);
# the runs and their arithmetic are in profiles/dense_gemm_decode_step_m8_pmc_traffic.md
RECORDED_TRAFFIC = {"bytes": 118344281, "source": "profiles/dense_gemm_decode_step_m8_pmc_traffic.md",
                    # the kernel configuration the counters were read on; another configuration reports no traffic
                    "tuning": {"engine": 2, "waves": 8, "row_tiles": 1, "depth": 2, "persistent_wgs_per_cu": 1, "wave_tiles": 6}}


def gemm_bytes(m, n, k):
    """Algorithmic bytes of one dense GEMM: fp8 A + fp8 B + bf16 D."""
    return k * (m + n) + 2 * m * n


def unrecorded_launch(sg, m, n, k):
    """What the library launches for the shape where no tuning record describes it, or None."""
    wide, line = sg.api.skinny_gemm_wide_choice(m, n, k), sg.api.skinny_gemm_line_choice(m, n, k)
    if wide:
        return "wide tile %d x %d, K split %d" % (32 * wide[0], 32 * wide[1], wide[2])
    if line:
        return "rows off their lines, tile %d x %d, K split %d" % (8 * line[0] * line[1], 32 * line[2], line[3])
    skinny = sg.api.skinny_gemm_skinny_line_choice(m, n, k)
    if skinny:
        return "rows off their lines, %d waves, %d rows, %d slots, K split %d%s" % (
            skinny[0], 16 * skinny[1], skinny[2], skinny[3], ", activations resident" if skinny[4] else "")
    return None


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--m", type=int, default=8, help="activation rows of the timed step")
    ap.add_argument("--random-codes", action="store_true",
                    help="fill the operands with uniformly random E4M3 codes from torch's generator (one kernel per buffer) "
                         "instead of the seeded N(0,1) recipe (dozens of elementwise kernels per buffer): for profiler runs "
                         "that serialise every dispatch; timings of such a run are not the benchmark's")
    ap.add_argument("--tuning", help="tuning table to load first (sg_tuning_load): every mode then runs the table's records")
    ap.add_argument("--replays", type=int, default=31, help="timed regions per measurement (the median is reported)")
    ap.add_argument("--no-sweep", action="store_true")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-warm", action="store_true", help="skip the cache-resident (same weight buffer) timings")
    ap.add_argument("--no-graph", action="store_true", help="launch eagerly instead of replaying HIP graphs (for counter runs)")
    ap.add_argument("--calibration-copy", action="store_true",
                    help="also run three 256 MiB device-to-device copies (known traffic, to scale profiler counters)")
    ap.add_argument("--launch-shapes", nargs="+", metavar="MxNxK",
                    help="launch the library's own choice for each dense shape three times, eagerly, on rotating cold weight "
                         "buffers, and exit (for kernel traces and counters of any shape; prints the chosen records)")
    ap.add_argument("--record", nargs=10, type=int, metavar="INT",
                    help="with --launch-shapes: launch this tuning record (the ten SgTuning fields: engine split_k waves "
                         "row_tiles m_blocks depth k_chunks non_temporal persistent_wgs_per_cu wave_tiles) for every shape "
                         "instead of the library's own choice")
    ap.add_argument("--several-tiles-counters", action="store_true",
                    help="more than 32 rows on small weight matrices (the skinny ring over several 32-row activation tiles): "
                         "launch the library's choice three times each on cold weights and exit (for HBM-traffic counters)")
    ap.add_argument("--mid-batch-counters", action="store_true",
                    help="only launch the mid-batch GEMMs (M = 64, 128, 256), eagerly, three times each, and exit "
                         "(for MFMA-utilisation counter runs; prints no JSON line)")
    ap.add_argument("--decode-counters", action="store_true",
                    help="only launch the decode-sweep GEMMs (four projection shapes x M = 1, 8, 32), eagerly, three "
                         "times each on cold weights, after three 256 MiB copies of known traffic, and exit "
                         "(for HBM-traffic counter runs; prints no JSON line)")
    ap.add_argument("--sparse-counters", action="store_true",
                    help="only launch the 2:4 GEMMs (14336 x 4096 and 28672 x 4096 at M = 8, 16; then 4096 x 14336 at M = 8, 16, 32 through the library's choice only), eagerly, three times each "
                         "on cold weights through the library's choice and three times through the one-wave-workgroup kernel "
                         "it replaced, after three 256 MiB copies of known traffic (for L2 / HBM traffic counter runs); then "
                         "graph-times K = 4224, 4480, 14464, 14720 - whole 128-k pieces that 512 does not divide - next to "
                         "the neighbouring multiples of 512 and prints that table; no JSON line")
    ap.add_argument("--sparse-metadata-fetch", action="store_true",
                    help="only compare the two ways the 2:4 kernels fetch their metadata on the 4096 x 14336 and 14336 x 4096 "
                         "shapes at M = 1, 8, 16, 32: by 64-byte pieces per row and stage, and by whole 128-byte lines per "
                         "row and pair of stages; three eager launches of each on cold weights (for L1 -> L2 request "
                         "counters), then alternating graph replays; prints a table, no JSON line")
    ap.add_argument("--k-tail-counters", action="store_true",
                    help="K that 256 does not divide: launch the library's choice (LDS ring with a partly used last stage) and the "
                         "register-streaming engine it replaced three times each on cold weights, next to the neighbouring "
                         "multiple of 256, and exit (for kernel traces and HBM-traffic counters)")
    ap.add_argument("--n-sweep", action="store_true",
                    help="only run 8 x N x 4096 for N = 4096 ... 57344 (1 ... 14 sixteen-row tiles per CU): the library's own "
                         "choice, the per-tile kernel (one wave, eight slots) and the read-only streaming yardstick "
                         "(sg_debug_read_stream), graph-timed on cold weights and then ten eager launches each (for a kernel "
                         "trace); prints a table and the straight-line fit fixed + bytes / rate, no JSON line")
    ap.add_argument("--codec-counters", action="store_true",
                    help="only launch the 8192 x 8192 row codec (encode, decode, reduce of 8), the fp32 batch sum "
                         "(8 x 1024 x 8192) and the read-only streaming yardstick on 28672 x 4096 three times each, eagerly, "
                         "after three 256 MiB copies of known traffic, and exit (for kernel traces and HBM-traffic counters)")
    ap.add_argument("--ring-ab", action="store_true",
                    help="only compare the producer/consumer ring (sg_skinny_gemm with producers > 0, best record of a sweep "
                         "over producers x consumers x b_lanes x qsize) with the library's own choice on the four projection "
                         "shapes at M = 8 and 32, cold weights; then launch each winner and each own choice ten times eagerly "
                         "(for a kernel trace); prints a table, no JSON line")
    ap.add_argument("--cu-ingest", action="store_true",
                    help="only run the ingest probe (sg_debug_cu_ingest): what a CU takes in through direct-to-LDS loads from "
                         "beyond its XCD's L2 (cold), from inside it (hot), and from both at once out of the same or out of "
                         "different waves, with 16 and with 256 workgroups; prints a table, no JSON line")
    ap.add_argument("--wide-against-mid", type=int, metavar="COUNT",
                    help="only time COUNT seeded random shapes (129..2048 rows) that the library runs on a wide tile against the "
                         "mid-batch record the tile replaces, in alternating rounds on cold weights; prints a table, no JSON line")
    ap.add_argument("--sparse", action="store_true",
                    help="with --stamps --launch-shapes: the 2:4 GEMM (sg_sparse24_gemm on weights pruned and compressed here) "
                         "instead of the dense one")
    ap.add_argument("--stamps", action="store_true",
                    help="only run the decode GEMMs (four projection shapes at M = --m) back to back from a HIP graph with "
                         "the library's per-workgroup time stamps switched on, and print where a launch period goes "
                         "(launch gap, prologue, first data, streaming, epilogue); prints no JSON line")
    args = ap.parse_args()
    if args.gpus != 1:
        sys.exit("bench.py: this build runs on exactly one GPU (no collectives, no sharding); use --gpus 1")

    import torch

    import rocm_dev_amd as sg
    from rocm_dev_amd._lib import lib

    assert torch.cuda.is_available(), "bench.py needs a GPU"
    torch.cuda.set_device(0)
    torch.manual_seed(0)
    if lib.sg_init() != 0:
        sys.exit("bench.py: sg_init failed")
    if args.tuning and lib.sg_tuning_load(args.tuning.encode()) != 0:
        sys.exit("bench.py: cannot load tuning table %s" % args.tuning)

    if args.cu_ingest:
        cold = torch.ones(4 << 30, device="cuda", dtype=torch.uint8)
        hot = torch.ones(8 << 20, device="cuda", dtype=torch.uint8)       # 1 MB per XCD: stays in its 4 MB L2
        counts = torch.zeros(2, device="cuda", dtype=torch.int64)
        ticks = 30000                                                      # 300 us per measurement

        def probe(wgs, waves, cold_waves, hot_per_cold, depth):
            for timed in (False, True):
                counts.zero_()
                rc = lib.sg_debug_cu_ingest(cold.data_ptr(), cold.numel(), hot.data_ptr(), hot.numel(), wgs, waves, cold_waves,
                                            hot_per_cold, depth, ticks if timed else 3000, counts.data_ptr(), None)
                if rc != 0:
                    raise RuntimeError("sg_debug_cu_ingest: %s" % sg.strerror(rc))
                torch.cuda.synchronize()
            c, h = (int(v) for v in counts.cpu())
            per_cu = 1024.0 / wgs / (ticks * 10e-9) / 1e9                  # GB/s per CU and instruction counted
            return c * per_cu, h * per_cu

        print("direct-to-LDS loads, 1 KB each (8 rows x 128 B), for 300 us; GB/s per CU (x workgroups = chip-wide TB/s)")
        print("cold = a region of its own per wave (L2 misses), hot = a 1 MB window per XCD shared by its workgroups (L2 hits)")
        print("| workgroups | waves x loads in flight | stream | cold GB/s | hot GB/s | sum | chip-wide TB/s | cold / cold alone + hot / hot alone |")
        print("|---|---|---|---|---|---|---|---|")
        for wgs in (16, 256):
            for waves, depth in ((4, 8), (8, 8), (16, 8)):
                alone_c, _ = probe(wgs, waves, waves, 0, depth)
                _, alone_h = probe(wgs, waves, 0, 0, depth)
                cases = [("all waves cold", waves, 0), ("all waves hot", 0, 0), ("every wave 1 hot : 1 cold", -1, 1),
                         ("every wave 3 hot : 1 cold", -1, 3), ("every wave 7 hot : 1 cold", -1, 7),
                         ("half of the waves cold, half hot", waves // 2, 0), ("a quarter of the waves cold, the others hot", waves // 4, 0)]
                for name, cw, hpc in cases:
                    c, h = probe(wgs, waves, cw, hpc, depth)
                    print("| %d | %d x %d | %s | %.1f | %.1f | %.1f | %.2f | %.2f |"
                          % (wgs, waves, depth, name, c, h, c + h, (c + h) * wgs / 1e3, c / alone_c + h / alone_h), flush=True)
        return

    if args.n_sweep:
        import ctypes
        import numpy as np
        from rocm_dev_amd import synth
        side = torch.cuda.Stream()
        m, k = 8, 4096
        one = torch.ones(1, device="cuda")
        a8 = synth.quantize_tensor(synth.normal_f32((m, k), 0, 1))[0]
        per_tile = sg.SgTuning(2, 1, 1, 1, 1, 8, 4, 1, 0, 0)

        def graph_us(fn, reps=24, replays=9):
            with torch.cuda.stream(side):
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g, stream=side):
                    st = torch.cuda.current_stream().cuda_stream
                    for i in range(reps):
                        if fn(i, st) != 0:
                            raise RuntimeError("launch failed")
                ts = []
                for r in range(replays + 3):
                    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                    a.record()
                    g.replay()
                    b.record()
                    torch.cuda.synchronize()
                    if r >= 3:
                        ts.append(a.elapsed_time(b) * 1e3 / reps)
            return sorted(ts)[len(ts) // 2]

        print("8 x N x 4096, cold weights, us per launch (median of 9 graph replays of 24 launches)")
        print("| N | tiles per CU | MB per launch | own choice | per-tile kernel (1 wave x 8 slots) | read-only yardstick |")
        print("|---|---|---|---|---|---|")
        xs, own_t, tile_t, read_t = [], [], [], []
        for n in (4096, 8192, 12288, 16384, 20480, 24576, 28672, 32768, 40960, 57344):
            copies = max(3, int(COLD_BYTES // (n * k)) + 1)
            wb = [synth.quantize_tensor(synth.normal_f32((n, k), c, 2))[0] for c in range(copies)]
            d = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)
            fns = (lambda i, st: lib.sg_skinny_gemm_auto(a8.data_ptr(), wb[i % copies].data_ptr(), d.data_ptr(), one.data_ptr(), m, n, k, k, st),
                   lambda i, st: lib.sg_skinny_gemm_tuned(a8.data_ptr(), wb[i % copies].data_ptr(), d.data_ptr(), one.data_ptr(), m, n, k, k,
                                                          ctypes.byref(per_tile), st),
                   lambda i, st: lib.sg_debug_read_stream(wb[i % copies].data_ptr(), n, k, k, 256, st))
            t = [graph_us(f) for f in fns]
            mb = gemm_bytes(m, n, k) / 1e6
            print("| %d | %.1f | %.1f | %.2f | %.2f | %.2f |" % (n, n / 16 / 256, mb, t[0], t[1], t[2]), flush=True)
            xs.append(mb); own_t.append(t[0]); tile_t.append(t[1]); read_t.append(t[2])
            for f in fns:                      # ten eager launches each, for rocprofv3 --kernel-trace
                for i in range(10):
                    f(i, None)
                torch.cuda.synchronize()
            del wb
        for label, ys in (("own choice", own_t), ("per-tile kernel", tile_t), ("read-only yardstick", read_t)):
            slope, fixed = np.polyfit(np.array(xs), np.array(ys), 1)
            print("%s: %.2f us fixed + bytes / %.2f TB/s (least squares over the ten sizes)" % (label, fixed, 1.0 / slope))
        return

    if args.codec_counters:
        from rocm_dev_amd import synth
        src = torch.empty(256 << 20, device="cuda", dtype=torch.uint8)
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        rows = cols = 8192
        xs = [synth.normal_f32((rows, cols), i, 3).bfloat16() for i in range(3)]
        q8 = torch.empty((8, rows, cols), device="cuda", dtype=torch.uint8)
        s8 = torch.empty((8, rows), device="cuda", dtype=torch.float32)
        y = torch.empty((rows, cols), device="cuda", dtype=torch.bfloat16)
        for i in range(8):
            lib.sg_fp8_encode_rows(xs[i % 3].data_ptr(), q8[i].data_ptr(), s8[i].data_ptr(), rows, cols, None)
        torch.cuda.synchronize()
        for i in range(3):
            lib.sg_fp8_encode_rows(xs[i].data_ptr(), q8[i].data_ptr(), s8[i].data_ptr(), rows, cols, None)
        torch.cuda.synchronize()
        for i in range(3):
            lib.sg_fp8_decode_rows(q8[3 + i].data_ptr(), s8[3 + i].data_ptr(), y.data_ptr(), rows, cols, None)
        torch.cuda.synchronize()
        for i in range(3):
            lib.sg_fp8_reduce_rows(q8.data_ptr(), s8.data_ptr(), y.data_ptr(), 8, rows * cols, rows, cols, None)
        torch.cuda.synchronize()
        del xs, q8, s8, y
        tb, tm, tn = 8, 1024, 8192
        ta = synth.normal_f32((tb, tm, tn), 0, 4)
        tbb = synth.normal_f32((tb, tm, tn), 0, 5)
        td = torch.empty((tm, tn), device="cuda", dtype=torch.float32)
        for i in range(3):
            lib.sg_tiled_sum_reduce(ta.data_ptr(), tbb.data_ptr(), td.data_ptr(), tb, tm, tn, None)
        torch.cuda.synchronize()
        del ta, tbb, td
        n, k = SHAPES["gate_up"]
        wb = [synth.quantize_tensor(synth.normal_f32((n, k), c, 2))[0] for c in range(6)]
        for i in range(6):
            lib.sg_debug_read_stream(wb[i].data_ptr(), n, k, k, 256, None)
        torch.cuda.synchronize()
        return

    if args.ring_ab:
        import itertools
        from rocm_dev_amd import autotune, synth
        side = torch.cuda.Stream()

        def time_us(fn, reps=20, replays=7):
            with torch.cuda.stream(side):
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g, stream=side):
                    st = torch.cuda.current_stream().cuda_stream
                    for i in range(reps):
                        if fn(i, st) != 0:
                            return None
                ts = []
                for r in range(replays + 2):
                    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                    a.record()
                    g.replay()
                    b.record()
                    torch.cuda.synchronize()
                    if r >= 2:
                        ts.append(a.elapsed_time(b) * 1e3 / reps)
            return sorted(ts)[len(ts) // 2]

        print("producer/consumer ring against the library's own choice; us per launch, median of 7 graph replays of 20 "
              "launches on cold weights")
        print("| shape | M | own choice (us) | best ring record (us) | ring / own | ring record: A producers, B producers, "
              "consumers, b_lanes, qsize |")
        print("|---|---|---|---|---|---|")
        eager = []
        for name, (n, k) in SHAPES.items():
            copies = max(3, int(COLD_BYTES // (n * k)) + 1)
            wb = [synth.quantize_tensor(synth.normal_f32((n, k), c, 2))[0] for c in range(copies)]
            one = torch.ones(1, device="cuda")
            for m in (8, 32):
                a8 = synth.quantize_tensor(synth.normal_f32((m, k), 0, 1))[0]
                d = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)
                op_m = 8 if m <= 8 else (16 if m <= 16 else 32)
                ops = 256 // (512 // op_m)
                own = time_us(lambda i, st: lib.sg_skinny_gemm_auto(a8.data_ptr(), wb[i % copies].data_ptr(), d.data_ptr(),
                                                                    one.data_ptr(), m, n, k, k, st))
                best = (1e30, None)
                for ap_, bp, cons, bl, qs in itertools.product((1, 2), (2, 4, 6, 8), (1, 2, 3, 4), (1, 2, 4), (2, 3, 4, 6, 8)):
                    if ap_ + bp + cons > 16 or qs < max(ap_, bp // bl, cons) or not autotune.pc_ring_fits(m, k, ap_, bp, cons, bl, qs):
                        continue
                    t = time_us(lambda i, st: lib.sg_skinny_gemm(a8.data_ptr(), wb[i % copies].data_ptr(), d.data_ptr(),
                                                                 one.data_ptr(), m, n, k, k, 1, ap_, bp, cons, bl, qs, op_m, ops, st),
                                reps=10, replays=3)
                    if t is not None and t < best[0]:
                        best = (t, (ap_, bp, cons, bl, qs))
                ap_, bp, cons, bl, qs = best[1]
                ring = time_us(lambda i, st: lib.sg_skinny_gemm(a8.data_ptr(), wb[i % copies].data_ptr(), d.data_ptr(),
                                                                one.data_ptr(), m, n, k, k, 1, ap_, bp, cons, bl, qs, op_m, ops, st))
                print("| %s %d x %d | %d | %.2f | %.2f | %.2f | %d, %d, %d, %d, %d |"
                      % (name, n, k, m, own, ring, ring / own, ap_, bp, cons, bl, qs), flush=True)
                eager.append((name, m, a8, d, best[1], op_m, ops))
            # ten eager launches of each (for rocprofv3 --kernel-trace --stats): the own choice, then the ring
            for (nm, m, a8, d, rec, op_m, ops) in [e for e in eager if e[0] == name]:
                for i in range(10):
                    lib.sg_skinny_gemm_auto(a8.data_ptr(), wb[i % copies].data_ptr(), d.data_ptr(), one.data_ptr(), m, n, k, k, None)
                for i in range(10):
                    lib.sg_skinny_gemm(a8.data_ptr(), wb[i % copies].data_ptr(), d.data_ptr(), one.data_ptr(), m, n, k, k, 1,
                                       rec[0], rec[1], rec[2], rec[3], rec[4], op_m, ops, None)
                torch.cuda.synchronize()
            del wb
        return

    if args.wide_against_mid:
        import math
        import random
        from rocm_dev_amd import autotune
        rng = random.Random(0)
        sg.tuning_clear()
        ratios = []
        print("| M x N x K | wide tile (split) | us | mid-batch record: tile (split) | us | ratio |\n|---|---|---|---|---|---|")
        while len(ratios) < args.wide_against_mid:
            m, n, k = (int(lo * (hi / lo) ** rng.random()) for lo, hi in ((129, 2049), (256, 60000), (256, 28672)))
            step = 128 if rng.random() < 0.5 else 16          # every other one with whole K blocks and whole groups of columns
            n, k = n // (64 if step == 128 else 2) * (64 if step == 128 else 2), k // step * step
            if k <= 128 or n < 256 or n * k > 400 << 20 or 2 * m * n * k > 4e11 or not sg.api.skinny_gemm_wide_choice(m, n, k):
                continue
            rg, mb, split = sg.api.skinny_gemm_wide_choice(m, n, k)
            mid, _ = sg.skinny_gemm_choice(m, n, k)
            bench = autotune.Bench(m, n, k)
            us = [[], []]
            for _ in range(4):
                for side, t in enumerate((sg.SgTuning(0, 1, 1, 1, 1, 2, 4, 1, 0, 0), mid)):
                    us[side].append(bench.time(lib, t, launches=8, repeats=2))
            wide_us, mid_us = (sorted(v)[1] for v in us)
            ratios.append(wide_us / mid_us)
            print("| %d x %d x %d | %d x %d (%d) | %.2f | %d x %d (%d) | %.2f | %.3f |"
                  % (m, n, k, 32 * rg, 32 * mb, split, wide_us, 8 * mid.row_tiles * mid.waves, 32 * mid.m_blocks, mid.split_k, mid_us,
                     ratios[-1]), flush=True)
            del bench
        print("geometric mean %.3f; %d of %d behind by more than 3 %%, the worst by %.0f %%"
              % (math.exp(sum(map(math.log, ratios)) / len(ratios)), sum(r > 1.03 for r in ratios), len(ratios), 100 * (max(ratios) - 1)))
        return

    if args.stamps:
        import numpy as np
        from rocm_dev_amd import synth as _synth
        quantize = _synth.quantize_tensor       # N(0,1) operands quantised per tensor, as in the timed runs
        one = torch.ones(1, device="cuda")
        reps = 24
        print("in-kernel time stamps, M = %d, graph of %d back-to-back launches on cold weights, medians over launches 4..%d"
              % (args.m, reps, reps - 1))
        print("all times in us; gap = first entry of a launch - last end of the one before; spread = last - first entry")
        side = torch.cuda.Stream()
        # the four decode projections at --m, or the shapes of --launch-shapes MxNxK (each with its own M)
        jobs = [(name, args.m, n, k) for name, (n, k) in SHAPES.items()]
        if args.launch_shapes:
            jobs = [(s, *[int(v) for v in s.lower().split("x")]) for s in args.launch_shapes]
        for name, m_, n, k in jobs:
            args.m = m_
            if args.record and not args.sparse:     # a given tuning record instead of the library's choice
                import ctypes
                forced = sg.SgTuning(*args.record)
                if lib.sg_tuning_set(m_, n, k, ctypes.byref(forced)) != 0:
                    sys.exit("bench.py: --record is not a valid tuning record")
            copies = max(3, int(COLD_BYTES // (n * k)) + 1)
            wb = [quantize(torch.randn((n, k), device="cuda", dtype=torch.float32))[0] for _ in range(copies)]
            if args.sparse:       # 2:4: prune and compress each weight buffer; a "copy" is then 0.625 of its dense bytes
                packed = []
                for w in wb:
                    v = torch.empty((n, k // 2), device="cuda", dtype=torch.uint8)
                    t = torch.empty((n, k // 8), device="cuda", dtype=torch.uint8)
                    if lib.sg_sparse24_compress(w.data_ptr(), v.data_ptr(), t.data_ptr(), n, k, k, None) != 0:
                        raise RuntimeError("sg_sparse24_compress failed")
                    packed.append((v, t))
                torch.cuda.synchronize()
                wb = packed + [(v.clone(), t.clone()) for v, t in packed]
                copies = len(wb)
            a8 = quantize(torch.randn((args.m, k), device="cuda", dtype=torch.float32))[0]
            d = torch.empty((args.m, n), device="cuda", dtype=torch.bfloat16)
            words = reps * 4096 * 8
            buf = torch.zeros(words, device="cuda", dtype=torch.int64)
            torch.cuda.synchronize()
            lib.sg_debug_stamps(buf.data_ptr(), words)
            with torch.cuda.stream(side):
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g, stream=side):
                    st = torch.cuda.current_stream().cuda_stream
                    for i in range(reps):
                        if args.sparse:
                            rc = lib.sg_sparse24_gemm(a8.data_ptr(), wb[i % copies][0].data_ptr(), wb[i % copies][1].data_ptr(),
                                                      d.data_ptr(), one.data_ptr(), args.m, n, k, st)
                        else:
                            rc = lib.sg_skinny_gemm_auto(a8.data_ptr(), wb[i % copies].data_ptr(), d.data_ptr(), one.data_ptr(),
                                                         args.m, n, k, k, st)
                        if rc != 0:
                            raise RuntimeError("%s: %s" % ("sg_sparse24_gemm" if args.sparse else "sg_skinny_gemm_auto", sg.strerror(rc)))
                lib.sg_debug_stamps(None, 0)
                ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                for _ in range(20):
                    g.replay()
                ev0.record()
                g.replay()
                ev1.record()
                torch.cuda.synchronize()
            period_ev = ev0.elapsed_time(ev1) * 1e3 / reps
            raw = buf.cpu().numpy().astype(np.uint64).reshape(-1, 8)
            used = int(np.count_nonzero(raw[:, 0]))
            grid = used // reps
            t = raw[:used].reshape(reps, grid, 8)
            tick = 0.01   # 100 MHz constant clock
            ent, iss, land, cons, end = (t[:, :, i].astype(np.int64) * tick for i in range(5))
            rows = []
            for j in range(4, reps):
                e0 = ent[j].min()
                rows.append({
                    "gap": e0 - end[j - 1].max(), "period": e0 - ent[j - 1].min(), "spread": ent[j].max() - e0,
                    "issue": np.median(iss[j] - ent[j]), "land_med": np.median(land[j] - ent[j]),
                    "land_max": (land[j] - ent[j]).max(), "stream": np.median(cons[j] - land[j]),
                    "epi": np.median(end[j] - cons[j]), "wg_med": np.median(end[j] - ent[j]), "wg_max": (end[j] - ent[j]).max(),
                    "span": end[j].max() - e0, "tail": end[j].max() - np.median(end[j]),
                    "mhz": np.median((t[j, :, 6].astype(np.int64) - t[j, :, 5].astype(np.int64)) / np.maximum(end[j] - ent[j], tick))})
            med = {key: float(np.median([r[key] for r in rows])) for key in rows[0]}
            t_choice, _ = sg.skinny_gemm_choice(args.m, n, k)
            what = ("2:4, the library's choice" if args.sparse else unrecorded_launch(sg, args.m, n, k) or
                    sg.api.tuning_as_dict(t_choice))
            print("%-18s %5d x %5d  grid %4d  event-pair period %.2f | period %.2f = gap %.2f + span %.2f | entry spread %.2f | "
                  "workgroup (median): prologue issue %.2f, first stage landed %.2f (max %.2f), streaming %.2f, reduce+store %.2f, "
                  "total %.2f (max %.2f) | last end - median end %.2f | shader clock %.0f MHz | %s"
                  % (name, n, k, grid, period_ev, med["period"], med["gap"], med["span"], med["spread"], med["issue"], med["land_med"],
                     med["land_max"], med["stream"], med["epi"], med["wg_med"], med["wg_max"], med["tail"], med["mhz"],
                     what), flush=True)
            # does the finish time depend on the XCD?  per XCC_ID: median and latest workgroup end after the launch's first entry
            xcc = (t[4:, :, 7] >> np.uint64(32)).astype(np.int64) & 0xF
            rel_end = end[4:] - ent[4:].min(axis=1, keepdims=True)
            line = []
            for x in sorted(set(xcc.ravel().tolist())):
                sel = rel_end[xcc == x]
                line.append("xcc%d %.2f/%.2f" % (x, float(np.median(sel)), float(np.median(np.where(xcc == x, rel_end, 0).max(axis=1)))))
            print("         workgroup end after first entry, median / median-of-latest per XCD: " + "  ".join(line), flush=True)
            # are the late workgroups the same ones in every launch (their share of the work, their CU) or any (queueing)?
            corr = [float(np.corrcoef(rel_end[j], rel_end[j + 1])[0, 1]) for j in range(rel_end.shape[0] - 1)]
            print("         workgroup end after first entry: median %.2f, 90th percentile %.2f, latest %.2f; correlation of a "
                  "workgroup's end between consecutive launches %.2f"
                  % (float(np.median(rel_end)), float(np.percentile(rel_end, 90)), float(np.median(rel_end.max(axis=1))),
                     float(np.median(corr))), flush=True)
            del wb, buf
        return

    if args.decode_counters:
        one = torch.ones(1, device="cuda")
        src = torch.empty(256 << 20, device="cuda", dtype=torch.uint8)
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        for name, (n, k) in SHAPES.items():
            copies = max(3, int(COLD_BYTES // (n * k)) + 1)
            wb = [torch.randint(0, 0x7E, (n, k), device="cuda", dtype=torch.uint8) for _ in range(copies)]
            for m in (1, 8, 32):
                a8 = torch.randint(0, 0x7E, (m, k), device="cuda", dtype=torch.uint8)
                d = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)
                for i in range(3):
                    w = wb[(3 * (m % 5) + i) % copies]
                    rc = lib.sg_skinny_gemm_auto(a8.data_ptr(), w.data_ptr(), d.data_ptr(), one.data_ptr(), m, n, k, k, None)
                    if rc != 0:
                        raise RuntimeError("sg_skinny_gemm_auto: %s" % sg.strerror(rc))
                torch.cuda.synchronize()
            del wb
        return

    if args.sparse_metadata_fetch:
        import ctypes
        one = torch.ones(1, device="cuda")
        side = torch.cuda.Stream()
        copies = 8
        # the records the library chooses for these shapes (engine, split_k, waves, row_tiles, m_blocks, depth, k_chunks,
        # non_temporal, persistent_wgs_per_cu, wave_tiles), written out so that k_chunks can say how the metadata is
        # fetched: 1 = by pieces, 8 = by lines.  (16 x 14336 x 4096: three slots - four do not fit next to the lines' ring.)
        cases = [(1, 14336, 4096, (2, 1, 1, 1, 1, 2, 0, 1, 0, 0)), (8, 14336, 4096, (2, 1, 4, 1, 1, 4, 0, 1, 1, 1)),
                 (16, 14336, 4096, (2, 1, 4, 1, 1, 3, 0, 1, 1, 1)), (32, 14336, 4096, (2, 1, 1, 2, 2, 2, 0, 1, 0, 0)),
                 (1, 4096, 14336, (2, 1, 2, 1, 1, 4, 0, 1, 0, 0)), (8, 4096, 14336, (2, 1, 2, 1, 1, 4, 0, 1, 0, 0)),
                 (16, 4096, 14336, (2, 1, 2, 1, 1, 4, 0, 1, 0, 0)), (32, 4096, 14336, (2, 1, 2, 1, 2, 3, 0, 1, 0, 0))]
        print("2:4 GEMM, metadata by 64-byte pieces per stage against whole 128-byte lines per pair of stages, us per launch "
              "(cold weights, graphs of %d launches, alternating replays, medians of 12)" % (4 * copies))
        print("| M x N x K | waves, row tiles, slots | pieces | lines | lines / pieces |")
        print("|---|---|---|---|---|")
        weights = {}
        for m, n, k, fields in cases:
            if (n, k) not in weights:
                weights.clear()
                vb, mb = [], []
                for _ in range(copies):
                    dense = torch.randint(0, 0x7E, (n, k), device="cuda", dtype=torch.uint8)
                    v = torch.empty((n, k // 2), device="cuda", dtype=torch.uint8)
                    t = torch.empty((n, k // 8), device="cuda", dtype=torch.uint8)
                    if lib.sg_sparse24_compress(dense.data_ptr(), v.data_ptr(), t.data_ptr(), n, k, k, None) != 0:
                        raise RuntimeError("sg_sparse24_compress failed")
                    vb.append(v)
                    mb.append(t)
                    del dense
                weights[(n, k)] = (vb, mb)
            vb, mb = weights[(n, k)]
            a8 = torch.randint(0, 0x7E, (m, k), device="cuda", dtype=torch.uint8)
            d = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)
            recs = {}
            for kc in (1, 8):
                f = list(fields)
                f[6] = kc
                recs[kc] = sg.SgTuning(*f)

            def launch(kc, i, stream):
                rc = lib.sg_sparse24_gemm_tuned(a8.data_ptr(), vb[i % copies].data_ptr(), mb[i % copies].data_ptr(), d.data_ptr(),
                                                one.data_ptr(), m, n, k, ctypes.byref(recs[kc]), stream)
                if rc != 0:
                    raise RuntimeError("sg_sparse24_gemm_tuned: %s" % sg.strerror(rc))

            for kc in (1, 8):           # for the counters: three cold launches of each
                for i in range(3):
                    launch(kc, 3 * (kc // 8) + i, None)
                torch.cuda.synchronize()
            graphs = {}
            with torch.cuda.stream(side):
                for kc in (1, 8):
                    g = torch.cuda.CUDAGraph()
                    with torch.cuda.graph(g, stream=side):
                        for i in range(4 * copies):
                            launch(kc, i, torch.cuda.current_stream().cuda_stream)
                    graphs[kc] = g
                times = {1: [], 8: []}
                for rep in range(14):
                    for kc in (1, 8):
                        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                        e0.record()
                        graphs[kc].replay()
                        e1.record()
                        torch.cuda.synchronize()
                        if rep >= 2:
                            times[kc].append(e0.elapsed_time(e1) * 1e3 / (4 * copies))
            med = {kc: sorted(v)[len(v) // 2] for kc, v in times.items()}
            print("| %d x %d x %d | %d, %d, %d%s | %.2f | %.2f | %.3f |" % (m, n, k, fields[2], fields[3], fields[5],
                  ", wave per tile" if fields[9] else "", med[1], med[8], med[8] / med[1]), flush=True)
        return

    if args.sparse_counters:
        import ctypes
        one = torch.ones(1, device="cuda")
        src = torch.empty(256 << 20, device="cuda", dtype=torch.uint8)
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        for (n, k) in ((14336, 4096), (28672, 4096)):
            copies = 6
            vb, mb = [], []
            for _ in range(copies):
                dense = torch.randint(0, 0x7E, (n, k), device="cuda", dtype=torch.uint8)
                v = torch.empty((n, k // 2), device="cuda", dtype=torch.uint8)
                t = torch.empty((n, k // 8), device="cuda", dtype=torch.uint8)
                if lib.sg_sparse24_compress(dense.data_ptr(), v.data_ptr(), t.data_ptr(), n, k, k, None) != 0:
                    raise RuntimeError("sg_sparse24_compress failed")
                vb.append(v)
                mb.append(t)
            del dense
            torch.cuda.synchronize()
            for m in (8, 16):
                a8 = torch.randint(0, 0x7E, (m, k), device="cuda", dtype=torch.uint8)
                d = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)
                # engine 0: the library's choice (wave-per-tile, activations resident in LDS);
                # then one-wave workgroups with the activations in every stage, two ring slots
                for rec in (sg.SgTuning(0, 1, 1, 1, 1, 2, 8, 1, 0, 0), sg.SgTuning(2, 1, 1, 1, 1, 2, 8, 1, 0, 0)):
                    for i in range(3):
                        rc = lib.sg_sparse24_gemm_tuned(a8.data_ptr(), vb[(3 * (m // 8) + i) % copies].data_ptr(),
                                                        mb[(3 * (m // 8) + i) % copies].data_ptr(), d.data_ptr(), one.data_ptr(),
                                                        m, n, k, ctypes.byref(rec), None)
                        if rc != 0:
                            raise RuntimeError("sg_sparse24_gemm_tuned: %s" % sg.strerror(rc))
                    torch.cuda.synchronize()
            del vb, mb
        # the long-K shape of the configuration (one 16-row tile per CU): the library's choice at 8, 16 and 32 rows
        n, k = 4096, 14336
        copies = 9
        vb, mb = [], []
        for _ in range(copies):
            dense = torch.randint(0, 0x7E, (n, k), device="cuda", dtype=torch.uint8)
            v = torch.empty((n, k // 2), device="cuda", dtype=torch.uint8)
            t = torch.empty((n, k // 8), device="cuda", dtype=torch.uint8)
            if lib.sg_sparse24_compress(dense.data_ptr(), v.data_ptr(), t.data_ptr(), n, k, k, None) != 0:
                raise RuntimeError("sg_sparse24_compress failed")
            vb.append(v)
            mb.append(t)
        del dense
        torch.cuda.synchronize()
        for j, m in enumerate((8, 16, 32)):
            a8 = torch.randint(0, 0x7E, (m, k), device="cuda", dtype=torch.uint8)
            d = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)
            for i in range(3):
                rc = lib.sg_sparse24_gemm(a8.data_ptr(), vb[3 * j + i].data_ptr(), mb[3 * j + i].data_ptr(), d.data_ptr(),
                                          one.data_ptr(), m, n, k, None)
                if rc != 0:
                    raise RuntimeError("sg_sparse24_gemm: %s" % sg.strerror(rc))
            torch.cuda.synchronize()
        # K that 512 does not divide next to its neighbours: graph-timed on cold weights (prints a table)
        side = torch.cuda.Stream()
        print("2:4 GEMM, K in whole 128-k pieces that 512 does not divide, us per launch (cold weights, graphs of 32 launches)")
        print("| M | N | " + " | ".join("K = %d" % kk for kk in (4096, 4224, 4480, 4608)) + " | N | " +
              " | ".join("K = %d" % kk for kk in (14336, 14464, 14720, 14848)) + " |")
        print("|---|---|---|---|---|---|---|---|---|---|---|")
        for m in (8, 16, 32):
            cells = []
            for n, ks in ((14336, (4096, 4224, 4480, 4608)), (4096, (14336, 14464, 14720, 14848))):
                cells.append(str(n))
                for kk in ks:
                    vb, mb = [], []
                    for _ in range(8):
                        dense = torch.randint(0, 0x7E, (n, kk), device="cuda", dtype=torch.uint8)
                        v = torch.empty((n, kk // 2), device="cuda", dtype=torch.uint8)
                        t = torch.empty((n, kk // 8), device="cuda", dtype=torch.uint8)
                        if lib.sg_sparse24_compress(dense.data_ptr(), v.data_ptr(), t.data_ptr(), n, kk, kk, None) != 0:
                            raise RuntimeError("sg_sparse24_compress failed")
                        vb.append(v)
                        mb.append(t)
                    del dense
                    a8 = torch.randint(0, 0x7E, (m, kk), device="cuda", dtype=torch.uint8)
                    d = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)
                    with torch.cuda.stream(side):
                        g = torch.cuda.CUDAGraph()
                        with torch.cuda.graph(g, stream=side):
                            st = torch.cuda.current_stream().cuda_stream
                            for i in range(32):
                                rc = lib.sg_sparse24_gemm(a8.data_ptr(), vb[i % 8].data_ptr(), mb[i % 8].data_ptr(), d.data_ptr(),
                                                          one.data_ptr(), m, n, kk, st)
                                if rc != 0:
                                    raise RuntimeError("sg_sparse24_gemm: %s" % sg.strerror(rc))
                        ts = []
                        for r in range(12):
                            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                            e0.record()
                            g.replay()
                            e1.record()
                            torch.cuda.synchronize()
                            if r >= 3:
                                ts.append(e0.elapsed_time(e1) * 1e3 / 32)
                    cells.append("%.2f" % sorted(ts)[len(ts) // 2])
                    del vb, mb, g
            print("| %d | " % m + " | ".join(cells) + " |", flush=True)
        return

    if args.launch_shapes:
        one = torch.ones(1, device="cuda")
        if args.calibration_copy:      # what FETCH_SIZE / WRITE_SIZE read for a copy of known size, in the same process
            src = torch.empty(256 << 20, dtype=torch.uint8, device="cuda")
            dst = torch.empty_like(src)
            for _ in range(3):
                dst.copy_(src)
            torch.cuda.synchronize()
            del src, dst
        for spec in args.launch_shapes:
            m, n, k = (int(v) for v in spec.lower().split("x"))
            copies = min(6, max(3, int(COLD_BYTES // (n * k)) + 1))
            from rocm_dev_amd import synth as _synth
            wb = [_synth.quantize_tensor(torch.randn((n, k), device="cuda", dtype=torch.float32))[0] for _ in range(copies)]
            a8 = _synth.quantize_tensor(torch.randn((m, k), device="cuda", dtype=torch.float32))[0]
            d = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)
            if args.record:
                import ctypes
                forced = sg.SgTuning(*args.record)
                if lib.sg_tuning_set(m, n, k, ctypes.byref(forced)) != 0:
                    sys.exit("bench.py: --record is not a valid tuning record")
            t, _ = sg.skinny_gemm_choice(m, n, k)
            print("%s: %s" % (spec, unrecorded_launch(sg, m, n, k) or
                              {f: getattr(t, f) for f in ("engine", "split_k", "waves", "row_tiles", "m_blocks", "depth", "k_chunks",
                                                          "persistent_wgs_per_cu", "wave_tiles")}), file=sys.stderr)
            for i in range(3):
                rc = lib.sg_skinny_gemm_auto(a8.data_ptr(), wb[i % copies].data_ptr(), d.data_ptr(), one.data_ptr(), m, n, k, k, None)
                if rc != 0:
                    raise RuntimeError("sg_skinny_gemm_auto(%s): %s" % (spec, sg.strerror(rc)))
            torch.cuda.synchronize()
            del wb
        return

    if args.several_tiles_counters:
        # more than 32 rows on small weight matrices: the skinny ring over several 32-row activation tiles
        one = torch.ones(1, device="cuda")
        for (m, n, k) in ((64, 4096, 4096), (128, 2048, 4096), (256, 1024, 4096), (128, 4096, 4096)):
            wb = [torch.randint(0, 0x7E, (n, k), device="cuda", dtype=torch.uint8) for _ in range(24)]
            a8 = torch.randint(0, 0x7E, (m, k), device="cuda", dtype=torch.uint8)
            d = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)
            for i in range(3):
                rc = lib.sg_skinny_gemm_auto(a8.data_ptr(), wb[i].data_ptr(), d.data_ptr(), one.data_ptr(), m, n, k, k, None)
                if rc != 0:
                    raise RuntimeError("sg_skinny_gemm_auto: %s" % sg.strerror(rc))
            torch.cuda.synchronize()
            del wb
        return

    if args.k_tail_counters:
        import ctypes
        one = torch.ones(1, device="cuda")
        for (m, n, k, k256) in ((8, 8192, 29568, 29696), (32, 8192, 29568, 29696), (8, 151936, 896, 1024), (8, 28672, 4224, 4096),
                                (8, 2048, 1408, 1536), (8, 8192, 3696, 3840), (128, 4096, 7392, 7424)):
            for kk in (k, k256):
                copies = max(3, int(COLD_BYTES // (n * kk)) + 1)
                wb = [torch.randint(0, 0x7E, (n, kk), device="cuda", dtype=torch.uint8) for _ in range(min(copies, 6))]
                a8 = torch.randint(0, 0x7E, (m, kk), device="cuda", dtype=torch.uint8)
                d = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)
                for i in range(3):
                    rc = lib.sg_skinny_gemm_auto(a8.data_ptr(), wb[i % len(wb)].data_ptr(), d.data_ptr(), one.data_ptr(), m, n, kk, kk, None)
                    if rc != 0:
                        raise RuntimeError("sg_skinny_gemm_auto: %s" % sg.strerror(rc))
                torch.cuda.synchronize()
                if kk == k:
                    # the register-streaming engine as it was chosen for such k: 64- or 128-byte stages, four or eight
                    # waves sharing K, two 16-row tiles per wave on very wide matrices
                    ku = 2 if k % 128 == 0 else 1
                    stages = -(-k // (64 * ku))
                    waves = 8 if stages >= 16 else 4
                    rec = sg.SgTuning(1, 1, waves, 2 if n >= 8 * 16 * 256 else 1, 1 if m <= 16 else 2, 4 if ku == 1 else 2, ku, 1, 0, 0)
                    for i in range(3):
                        rc = lib.sg_skinny_gemm_tuned(a8.data_ptr(), wb[i % len(wb)].data_ptr(), d.data_ptr(), one.data_ptr(), m, n, k, k,
                                                      ctypes.byref(rec), None)
                        if rc != 0:
                            raise RuntimeError("sg_skinny_gemm_tuned (direct): %s" % sg.strerror(rc))
                    torch.cuda.synchronize()
                del wb
        return

    if args.mid_batch_counters:
        one = torch.ones(1, device="cuda")
        for (n, k) in ((10240, 8192), (8192, 8192), (57344, 8192), (8192, 28672)):
            wb = [torch.randint(0, 0x7E, (n, k), device="cuda", dtype=torch.uint8) for _ in range(2)]
            for m in (64, 128, 256):
                a8 = torch.randint(0, 0x7E, (m, k), device="cuda", dtype=torch.uint8)
                d = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)
                for i in range(3):
                    rc = lib.sg_skinny_gemm_auto(a8.data_ptr(), wb[i % 2].data_ptr(), d.data_ptr(), one.data_ptr(), m, n, k, k, None)
                    if rc != 0:
                        raise RuntimeError("sg_skinny_gemm_auto: %s" % sg.strerror(rc))
                torch.cuda.synchronize()
            del wb
        # stacked activation tiles on weight tile counts that 8 (the XCDs) does not divide, or over more than one round
        for (m, n, k) in ((288, 11008, 4096), (448, 13824, 5120), (320, 22016, 4096), (200, 28672, 8192)):
            wb = [torch.randint(0, 0x7E, (n, k), device="cuda", dtype=torch.uint8) for _ in range(2)]
            a8 = torch.randint(0, 0x7E, (m, k), device="cuda", dtype=torch.uint8)
            d = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)
            for i in range(3):
                rc = lib.sg_skinny_gemm_auto(a8.data_ptr(), wb[i % 2].data_ptr(), d.data_ptr(), one.data_ptr(), m, n, k, k, None)
                if rc != 0:
                    raise RuntimeError("sg_skinny_gemm_auto: %s" % sg.strerror(rc))
            torch.cuda.synchronize()
            del wb
        return

    from rocm_dev_amd import synth

    def quantize(x):
        """Per-tensor scale absmax/448 and OCP E4M3 codes (round to nearest even)."""
        return synth.quantize_tensor(x)

    if args.random_codes:
        class _Codes:   # stands in for the seeded generator: same shapes, arbitrary finite codes
            @staticmethod
            def normal_f32(shape, seed, stream_id):
                return torch.randint(0, 0x7E, shape, device="cuda", dtype=torch.uint8)

            @staticmethod
            def quantize_tensor(x):
                return x, torch.full((), 1e-4, device="cuda")
        synth = _Codes
        quantize = _Codes.quantize_tensor

    # ---- synthetic operands, resident in HBM: the seeded counter generator of rocm_dev_amd.synth ------------
    # (seed 0, stream 1) = activations, (seed c, stream 2) = copy c of a weight matrix: copy 0 is the configuration's
    # own "N(0,1), seed 0" recipe, the further copies only exist so that the weights are cold
    weights, scales_b = {}, {}
    for name, (n, k) in SHAPES.items():
        copies = max(2, int(COLD_BYTES // (n * k)) + 1)
        bufs = []
        for c in range(copies):
            q, sb = quantize(synth.normal_f32((n, k), c, 2))
            bufs.append(q)
            if c == 0:
                scales_b[name] = sb
        weights[name] = bufs
    acts, outs, scl = {}, {}, {}
    for m in M_SWEEP:
        for name, (n, k) in SHAPES.items():
            a8, sa = quantize(synth.normal_f32((m, k), 0, 1))
            acts[(name, m)] = a8
            outs[(name, m)] = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)
            scl[(name, m)] = (sa * scales_b[name]).reshape(1).float().contiguous()
    torch.cuda.synchronize()

    warm_cache = [False]     # True: every launch reads the same weight buffer (stays in the 256 MB last-level cache)

    def launch(name, m, i, stream):
        n, k = SHAPES[name]
        w = weights[name]
        if warm_cache[0]:
            i = 0
        rc = lib.sg_skinny_gemm_auto(acts[(name, m)].data_ptr(), w[i % len(w)].data_ptr(), outs[(name, m)].data_ptr(),
                                     scl[(name, m)].data_ptr(), m, n, k, k, stream)
        if rc != 0:
            raise RuntimeError("sg_skinny_gemm_auto: %s" % sg.strerror(rc))

    order = ("qkv", "o", "gate_up", "down")

    def step(i, stream):
        for name in order:
            launch(name, args.m, i, stream)

    REPLAYS = max(1, args.replays)

    def stats(samples):
        """median, 10th / 90th percentile and minimum of a list of timings"""
        ts = sorted(samples)
        pick = lambda q: ts[min(len(ts) - 1, int(round(q * (len(ts) - 1))))]
        return {"median": ts[len(ts) // 2], "p10": pick(0.1), "p90": pick(0.9), "min": ts[0], "samples": len(ts)}

    def timed_replays(fn, reps, replays=REPLAYS, settle_ms=25.0, region_ms=0.0, info=None):
        """Captures `reps` calls of fn(i, stream) into one HIP graph, replays it untimed until `settle_ms` of GPU work
        have gone by (after other large kernels some launches stay a few per cent slow for about 8 ms of sustained
        work), then times `replays` regions, each inside its own event pair on the launch stream.  A region is one
        replay of the graph or, with region_ms, as many back-to-back replays as make it at least that long: the
        first graph launch inside an event pair costs tens of microseconds of its own (68 us for the 80 nodes of 20
        decode steps), which a short region would carry into the per-call figure and a long one does not.  Returns
        the time per call in us of every region; info["graph_replays_per_region"] says how many replays one held.
        Without graphs (--no-graph) the calls are enqueued eagerly."""
        out = []
        with torch.cuda.stream(side):
            st = torch.cuda.current_stream().cuda_stream
            if args.no_graph:
                run = lambda: [fn(i, st) for i in range(reps)]
            else:
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g, stream=side):
                    st_c = torch.cuda.current_stream().cuda_stream
                    for i in range(reps):
                        fn(i, st_c)
                run = g.replay
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            spent, n_warm = 0.0, 0
            while spent < settle_ms and n_warm < 400:
                a.record()
                run()
                b.record()
                torch.cuda.synchronize()
                spent += a.elapsed_time(b)
                n_warm += 1
            inner = 1
            if region_ms > 0.0:
                a.record()
                run()
                b.record()
                torch.cuda.synchronize()
                inner = max(1, min(64, int(region_ms / max(a.elapsed_time(b), 1e-3) + 0.999)))
            if info is not None:
                info["graph_replays_per_region"] = inner
            for _ in range(replays):
                a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                a.record()
                for _ in range(inner):
                    run()
                b.record()
                torch.cuda.synchronize()
                out.append(a.elapsed_time(b) * 1e3 / (reps * inner))
        return out

    # ---- W warm-up steps, then exactly K steps inside one event pair (captured once in a HIP graph); the timed
    # region is repeated REPLAYS times and `value` is its median, so that one lucky or unlucky replay does not
    # decide the headline; the first replay, the fastest and the 10th / 90th percentiles are reported beside it
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        st = torch.cuda.current_stream().cuda_stream
        for i in range(args.warmup):
            step(i, st)
        torch.cuda.synchronize()
    t_host0 = time.perf_counter()
    # K steps are captured once; a timed region replays that graph until it holds at least 5 ms of work, so that
    # `value` does not depend on K (one replay of 20 steps is 0.9 ms, of which the graph launch itself is 0.07)
    region_info = {}
    step_us = timed_replays(lambda i, st: step(args.warmup + i, st), args.steps, settle_ms=0.0, region_ms=5.0, info=region_info)
    t_host1 = time.perf_counter()
    if args.calibration_copy:
        src = torch.empty(256 << 20, dtype=torch.uint8, device="cuda")
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        del src, dst
    step_stats = stats(step_us)
    ms_per_step = step_stats["median"] * 1e-3
    step_bytes = sum(gemm_bytes(args.m, *SHAPES[name]) for name in order)
    value_tbs = step_bytes / (ms_per_step * 1e-3) / 1e12

    def gemm_stats(name, m, reps=60, replays=REPLAYS):
        """Back-to-back launches of one shape on rotating (cold) weight buffers: us per launch, dispatch gaps included."""
        return stats(timed_replays(lambda i, st: launch(name, m, i, st), reps, replays))

    def per_launch_us(name, m, reps):
        """Every launch inside its own event pair on the launch stream (eager): mean and median."""
        with torch.cuda.stream(side):
            st = torch.cuda.current_stream().cuda_stream
            for i in range(5):
                launch(name, m, i, st)
            evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(reps)]
            torch.cuda.synchronize()
            for i, (a, b) in enumerate(evs):
                a.record()
                launch(name, m, 5 + i, st)
                b.record()
            torch.cuda.synchronize()
        ts = sorted(a.elapsed_time(b) * 1e3 for a, b in evs)
        return sum(ts) / len(ts), ts[len(ts) // 2]

    def choice(m, n, k):
        t, from_table = sg.skinny_gemm_choice(m, n, k)
        wide, line = sg.api.skinny_gemm_wide_choice(m, n, k), sg.api.skinny_gemm_line_choice(m, n, k)
        d = (dict(zip(("wide_row_tiles", "wide_m_blocks", "split_k"), wide)) if wide else
             dict(zip(("line_waves", "line_row_tiles", "line_m_blocks", "split_k"), line)) if line else sg.api.tuning_as_dict(t))
        d["from_table"] = bool(from_table)
        return d

    # The dominant kernel: 60 launches on rotating (cold) weight buffers inside one event pair on the launch stream,
    # median over REPLAYS such regions; the average over a region is what rocprofv3 --kernel-trace reports per launch
    # plus the dispatch gap.
    dom = "gate_up"
    dom_stats = gemm_stats(dom, args.m)
    dom_us = dom_stats["median"]
    dom_ev_mean_us, _ = per_launch_us(dom, args.m, 60)
    dom_bytes = gemm_bytes(args.m, *SHAPES[dom])
    achieved = dom_bytes / (dom_us * 1e-6) / 1e9
    dom_choice = choice(args.m, *SHAPES[dom])
    # HBM bytes per launch from rocprofv3 counters are only valid for the kernel configuration they were measured on
    traffic = None
    if args.m == 8 and all(dom_choice.get(key) == val for key, val in RECORDED_TRAFFIC["tuning"].items()):
        traffic = RECORDED_TRAFFIC["bytes"]
    roofline = {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": round(achieved / HBM_PEAK_GBS, 4), "traffic": traffic,
                "traffic_source": RECORDED_TRAFFIC["source"] if traffic else None,
                "kernel": "dense skinny GEMM, gate_up 28672x4096, M=%d" % args.m,
                "bytes_per_launch": dom_bytes, "us_per_launch": round(dom_us, 3),
                "us_per_launch_p10_p90_min": [round(dom_stats[key], 3) for key in ("p10", "p90", "min")],
                "replays": dom_stats["samples"], "launches_per_replay": 60,
                "us_per_launch_own_event_pair": round(dom_ev_mean_us, 3)}

    per_shape = {}
    for name in order:
        st_ = dom_stats if name == dom else gemm_stats(name, args.m)
        nb = gemm_bytes(args.m, *SHAPES[name])
        per_shape[name] = {"us": round(st_["median"], 3), "us_p10": round(st_["p10"], 3), "us_p90": round(st_["p90"], 3),
                           "us_min": round(st_["min"], 3), "TBps": round(nb / st_["median"] / 1e6, 3),
                           "frac_peak": round(nb / st_["median"] / 1e6 / 8.0, 4), "tuning": choice(args.m, *SHAPES[name])}
        # the same launches on ONE weight buffer: weights served by the last-level cache, not HBM - reported apart,
        # never part of `value` or `roofline`
        if not args.no_warm:
            warm_cache[0] = True
            per_shape[name]["warm_cache_us"] = round(gemm_stats(name, args.m, replays=11)["median"], 3)
            warm_cache[0] = False

    sweep = None
    if not args.no_sweep:
        sweep = []
        for name in order:
            for m in M_SWEEP:
                st_ = gemm_stats(name, m, reps=40, replays=15)
                nb = gemm_bytes(m, *SHAPES[name])
                sweep.append({"shape": name, "m": m, "n": SHAPES[name][0], "k": SHAPES[name][1],
                              "us": round(st_["median"], 3), "us_min": round(st_["min"], 3),
                              "TBps": round(nb / st_["median"] / 1e6, 3),
                              "frac_peak": round(nb / st_["median"] / 1e6 / 8.0, 4)})

    # ---- the other configurations of the path, one timing each (not part of `value`) ---------
    def graph_time_us(fn, reps):
        """median us per call over 11 replays of a graph of `reps` calls (25 ms of untimed replays first)"""
        return stats(timed_replays(fn, reps, replays=11))["median"]

    others = None
    if not args.no_sweep:
        others = {}
        # per-row FP8 codec, 8192 x 8192 (encode bf16 -> e4m3 + row scales; decode + reduce of 8 buffers)
        rows = cols = 8192
        xs = [torch.randn((rows, cols), device="cuda").bfloat16() for _ in range(4)]      # 4 x 128 MiB, rotated
        q8 = torch.empty((8, rows, cols), device="cuda", dtype=torch.uint8)
        s8 = torch.empty((8, rows), device="cuda", dtype=torch.float32)
        y = torch.empty((rows, cols), device="cuda", dtype=torch.bfloat16)
        for i in range(8):
            lib.sg_fp8_encode_rows(xs[i % 4].data_ptr(), q8[i].data_ptr(), s8[i].data_ptr(), rows, cols, None)
        torch.cuda.synchronize()
        enc_us = graph_time_us(lambda i, st: lib.sg_fp8_encode_rows(xs[i % 4].data_ptr(), q8[i % 8].data_ptr(),
                                                                    s8[i % 8].data_ptr(), rows, cols, st), 16)
        dec_us = graph_time_us(lambda i, st: lib.sg_fp8_decode_rows(q8[i % 8].data_ptr(), s8[i % 8].data_ptr(),
                                                                    y.data_ptr(), rows, cols, st), 16)
        red_us = graph_time_us(lambda i, st: lib.sg_fp8_reduce_rows(q8.data_ptr(), s8.data_ptr(), y.data_ptr(), 8,
                                                                    rows * cols, rows, cols, st), 8)
        enc_b, dec_b, red_b = 3 * rows * cols + 4 * rows, 3 * rows * cols + 4 * rows, 8 * (rows * cols + 4 * rows) + 2 * rows * cols
        others["fp8_codec_8192x8192"] = {
            "encode_us": round(enc_us, 2), "encode_TBps": round(enc_b / enc_us / 1e6, 3),
            "decode_us": round(dec_us, 2), "decode_TBps": round(dec_b / dec_us / 1e6, 3),
            "reduce8_us": round(red_us, 2), "reduce8_TBps": round(red_b / red_us / 1e6, 3),
            "note": "reduce reads 512 MiB per launch; the 8 encoded buffers are re-read every launch (beyond the 256 MB cache)"}
        del xs, q8, s8, y
        # mid-batch GEMMs (Llama-3-70B-sized layers)
        mid = []
        for (n, k) in ((10240, 8192), (8192, 8192), (57344, 8192), (8192, 28672)):
            copies = max(2, int(COLD_BYTES // (n * k)) + 1)
            # N(0,1) operands quantised per tensor, as in the decode step (the code distribution matters: the
            # MFMA-heavy shapes are power-limited, and uniformly random codes draw more power than real weights)
            wb = [quantize(torch.randn((n, k), device="cuda", dtype=torch.float32))[0] for _ in range(copies)]
            for m in (64, 128, 256):
                a8 = quantize(torch.randn((m, k), device="cuda", dtype=torch.float32))[0]
                d = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)
                one = torch.ones(1, device="cuda")
                us = graph_time_us(lambda i, st: lib.sg_skinny_gemm_auto(a8.data_ptr(), wb[i % copies].data_ptr(), d.data_ptr(),
                                                                         one.data_ptr(), m, n, k, k, st), max(2 * copies, 8))
                mid.append({"m": m, "n": n, "k": k, "us": round(us, 2), "TBps": round(gemm_bytes(m, n, k) / us / 1e6, 3),
                            "TFLOPs": round(2.0 * m * n * k / us / 1e6, 1), "frac_fp8_peak": round(2.0 * m * n * k / us / 1e6 / 5000.0, 4)})
            del wb
        others["mid_batch"] = mid
        # the one shape the reference's only published timing can be tied to: its profiler launcher's m = 8, n = 6656,
        # k = 16384 (skinny_gemm/prof.cu:9-11); the 24.79 us quoted in skinny_gemm/bench.cu:79-85 names neither shape
        # nor device (MI300X implied by its 304-CU grid), so it is context, not a baseline
        pm, pn, pk = 8, 6656, 16384
        copies = max(2, int(COLD_BYTES // (pn * pk)) + 1)
        wb = [quantize(torch.randn((pn, pk), device="cuda", dtype=torch.float32))[0] for _ in range(copies)]
        a8 = quantize(torch.randn((pm, pk), device="cuda", dtype=torch.float32))[0]
        d = torch.empty((pm, pn), device="cuda", dtype=torch.bfloat16)
        one = torch.ones(1, device="cuda")
        us = graph_time_us(lambda i, st: lib.sg_skinny_gemm_auto(a8.data_ptr(), wb[i % copies].data_ptr(), d.data_ptr(),
                                                                 one.data_ptr(), pm, pn, pk, pk, st), max(2 * copies, 12))
        pb = gemm_bytes(pm, pn, pk)
        others["reference_profiler_shape_8x6656x16384"] = {
            "us": round(us, 2), "TBps": round(pb / us / 1e6, 3), "frac_peak": round(pb / us / 1e6 / 8.0, 4), "bytes": pb,
            "tuning": choice(pm, pn, pk),
            "reference_context": "skinny_gemm/bench.cu:79-85 quotes 24.79 us mean with neither shape nor device stated; if it "
                                 "was this shape on an MI300X (5.3 TB/s peak) that is 4.4 TB/s"}
        del wb, a8, d
        # fp32 batch sum D = sum_b (A_b + B_b): what the reference's split-K experiments reduce their partials with
        tb, tm, tn = 8, 1024, 8192
        ta = torch.randn((tb, tm, tn), device="cuda", dtype=torch.float32)
        tbb = torch.randn((tb, tm, tn), device="cuda", dtype=torch.float32)
        td = torch.empty((tm, tn), device="cuda", dtype=torch.float32)
        tsr_us = graph_time_us(lambda i, st: lib.sg_tiled_sum_reduce(ta.data_ptr(), tbb.data_ptr(), td.data_ptr(), tb, tm, tn, st), 8)
        tsr_q_us = graph_time_us(lambda i, st: lib.sg_tiled_sum_reduce_async(ta.data_ptr(), tbb.data_ptr(), td.data_ptr(), tb, tm, tn, st), 8)
        tsr_bytes = (2 * tb + 1) * tm * tn * 4
        others["tiled_sum_reduce_8x1024x8192"] = {"us": round(tsr_us, 2), "TBps": round(tsr_bytes / tsr_us / 1e6, 3),
                                                  "lds_queue_us": round(tsr_q_us, 2), "lds_queue_TBps": round(tsr_bytes / tsr_q_us / 1e6, 3),
                                                  "note": "reads 512 MiB per launch (beyond the 256 MB cache), writes 32 MiB; "
                                                          "lds_queue = sg_tiled_sum_reduce_async"}
        del ta, tbb, td
        # bf16 activations quantised per row inside the GEMM (one launch) against the two launches it replaces
        # (sg_fp8_encode_rows, then sg_skinny_gemm_rowcol with the library's own configuration), cold weights
        fused_rows = []
        for name in order:
            n, k = SHAPES[name]
            for m in (8, 16):
                xb = synth.normal_f32((m, k), 1, 1).bfloat16()
                q = torch.empty((m, k), device="cuda", dtype=torch.uint8)
                rs = torch.empty((m,), device="cuda", dtype=torch.float32)
                cs = torch.ones((n,), device="cuda", dtype=torch.float32)
                d = outs[(name, m)]
                w = weights[name]
                _, is_fused = sg.skinny_gemm_bf16act_choice(m, n, k)

                def one(i, st):
                    rc = lib.sg_skinny_gemm_bf16act(xb.data_ptr(), w[i % len(w)].data_ptr(), d.data_ptr(), scl[(name, m)].data_ptr(),
                                                    cs.data_ptr(), None, m, n, k, k, st)
                    if rc != 0:
                        raise RuntimeError("sg_skinny_gemm_bf16act: %s" % sg.strerror(rc))

                def two(i, st):
                    rc = lib.sg_fp8_encode_rows(xb.data_ptr(), q.data_ptr(), rs.data_ptr(), m, k, st)
                    rc = rc or lib.sg_skinny_gemm_rowcol(q.data_ptr(), w[i % len(w)].data_ptr(), d.data_ptr(), scl[(name, m)].data_ptr(),
                                                         rs.data_ptr(), cs.data_ptr(), m, n, k, k, st)
                    if rc != 0:
                        raise RuntimeError("encode_rows + rowcol: %s" % sg.strerror(rc))

                fused_rows.append({"shape": name, "m": m, "n": n, "k": k, "single_launch": bool(is_fused),
                                   "bf16act_us": round(graph_time_us(one, 40), 3),
                                   "encode_then_rowcol_us": round(graph_time_us(two, 40), 3)})
        others["bf16_activations"] = fused_rows
        # 2:4 sparse GEMMs
        sp = []
        for (n, k) in ((4096, 14336), (14336, 4096)):
            copies = max(2, int(COLD_BYTES // (n * k * 0.625)) + 1)
            # N(0,1) weights quantised per tensor, then pruned 2:4 and compressed on the device
            vb, mb = [], []
            for _ in range(copies):
                dense = quantize(torch.randn((n, k), device="cuda", dtype=torch.float32))[0]
                v = torch.empty((n, k // 2), device="cuda", dtype=torch.uint8)
                t = torch.empty((n, k // 8), device="cuda", dtype=torch.uint8)
                rc = lib.sg_sparse24_compress(dense.data_ptr(), v.data_ptr(), t.data_ptr(), n, k, k, None)
                if rc != 0:
                    raise RuntimeError("sg_sparse24_compress: %s" % sg.strerror(rc))
                vb.append(v)
                mb.append(t)
            torch.cuda.synchronize()
            del dense
            for m in (1, 8, 16, 32):
                a8 = quantize(torch.randn((m, k), device="cuda", dtype=torch.float32))[0]
                d = torch.empty((m, n), device="cuda", dtype=torch.bfloat16)
                one = torch.ones(1, device="cuda")
                us = graph_time_us(lambda i, st: lib.sg_sparse24_gemm(a8.data_ptr(), vb[i % copies].data_ptr(), mb[i % copies].data_ptr(),
                                                                      d.data_ptr(), one.data_ptr(), m, n, k, st), max(2 * copies, 8))
                nb = m * k + 0.625 * n * k + 2 * m * n
                sp.append({"m": m, "n": n, "k": k, "us": round(us, 2), "TBps": round(nb / us / 1e6, 3)})
            del vb, mb
        others["sparse24"] = sp

    # ---- CPU baseline: the oracle's all-core loop on the same step (rank 0, N = 1 only) ------
    cpu = None
    if not args.no_cpu:
        import oracle
        t_cpu = 0.0
        for name in order:
            n, k = SHAPES[name]
            a8 = acts[(name, args.m)].cpu().numpy()
            b8 = weights[name][0].cpu().numpy()
            s = float(scl[(name, args.m)].item())
            t0 = time.perf_counter()
            oracle.gemm_omp(a8, b8, s)
            t_cpu += time.perf_counter() - t0
        # the faithful one-core loop of the reference's test on a slice of the O projection
        n, k = SHAPES["o"]
        a8 = acts[("o", args.m)].cpu().numpy()
        b8 = weights["o"][0].cpu().numpy()[:512]
        t0 = time.perf_counter()
        oracle.gemm_ref(a8, b8, 1.0)
        t_ref = (time.perf_counter() - t0) * (n / 512.0)
        cpu = {"value": round(step_bytes / t_cpu / 1e12, 6), "unit": "TB/s", "cores": oracle.num_threads(),
               "kind": "port", "sample": "one full step (4 GEMMs, M=%d) with the oracle's OpenMP loop: %.3f s; "
               "single-core reference loop on the O projection (512-row slice scaled to 4096 rows): %.3f s"
               % (args.m, t_cpu, t_ref), "ms_per_step": round(t_cpu * 1e3, 2), "one_core_o_proj_s": round(t_ref, 3)}
        # the reference's own host loop (skinny_gemm/test.cu:7-39, compiled from its source into oracle/_ref where
        # the reference tree was present at build time), one core, same slice; it reads the bytes as E4M3 FNUZ
        ref_lib = os.path.join(ROOT, "oracle", "_ref", "libref_host.so")
        if os.path.exists(ref_lib):
            import ctypes
            import numpy as np
            rl = ctypes.CDLL(ref_lib)
            rl.ref_host_skinny_gemm_f32.argtypes = [ctypes.c_void_p] * 3 + [ctypes.c_float] + [ctypes.c_int] * 3
            d = np.empty((args.m, 512), np.float32)
            t0 = time.perf_counter()
            rl.ref_host_skinny_gemm_f32(a8.ctypes.data, b8.ctypes.data, d.ctypes.data, 1.0, args.m, 512, k)
            cpu["reference_host_loop_o_proj_s"] = round((time.perf_counter() - t0) * (n / 512.0), 3)

    out = {
        "metric": "achieved HBM TB/s (and us/GEMM), FP8 skinny GEMM, M=%d, Llama-3-8B projection shapes, 1 MI355X" % args.m,
        "value": round(value_tbs, 4), "unit": "TB/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 5), "ms_per_step_p10_p90_min_first": [round(step_stats[key] * 1e-3, 5) for key in ("p10", "p90", "min")] + [round(step_us[0] * 1e-3, 5)],
        "timed_regions": step_stats["samples"], "graph_replays_per_region": region_info.get("graph_replays_per_region", 1),
        "steps_per_region": args.steps * region_info.get("graph_replays_per_region", 1), "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "fp8_e4m3 (fp32 accumulate, bf16 out)", "data": "synthetic",
        "config": {"workload": "decode sweep, Llama-3-8B projections (QKV, O, gate_up, down), M=%d, cold weights "
                   "(rotating buffers > 2x MALL)" % args.m, "step_bytes": step_bytes,
                   "us_per_gemm_in_step": round(ms_per_step * 1e3 / 4, 3), "frac_hbm_peak": round(value_tbs / 8.0, 4),
                   "host_wall_ms": round((t_host1 - t_host0) * 1e3, 3)},
        "roofline": roofline, "cpu_baseline": cpu, "per_shape": per_shape, "sweep": sweep, "other_configs": others,
    }
    print(json.dumps(out))


if __name__ == "__main__":
    main()
