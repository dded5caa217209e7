"""The builds of the batch sum (csrc/sg_tsr.hip): one by one at the largest size each takes and one float beyond, with whole
groups of the batches that it asks for at once and with part of one."""
import launch_recorder
import pytest
import torch

CU = 256
# floats -> (pieces a lane, batches at once, threads) at 2 and at 9 batches
ONE = (1, 1, 256)
BUILDS = {257: ((1, 8, 64),) * 2, 1152 * CU: ((1, 8, 64),) * 2, 1152 * CU + 1: ((2, 4, 256),) * 2, 2048 * CU: ((2, 4, 256),) * 2,
          2048 * CU + 1: (ONE,) * 2, 2944 * CU + 1: (ONE, (2, 1, 256)), 4096 * CU: (ONE, (2, 1, 256)), 4096 * CU + 1: (ONE,) * 2,
          5120 * CU + 3: ((2, 1, 256),) * 2, 6144 * CU + 1: ((4, 1, 512),) * 2, 8192 * CU: ((4, 1, 512),) * 2,
          8192 * CU + 1: ((2, 1, 256),) * 2, 9728 * CU + 2: ((4, 1, 256),) * 2,
          12288 * CU + 1: ((8, 1, 256),) * 2, 16384 * CU + 1: ((4, 1, 256),) * 2, 20480 * CU + 1: ((2, 1, 256), (8, 1, 256))}
# other numbers of batches: (floats, batches) -> build
OTHERS = {(256, 2): ONE, (256, 9): ONE, (257, 1): ONE, (4096 * CU, 4): ONE, (4096 * CU, 5): (2, 1, 256)}


def build_of(mn, b):
    """(pieces a lane, batches at once, threads)"""
    if (mn, b) in OTHERS:
        return OTHERS[mn, b]
    return ONE if b == 1 and mn <= 4096 * CU else BUILDS[mn][b == 9]


def choices(rec):
    out = []
    for mn, b in [(mn, b) for mn in BUILDS for b in (2, 9, 1)] + list(OTHERS):
        rc, launches = rec.of("sg_tiled_sum_reduce", rec.A, rec.B, rec.D, b, 1, mn, None)
        assert rc == 0 and len(launches) == 1
        out.append([mn, b, launches[0][0], launches[0][1], launches[0][2]])
    return out


def test_build_of_every_size(tmp_path):
    for mn, b, kernel, grid, threads in launch_recorder.scenario(launch_recorder.build(tmp_path), "test_gpu_batch_sum_builds", "choices"):
        pieces, batches, wide = build_of(mn, b)
        assert "tiled_sum_reduce_kernel<%d, %d, %d," % (pieces, batches, wide) in kernel and threads == wide, (mn, b, kernel)
        # whole workgroups, then one-piece workgroups over what they leave
        whole = mn // (4 * wide * pieces)
        assert grid == whole + -(-(mn - whole * 4 * wide * pieces) // (4 * wide)), (mn, b)


@pytest.mark.gpu
@pytest.mark.parametrize("mn", sorted(BUILDS) + [300, 1028])
def test_bits_at_the_edges(mn):
    import rocm_dev_amd as sg
    g = torch.Generator(device="cuda").manual_seed(mn)
    for b in (1, 2, 3, 4, 7, 8, 9, 15, 16, 17) if mn <= 2048 * CU + 1 else (1, 2, 5):
        A, B = (torch.randn((b, 1, mn), generator=g, device="cuda") for _ in range(2))
        guarded = torch.full((mn + 512,), 7.0, device="cuda")
        D = guarded[256:256 + mn].view(1, mn)
        assert sg.tiled_sum_reduce(A, B, D) == 0
        want = torch.zeros((1, mn), device="cuda")
        for i in range(b):
            want = want + (A[i] + B[i])      # the batches in order, each sum rounded
        assert torch.equal(D.view(torch.int32), want.view(torch.int32)), (b, mn)
        assert bool((guarded[:256] == 7).all() and (guarded[256 + mn:] == 7).all()), (b, mn)
