"""The generated code of the wide-tile GEMM (csrc/sg_wide_kernel.h).  Its matrix instructions are inline text, so the compiler
knows nothing of their latency: no hazard it inserts idle states for, no reason to keep a copy or a spill of an accumulator
away from the instruction that is still writing it.  What the kernel does about that is checked in the assembly."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rocm_dev_amd", "csrc")
TILES = [(4, 8), (5, 8), (6, 8), (7, 8), (8, 8), (8, 4), (4, 4)]
# A vector or memory instruction may read a 16-pass matrix instruction's result 19 wait states after it; an instruction is one.
WAIT_STATES = 19


@pytest.fixture(scope="module")
def kernels():
    """{(row tiles, m blocks, partial last block): instructions}, and the resource report of each."""
    if not shutil.which("hipcc") and not os.path.exists("/opt/rocm/bin/hipcc"):
        pytest.skip("no hipcc")
    subprocess.run(["make", "-s", "-C", CSRC, "obj/sg_wide_inst.s"], check=True, capture_output=True)
    text = open(os.path.join(CSRC, "obj", "sg_wide_inst.s")).read()
    out = {}
    for m in re.finditer(r"^(_ZN2sg16wide_gemm_kernelILi(\d)ELi(\d)E\w*?ELb(\d)E\w*):[^\n]*\n(.*?)^\s*\.section", text, re.S | re.M):
        code = [line.split(";")[0].strip() for line in m.group(5).splitlines()]
        report = re.search(r"\.name:\s*%s\n(.*?)\.wavefront_size" % m.group(1), text, re.S).group(1)
        out[int(m.group(2)), int(m.group(3)), m.group(4) == "1"] = ([c for c in code if c and not c.startswith(".")], report)
    return out


def _accumulators(instruction):
    regs = set()
    for lo, hi in re.findall(r"\ba\[(\d+):(\d+)\]", instruction):
        regs.update(range(int(lo), int(hi) + 1))
    regs.update(int(r) for r in re.findall(r"\ba(\d+)\b", instruction))
    return regs


@pytest.mark.parametrize("rg,mb", TILES)
@pytest.mark.parametrize("tail", [False, True])
def test_no_accumulator_is_touched_while_it_is_being_written(kernels, rg, mb, tail):
    code, report = kernels[rg, mb, tail]
    busy = {}                                    # accumulator register -> wait states since its matrix instruction
    matrix = 0
    for instruction in code:
        regs = _accumulators(instruction)
        if instruction.startswith("v_mfma"):
            matrix += 1
            busy = {r: s + 1 for r, s in busy.items()}
            busy.update({r: 0 for r in regs})
            continue
        early = [r for r in regs if busy.get(r, WAIT_STATES) < WAIT_STATES]
        assert not early, "%s: a%d is read %d wait states behind its matrix instruction" % (instruction, early[0], busy[early[0]])
        nop = re.match(r"s_nop (\d+)", instruction)
        busy = {r: s + (int(nop.group(1)) + 1 if nop else 1) for r, s in busy.items()}
    assert matrix == 3 * rg * mb                 # the unrolled pair of stages and the odd last one
    # every accumulator stays in its register: a spill is one more access that nothing orders
    for key in ("vgpr_spill_count", "sgpr_spill_count"):
        assert int(re.search(r"\.%s:\s*(\d+)" % key, report).group(1)) == 0, key
