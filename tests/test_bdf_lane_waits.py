"""Wait states around the whole-wave BDF solver's multiply-adds with a broadcast
operand.  They are inline assembly, for which the compiler adds no waits: a
vector instruction that writes the operand has to be two wait states away, and so
does the lane operation that reads a result.  Checked on the assembly of the
solver as it is built and as other instruction schedulers order it."""
import concurrent.futures as cf
import os
import re
import subprocess

import pytest

from bacon_amd import build as B

SRC = """#include "%s/bdf_device.h"
namespace bg {
template __global__ void bdf_wave_kernel<RhsBrusselatorG<16>, 3, BdfSem<false>, %%s, 4>(
    bg_ensemble_desc, uint32_t *);
}
""" % B.CSRC


def _regs(operand):
    m = re.match(r"v\[(\d+):(\d+)\]", operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.match(r"v(\d+)\b", operand)
    return {int(m[1])} if m else set()


def _hazards(text):
    """(broadcast multiply-adds, those and other lane operations that read a
    register within two wait states of its write)"""
    n, bad, past = 0, [], []
    for line in text.split("\n"):
        m = re.match(r"\s+([a-z]\w+)\s+(.*)", line.split(";")[0])
        if not m:
            continue
        op, args = m[1], [a.strip() for a in m[2].split(",")]
        if op == "s_nop":
            past.append((set(), int(args[0], 0) + 1))
            continue
        permlane = op.startswith("v_permlane")
        reads = set()
        if "row_newbcast" in line:
            n += 1
            reads = _regs(args[1])
        elif permlane or "_dpp" in op:
            reads = set().union(*(_regs(a) for a in (args if permlane else args[1:])))
        states = 0
        for written, length in reversed(past[-3:]):
            if states >= 2:
                break
            if written & reads:
                bad.append(line.strip())
            states += length
        writes = set()
        if op.startswith("v_") and not op.startswith(("v_cmp", "v_readlane", "v_readfirstlane")):
            writes = _regs(args[0]) | (_regs(args[1]) if permlane else set())
        past.append((writes, 1))
    return n, bad


def test_the_check_sees_a_missing_wait():
    write, use = "\tv_cndmask_b32_e32 v4, v1, v2, vcc", (
        "\tv_fmac_f64_dpp v[8:9], v[4:5], v[6:7] row_newbcast:3 row_mask:0xf bank_mask:0xf")
    assert len(_hazards("\n".join([write, use]))[1]) == 1
    assert len(_hazards("\n".join([write, "\ts_nop 0", use]))[1]) == 1
    assert _hazards("\n".join([write, "\ts_nop 1", use])) == (1, [])


@pytest.mark.parametrize("inverse", ["double", "float"])
def test_wait_states(tmp_path, inverse):
    if not os.path.exists(B.hipcc()):
        pytest.skip("no hipcc")
    src = tmp_path / "solver.hip"
    src.write_text(SRC % inverse)

    def compile_with(extra):
        out = tmp_path / ("_".join(extra) + ".s")
        subprocess.run([B.hipcc(), *B.HIPFLAGS, "-w", "--cuda-device-only", "-S", *extra,
                        str(src), "-o", str(out)], check=True, timeout=300)
        return _hazards(out.read_text())

    schedules = ([], ["-mllvm", "-misched=ilpmax"], ["-mllvm", "-misched=gcn-iterative-ilp"],
                 ["-mllvm", "-enable-post-misched=0"])
    with cf.ThreadPoolExecutor(4) as ex:
        for n, bad in ex.map(compile_with, schedules):
            assert n > 1000 and not bad, bad[:5]
