"""Wait states of the device code that is built for gfx950: a vector instruction that reads a scalar
register (VCC among them) comes at least two wait states after the vector instruction that wrote it. The
compiler keeps this in the code it schedules and not inside inline assembly. Checked on the assembly of the
sources that hold instructions of their own."""

import glob
import os
import re
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "hoomd-blue_amd", "csrc")
WAIT = 2


def registers(operand):
    """Scalar registers named by an operand of a vector instruction."""
    if operand == "vcc":
        return {"vcc_lo", "vcc_hi"}
    if operand in ("vcc_lo", "vcc_hi"):
        return {operand}
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if m:
        return {f"s{k}" for k in range(int(m[1]), int(m[2]) + 1)}
    return {operand} if re.fullmatch(r"s\d+", operand) else set()


def violations(asm):
    age, bad = {}, []  # wait states since the vector write of each scalar register
    for no, line in enumerate(asm.splitlines(), 1):
        text = line.split(";")[0].strip()
        if not text or text.startswith("."):
            if text.endswith(":"):
                age = {}
            continue
        if text.endswith(":"):
            age = {}
            continue
        op, _, rest = text.partition(" ")
        operands = [o.strip().strip("|-") for o in rest.split(",")]
        reads, writes = set(), set()
        if op.startswith("v_"):
            if op.startswith(("v_cmp", "v_readlane", "v_readfirstlane")):
                dst = [0]
            elif re.match(r"v_(add|sub|addc|subb|subbrev|subrev)_co_|v_div_scale|v_mad_[ui]64_", op):
                dst = [0, 1]
            else:
                dst = [0]
            for k, o in enumerate(operands):
                (writes if k in dst else reads).update(registers(o))
        bad += [(no, r, text) for r in reads if age.get(r, WAIT) < WAIT]
        step = int(operands[0]) + 1 if op == "s_nop" else 1
        age = {r: a + step for r, a in age.items() if a + step < WAIT}
        for r in writes:
            age[r] = 0
        if op.startswith("s_"):  # a scalar write takes the register over
            for r in registers(operands[0]):
                age.pop(r, None)
    return bad


def with_assembly():
    """The sources with instructions of their own, and the column list build."""
    own = {os.path.join(CSRC, "tile.hip")}
    for f in glob.glob(os.path.join(CSRC, "*")):
        if re.search(r'\basm\b[^;]*?\(\s*"[^"]', open(f).read()):
            own.add(f)
    return sorted(os.path.basename(f) for f in own)


def test_the_scan_finds_a_missing_wait():
    pair = "v_cmp_ge_f32 vcc, 0, v1\n{}v_addc_co_u32 v0, vcc, v0, v0, vcc\n"
    assert len(violations(pair.format(""))) == 2
    assert len(violations(pair.format("s_nop 0\n"))) == 2
    assert not violations(pair.format("s_nop 1\n"))
    assert not violations(pair.format("v_mov_b32 v2, 0\nv_mov_b32 v3, 0\n"))


@pytest.mark.parametrize("src", with_assembly())
def test_vector_reads_wait_for_vector_writes(src, tmp_path):
    import sys
    sys.path.insert(0, os.path.join(ROOT, "hoomd-blue_amd"))
    import build
    out = tmp_path / "device.s"
    subprocess.run([build.hipcc()] + build.CFLAGS + ["-S", "--cuda-device-only", os.path.join(CSRC, src),
                                                     "-o", str(out)], check=True, capture_output=True)
    bad = violations(out.read_text())
    assert not bad, (len(bad), bad[:4])
