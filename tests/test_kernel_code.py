"""The traversal kernels' generated code keeps the wait states between a vector instruction that writes a
scalar mask and one that reads it.

On gfx940-class hardware (gfx950 among it) a vector instruction that reads an SGPR or VCC which a vector
instruction wrote must come at least two wait states after it.  The compiler sees to it in the code it
generates, but not inside inline assembly.
"""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "metal-vibe-tracer_amd")
HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")
WAIT = 2


def scalar_registers(operand):
    operand = operand.strip()
    if operand == "vcc":
        return {"vcc"}
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if m:
        return {f"s{i}" for i in range(int(m[1]), int(m[2]) + 1)}
    return {operand} if re.fullmatch(r"s\d+", operand) else set()


def missing_waits(text):
    """(writer, reader) pairs closer than WAIT wait states, in the order of the listing."""
    recent, found = [], []  # recent: [registers written, wait states since, instruction]
    for line in text.splitlines():
        m = re.match(r"\s+([a-z]\w+)\s*([^;]*)", line)
        if not m:
            continue
        op, args = m[1], [a for a in re.split(r",\s*(?![^\[]*\])", m[2].strip()) if a]
        passed, written = 1, set()
        if op == "s_nop":
            passed = int(args[0], 0) + 1
        elif op.startswith("v_"):
            outputs = 2 if re.search(r"_co_|div_scale", op) else 1
            read = set().union(*map(scalar_registers, args[outputs:]))
            found += [(w, line.strip()) for regs, waited, w in recent if regs & read and waited < WAIT]
            written = set().union(*map(scalar_registers, args[:outputs]))
        recent = [[r, n + passed, w] for r, n, w in recent if n + passed < WAIT]
        if written:
            recent.append([written, 0, line.strip()])
    return found


def test_checker_sees_a_missing_wait():
    pair = "\tv_cmp_le_f32 vcc, v1, v2\n{}\tv_addc_co_u32 v3, vcc, v3, v3, vcc\n"
    assert len(missing_waits(pair.format(""))) == 1
    assert len(missing_waits(pair.format("\ts_nop 0\n"))) == 1
    assert not missing_waits(pair.format("\ts_nop 1\n"))
    assert not missing_waits(pair.format("\tv_mov_b32_e32 v4, v5\n\ts_nop 0\n"))
    assert len(missing_waits("\tv_cmp_le_f32_e64 s[4:5], v1, v2\n\tv_cndmask_b32_e64 v3, 0, 1, s[4:5]\n")) == 1


def test_traversal_kernels_wait_for_masks(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("needs hipcc")
    out = tmp_path / "trace.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-device-only", "-S", "-O3", "-std=c++17", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(PKG, "csrc"), os.path.join(PKG, "csrc", "trace.hip"), "-o", str(out)],
                   check=True, capture_output=True)
    text = out.read_text()
    assert "trace_refill_kernel" in text and "v_cmp_le_f32" in text
    found = missing_waits(text)
    assert not found, f"{len(found)} reads too early, first: {found[0]}"
