"""CPU: broadcasts inside vector instructions (DPP) that are written as inline assembly.

A vector register may be a DPP source no sooner than two wait states after a vector instruction wrote it.  The compiler sees to that for
its own instructions and does not look into assembly, so a statement with such an instruction either brings its wait states along or takes
its source from LDS or from before a loop.  The first is checked on the source text, both on the ISA that hipcc emits (no GPU needed)."""
import os
import re
import subprocess

import pytest

from rwkv_cuda_amd._lib import HIPCC_FLAGS

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "rwkv_cuda_amd", "csrc")


def _read(name):
    with open(os.path.join(CSRC, name)) as f:
        return re.sub(r"//[^\n]*", "", f.read())


def _asm_helpers():
    """Function of common.h -> the templates of its asm statements that are not empty, up to the first macro."""
    out = {}
    for m in re.finditer(r"DEVINL \w+ (\w+)\([^\n]*\) \{ *\n(.*?)\n\}", _read("common.h"), re.S):
        bodies = [b for b in re.findall(r"\basm\b(?:\s+volatile)?\s*\(\s*\"([^\"]*)\"", m.group(2)) if b]
        if bodies:
            out[m.group(1)] = bodies
    return out


@pytest.mark.parametrize("name", ["split3.h", "rwkv7_chunk.hip"])
def test_assembly_of_the_matrix_kernels_brings_its_wait_states(name):
    """These files have no instruction in assembly of their own (tests/test_rwkv7_split.py); this is about what they call."""
    helpers, text = _asm_helpers(), _read(name)
    assert {"fmac_bc", "mul_bc", "solve_bc", "allreduce_rows"} <= set(helpers)
    for helper, bodies in helpers.items():
        if re.search(r"\b%s\s*[<(]" % helper, text):
            assert all(b.startswith("s_nop 1\\n") for b in bodies), helper


def _registers(operand):
    m = re.fullmatch(r"v(\d+)|v\[(\d+):(\d+)\]", operand.strip().lstrip("-|").rstrip("|"))
    return range(0) if not m else range(int(m.group(1)), int(m.group(1)) + 1) if m.group(1) else range(int(m.group(2)), int(m.group(3)) + 1)


def _too_soon(asm):
    """(number of DPP instructions, those whose source a vector instruction wrote less than two wait states before)"""
    written, now, count, bad = {}, 0, 0, []
    for line in asm.splitlines():
        line = line.split(";")[0].strip()
        m = re.match(r"([a-z]\w+)\s*(.*)", line)
        if not m or line.endswith(":"):
            continue
        op, args = m.group(1), m.group(2).split(",")
        if "_dpp" in op:
            count += 1
            source = args[1].split()[0]
            if any(now - written.get(r, -9) < 2 for r in _registers(source)):
                bad.append(line)
        now += int(args[0]) + 1 if op == "s_nop" else 1
        if op.startswith("v_") and not op.startswith("v_cmp"):
            for operand in args[:2] if "_swap" in op else args[:1]:
                for r in _registers(operand.split()[0] if operand.split() else ""):
                    written[r] = now
    return count, bad


def test_the_scan_finds_a_source_that_was_just_written():
    dpp = "v_fmac_f32_dpp v1, v2, v3 row_newbcast:4 row_mask:0xf bank_mask:0xf"
    assert _too_soon("v_mov_b32_e32 v2, v9\n%s" % dpp) == (1, [dpp])
    assert _too_soon("v_mov_b32_e32 v2, v9\nv_add_f32_e32 v7, v8, v9\n%s" % dpp) == (1, [dpp])
    assert _too_soon("v_mfma_f32_16x16x32_bf16 v[0:3], v[4:7], v[8:11], 0\ns_nop 0\n%s" % dpp) == (1, [dpp])
    assert _too_soon("v_mov_b32_e32 v2, v9\ns_nop 1\n%s" % dpp) == (1, [])
    assert _too_soon("v_mov_b32_e32 v3, v9\nds_read_b32 v2, v8\n%s" % dpp) == (1, [])


@pytest.mark.parametrize("name", ["rwkv7_chunk.hip", "rwkv7.hip", "wkv6_bwd_f.hip"])
def test_no_broadcast_of_a_register_that_was_just_written(name):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    flags = [f for f in HIPCC_FLAGS if not f.startswith("-Rpass")]
    cmd = [hipcc] + flags + ["--cuda-device-only", "-S", "-I", os.path.join(ROOT, "include"), "-I", CSRC, "-o", "-", os.path.join(CSRC, name)]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    count, bad = _too_soon(res.stdout)
    assert count > 0 and not bad, bad[:5]
