"""CPU: the build's limits on spilled registers name every kernel that holds a segment's inputs in registers."""
import os
import re
import subprocess

import pytest

from rwkv_cuda_amd._lib import HIPCC_FLAGS, SPILL_LIMIT

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "rwkv_cuda_amd", "csrc")


def test_wkv4_kernels_with_inputs_in_registers_have_a_limit():
    """Every instantiation of the register and block kernels is matched by one entry (what matches none is never looked at), and keeps to it."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    cmd = [hipcc] + HIPCC_FLAGS + ["--cuda-device-only", "-S", "-I", os.path.join(ROOT, "include"), "-I", CSRC, "-o", os.devnull, os.path.join(CSRC, "wkv4.hip")]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    spilled = re.findall(r"remark: Function Name: (\S+).*?VGPRs Spill: (\d+)", res.stderr, re.S)
    held = [(name, int(n)) for name, n in spilled if re.search(r"wkv4_(fwd|bwd)_(reg|blk)", name)]
    assert len(held) >= 20
    for name, n in held:
        limits = [limit for key, limit in SPILL_LIMIT.items() if key in name]
        assert len(limits) == 1 and n <= limits[0], (name, n, limits)
