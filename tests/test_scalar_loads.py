"""Build check of the K-logit kernels' scalar loads (CPU only).

A scalar load's address is the sum of a base, a register offset and a
constant, and the hardware drops the two low bits of each of them before it
adds.  The compiler has formed the address of a 64-bit table entry as
(kernel arguments + 2 kv) + 6 kv, sharing the first sum with the 16-bit table
KArgs::krank: right as arithmetic, but 4 bytes low for odd kv once the low
bits are gone, and the offset read there led outside every address range (a
variant of the warp-specialised kernel that was never committed; the GPU
reported an aperture violation).  This test compiles the sources whose
kernels index tables in their arguments and fails if a scalar load with a
register offset takes a base or an offset that is not a multiple of 4 by its
last definition before the load.
"""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "star-kv_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def _code(src, tmp_path):
    out = tmp_path / (src + ".s")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-S", "-o", str(out),
                    os.path.join(CSRC, src)], check=True, capture_output=True)
    lines = (ln.split(";")[0].strip() for ln in out.read_text().splitlines())
    return [ln for ln in lines if ln and not ln.startswith((".", "#", "//"))]


def _definition(code, i, reg):
    """The last instruction before code[i] that writes scalar register `reg`."""
    for j in range(i - 1, -1, -1):
        m = re.match(r"s_\w+\s+s(?:(\d+)|\[(\d+):(\d+)\])\s*,", code[j])
        if m and not code[j].startswith(("s_cmp", "s_bitcmp", "s_store")):
            lo, hi = (int(m.group(1)),) * 2 if m.group(1) else (int(m.group(2)), int(m.group(3)))
            if lo <= reg <= hi:
                return j, code[j]
        if code[j].startswith("_ZN") and code[j].endswith(":"):
            break
    return None, ""


def _misaligned(code, i, reg, depth=0):
    """Whether register `reg` at code[i] is seen to be no multiple of 4."""
    j, d = _definition(code, i, reg)
    if j is None or depth > 4:
        return False
    if m := re.match(r"s_lshl_b(?:32|64)\s+\S+,\s*\S+,\s*(\d+)$", d):
        return int(m.group(1)) < 2
    if m := re.match(r"s_mul_i32\s+\S+,\s*s\d+,\s*(0x[0-9a-f]+|\d+)$", d):
        return int(m.group(1), 0) % 4 != 0
    if re.match(r"s_lshl1_add_u32\s", d):
        return True
    if m := re.match(r"s_add_[ui]32\s+\S+,\s*(\S+),\s*(\S+)$", d):
        return any(_misaligned(code, j, int(o[1:]), depth + 1) if re.match(r"s\d+$", o) else
                   re.match(r"(0x[0-9a-f]+|\d+)$", o) is not None and int(o, 0) % 4 != 0 for o in m.groups())
    return False


def bad_loads(code):
    bad, seen = [], 0
    for i, ln in enumerate(code):
        m = re.match(r"s_load_dword\w*\s+\S+,\s*s\[(\d+):\d+\],\s*s(\d+)\b", ln)
        if not m:
            continue
        seen += 1
        if any(_misaligned(code, i, int(r)) for r in m.groups()):
            bad.append(ln)
    return bad, seen


def test_the_check_sees_the_form_it_guards():
    code = ["_ZN1k:", "s_lshl_b32 s3, s50, 1", "s_add_u32 s38, s0, s3", "s_addc_u32 s39, s1, 0", "s_mul_i32 s8, s50, 6",
            "s_load_dwordx2 s[12:13], s[38:39], s8 offset:0x708"]
    assert bad_loads(code) == ([code[-1]], 1)
    code[1], code[4] = "s_lshl_b32 s3, s50, 2", "s_lshl_b32 s8, s50, 2"
    assert bad_loads(code) == ([], 1)


@pytest.mark.skipif(not shutil.which(HIPCC) and not os.path.exists(HIPCC), reason="hipcc not installed")
@pytest.mark.parametrize("src", ["k_logits.hip", "k_logits_ws.hip", "k_logits_gqa.hip"])
def test_scalar_load_components_are_dwords(src, tmp_path):
    bad, seen = bad_loads(_code(src, tmp_path))
    assert seen > 0, "no scalar load with a register offset: the check no longer sees what it guards"
    assert not bad, bad[:8]
