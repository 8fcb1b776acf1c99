"""What the compiler does not check around the loads that tl1_gemm.hip issues from assembly,
checked in the gfx950 assembly of that source (CPU: compiled here, nothing runs):

* a vector memory instruction reads a scalar register at least five wait states after a vector
  instruction has written it;
* M0, which the assembly sets, is used by nothing else in those kernels."""
import os
import re
import subprocess

import pytest

from tenzo_amd import build

LOAD = re.compile(r"buffer_load_dwordx4 v\d+, s\[(\d+):(\d+)\], \S+ offen lds")


def kernels(text):
    """{name: its lines} of the functions with such loads in assembly blocks."""
    found = {}
    for m in re.finditer(r"^(\w+):[^\n]*\n(.*?)^\.Lfunc_end", text, re.S | re.M):
        lines, app = [], False
        for line in m.group(2).split("\n"):
            app = (app or "#APP" in line or "#ASMSTART" in line) and not (
                "#NO_APP" in line or "#ASMEND" in line)
            code = line.split(";")[0].strip()
            if code and not code.startswith(".") and not code.endswith(":"):
                lines.append((code, app))
        if any(a and LOAD.search(c) for c, a in lines):
            found[m.group(1)] = lines
    return found


def scalar_writes(code):
    """Scalar registers that a vector instruction writes."""
    if not code.startswith("v_"):
        return set()
    dst = code.split(None, 1)[1].split(",")[0] if " " in code or "\t" in code else ""
    one, many = re.fullmatch(r"s(\d+)", dst), re.fullmatch(r"s\[(\d+):(\d+)\]", dst)
    if one:
        return {int(one[1])}
    return set(range(int(many[1]), int(many[2]) + 1)) if many else set()


def hazards(lines):
    bad = []
    for i, (code, app) in enumerate(lines):
        m = LOAD.search(code)
        if not (m and app):
            continue
        words, wait, j = set(range(int(m[1]), int(m[2]) + 1)), 0, i - 1
        while wait < 5 and j >= 0:
            prev = lines[j][0]
            if scalar_writes(prev) & words:
                bad.append((prev, code, wait))
            nop = re.fullmatch(r"s_nop (\d+)", prev)
            wait += int(nop[1]) + 1 if nop else 1
            j -= 1
    return bad


def test_a_planted_hazard_is_seen():
    load = ("buffer_load_dwordx4 v1, s[12:15], 0 offen lds", True)
    late = [("v_readlane_b32 s13, v40, 3", False), ("s_mov_b32 m0, s4", True), ("s_nop 0", True), load]
    assert hazards(late) and not hazards(late[:1] + [("s_nop 4", False)] + late[1:])
    assert not hazards([("v_readlane_b32 s16, v40, 3", False)] + late[1:])
    assert hazards([("v_cmp_eq_u32_e64 s[14:15], v1, v2", False)] + late[1:])


def test_assembly_loads_are_spaced(tmp_path):
    if not os.path.exists(build.HIPCC):
        pytest.skip("needs hipcc")
    out = str(tmp_path / "tl1_gemm.s")
    subprocess.run([build.HIPCC, *build.FLAGS, "--cuda-device-only", "-S",
                    os.path.join(build.CSRC, "tl1_gemm.hip"), "-o", out], check=True,
                   capture_output=True)
    with open(out) as f:
        found = kernels(f.read())
    assert len(found) >= 8  # every shape of tl1_mfma_wide_kernel
    for name, lines in found.items():
        assert not hazards(lines), (name, hazards(lines)[:3])
        assert not [c for c, app in lines if not app and re.search(r"\bm0\b", c)], name
