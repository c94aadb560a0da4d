"""The global-to-LDS copies that psoci_amd/csrc/strsig.hip writes as asm, in
the assembly it compiles to: a copy takes its LDS address from M0, and the
instruction after a write to M0 may not be such a copy (one wait state); an
address base in scalar registers may not come from a vector instruction within
five wait states.  The compiler keeps these rules for its own instructions and
not inside asm."""
import os
import re
import subprocess

import pytest

from psoci_amd import build

HIPCC = build.HIPCC


def _violations(lines):
    code, copies, bad = [], 0, []
    for line in lines:
        line = line.split(";")[0].strip()
        if not line or line.startswith((".", "//")) or line.endswith(":"):
            continue
        if "global_load_lds" in line:
            copies += 1
            if code and re.match(r"s_\w+ m0,", code[-1]):
                bad.append((code[-1], line))
            base = re.search(r"s\[(\d+):(\d+)\]", line)
            if base:
                regs = set(range(int(base[1]), int(base[2]) + 1))
                states = 0
                for prev in reversed(code[-5:]):
                    w = re.match(r"v_read(?:first)?lane_b32 s(\d+)", prev)
                    if w and int(w[1]) in regs and states < 5:
                        bad.append((prev, line))
                    nop = re.match(r"s_nop (\d+)", prev)
                    states += 1 + (int(nop[1]) if nop else 0)
        code.append(line)
    return copies, bad


def test_scan_finds_missing_wait_states():
    adjacent = ["s_mov_b32 m0, s3", "global_load_lds_dwordx4 v[6:7], off"]
    assert _violations(adjacent) == (1, [tuple(adjacent)])
    apart = ["s_mov_b32 m0, s3", "s_nop 0", "global_load_lds_dwordx4 v[6:7], off"]
    assert _violations(apart) == (1, [])
    base = ["v_readfirstlane_b32 s4, v1", "s_mov_b32 m0, s3", "s_nop 0", "global_load_lds_dwordx4 v2, s[4:5]"]
    assert len(_violations(base)[1]) == 1


def test_copies_wait_for_m0(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    out = str(tmp_path / "strsig.s")
    subprocess.run([HIPCC, *[f for f in build.FLAGS if f != "-fPIC"], "-x", "hip", "--cuda-device-only", "-S",
                    os.path.join(build.CSRC, "strsig.hip"), "-o", out], check=True, capture_output=True)
    with open(out) as f:
        copies, bad = _violations(f)
    assert copies > 0
    assert not bad, bad[:3]
