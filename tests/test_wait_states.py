"""Wait states that inline assembly has to bring along, checked in the device code the compiler makes of the sources.

The compiler puts the wait states that gfx9's instructions need from software between instructions of its own; what stands inside an
assembly block, or between a block and the code in front of it, it does not see.  Of the blocks here two matter: a copy into LDS one
wait state behind a scalar write of m0, and a vector memory instruction five behind a vector instruction's write of a scalar
register that it reads.  A block that does not put m0 back is one more thing to look at: nothing but blocks may use it in such a
kernel."""
import os
import re
import shutil
import subprocess

import pytest

from tinytitan_amd import build


def _scalars(text):
    found = set()
    for m in re.finditer(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b", text):
        found |= set(range(int(m[1]), int(m[2]) + 1)) if m[1] else {int(m[3])}
    return found


def _missing(listing):
    function, states, m0_at, scalar_at, missing, copies, in_block, kept, writers, m0_users = "", 0, -1, {}, [], 0, False, set(), set(), set()
    for line in listing.splitlines():
        label = re.match(r"(_Z\w+):", line)
        if label:
            function, m0_at, scalar_at = label[1], -1, {}
        if "#ASMSTART" in line or "#ASMEND" in line:
            in_block = "#ASMSTART" in line
        text = line.split(";")[0].strip()
        if not text or text.startswith(".") or text.endswith(":"):
            continue
        op, _, operands = text.partition(" ")
        if op.startswith(("global_", "buffer_", "flat_", "scratch_")):
            if "lds" in op:
                copies += 1
                if m0_at >= 0 and states - m0_at < 1:
                    missing.append((function, text))
            missing += [(function, text) for s in _scalars(operands) if states - scalar_at.get(s, -9) < 5]
        states += int(operands, 0) + 1 if op == "s_nop" else 1
        target = operands.split(",")[0]
        if op.startswith("s_") and target.strip() == "m0":
            m0_at = states
        if re.search(r"\bm0\b", operands):
            if not in_block:
                m0_users.add(function)
            elif target.strip() != "m0":
                kept.add(function)  # its blocks save m0 (and put it back)
            else:
                writers.add(function)
        if op.startswith(("v_readfirstlane", "v_readlane", "v_cmp")):
            scalar_at.update({s: states for s in _scalars(target)})
    return missing, copies, (writers - kept) & m0_users


@pytest.mark.skipif(shutil.which(build.HIPCC) is None, reason="no hipcc")
@pytest.mark.parametrize("source", ["attn_prefill.hip", "affine_proj.hip"])
def test_copies_into_lds_wait_for_what_they_read(tmp_path, source):
    listing = tmp_path / "device.s"
    subprocess.run([build.HIPCC, *build.FLAGS, "--cuda-device-only", "-S", os.path.join(build.CSRC, source), "-o", str(listing)],
                   check=True, capture_output=True)
    missing, copies, clobbered = _missing(listing.read_text())
    assert copies > 50
    assert not clobbered
    assert not missing, f"{len(missing)}, e.g. {missing[0]}"
