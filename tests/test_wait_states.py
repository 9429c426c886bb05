"""Wait states around lane reads in the built GPU code: a vector instruction that reads a scalar register
written by v_readlane / v_readfirstlane stands at least two wait states after it (an instruction is one, s_nop N
is N + 1).  The compiler keeps this for the instructions it generates; inside inline assembly nobody does."""
import os
import re
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
SREG = re.compile(r"s\[(\d+):(\d+)\]|\bs(\d+)\b|\bvcc\b")


def sregs(op):
    out = set()
    for m in SREG.finditer(op):
        if m.group(3):
            out.add(int(m.group(3)))
        elif m.group(1):
            out.update(range(int(m.group(1)), int(m.group(2)) + 1))
        else:
            out.add("vcc")
    return out


def too_close(listing):
    """(function, instruction) of every read that comes too early."""
    found, written, t, fn = [], {}, 0, ""
    for line in listing.splitlines():
        if line.endswith(">:"):
            fn, written = line.split("<")[-1][:-2], {}
            continue
        ins = line.split("//")[0].strip()
        if not re.match(r"[vs]_|ds_|buffer_|global_|flat_|scratch_", ins):
            continue
        mn, _, rest = ins.partition(" ")
        ops = [o.strip() for o in rest.split(",")]
        if mn == "s_nop":
            t += int(ops[0], 0) + 1
            continue
        if mn.startswith("v_"):
            # a second destination (carry, scale flag, 64-bit product) is no source; a lane select has a rule of its own
            first = 2 if re.search(r"_co_|div_scale|v_mad_[ui]64", mn) else 1
            for o in ops[first:2] if mn.startswith("v_readlane") else ops[first:]:
                if any(t - written[r] < 2 for r in sregs(o) if r in written):
                    found.append((fn, ins))
        t += 1
        if mn.startswith(("v_readlane", "v_readfirstlane")):
            written.update((r, t) for r in sregs(ops[0]))
        elif mn.startswith("s_"):
            for r in sregs(ops[0]):
                written.pop(r, None)
            if mn.startswith(("s_branch", "s_cbranch", "s_setpc", "s_swappc", "s_endpgm")):
                written = {}
    return found


def test_rule_on_a_listing():
    code = "0 <f>:\n\tv_readlane_b32 s4, v1, 3 // 0\n%s\tv_writelane_b32 v2, s4, 3 // 8\n"
    assert too_close(code % "") == [("f", "v_writelane_b32 v2, s4, 3")]
    assert len(too_close(code % "\ts_nop 0 // 4\n")) == 1
    assert too_close(code % "\ts_nop 1 // 4\n") == []
    assert too_close(code % "\tv_mov_b32_e32 v7, v8 // 4\n\ts_nop 0 // 6\n") == []


def test_built_library(tmp_path):
    from fortrancfd_amd.build import LIB
    if not os.path.isfile(OBJDUMP):
        pytest.skip("no llvm-objdump")
    lib = tmp_path / "lib.so"
    os.symlink(LIB, lib)
    subprocess.run([OBJDUMP, "--offloading", str(lib)], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    objects = sorted(p for p in os.listdir(tmp_path) if p.endswith("gfx950"))
    assert objects
    for p in objects:
        out = subprocess.run([OBJDUMP, "-d", p], cwd=tmp_path, check=True, capture_output=True, text=True).stdout
        bad = too_close(out)
        assert not bad, f"{len(bad)} reads too early, the first: {bad[:3]}"
