"""LDS reads written as inline asm are in flight until a wait that the source writes itself; the compiler takes their
destinations as written at once. So on no path may an instruction touch such a register before the wait, and a path
that leaves the reads unused has to wait too: there the compiler gives the registers to other values, addresses among
them, which the landing data would overwrite. This compiles the attention kernels for gfx950 and follows every path
through the emitted code."""
import os
import re
import shutil
import subprocess
from pathlib import Path

import pytest

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
CSRC = Path(__file__).resolve().parent.parent / "torchair_amd" / "csrc"


def _regs(text):
    out = set()
    for kind in "va":
        out |= {(kind, int(m.group(1))) for m in re.finditer(rf"\b{kind}(\d+)\b", text)}
        for m in re.finditer(rf"\b{kind}\[(\d+):(\d+)\]", text):
            out |= {(kind, i) for i in range(int(m.group(1)), int(m.group(2)) + 1)}
    return frozenset(out)


def _parse(lines):
    """[(instruction, written as inline asm, registers)] and the index each label stands before."""
    ins, labels, inline = [], {}, False
    for line in lines:
        if "#ASMSTART" in line or "#ASMEND" in line:
            inline = "#ASMSTART" in line
            continue
        text = line.split(";")[0].strip()
        if m := re.match(r"(\.?L\w+):", text):
            labels[m.group(1)] = len(ins)
        elif text and not text.startswith(".") and not text.endswith(":"):
            ins.append((text, inline, _regs(text)))
    return ins, labels


def _after_wait(pending, text):
    """The LDS operations that may still be in flight after an s_waitcnt (they complete in order)."""
    if m := re.search(r"lgkmcnt\((\d+)\)", text):
        n = int(m.group(1))
    elif m := re.match(r"s_waitcnt\s+(0x[0-9a-f]+|\d+)$", text):
        n = (int(m.group(1), 0) >> 8) & 0xF
    else:
        return pending
    return pending if n >= len(pending) else pending[len(pending) - n:] if n else ()


def touched_in_flight(lines, only_past=None):
    """(instruction, read) pairs that meet on some path. only_past: count a read only once an instruction starting
    so has been passed (which leaves out paths that cannot be taken, where one flag decides two branches)."""
    ins, labels = _parse(lines)
    found, seen, work = set(), set(), [(0, ())]
    while work:
        i, pending = work.pop()
        while i < len(ins):
            text, inline, regs = ins[i]
            op = text.split()[0]
            if op == "s_waitcnt":
                pending = _after_wait(pending, text)
            else:
                found |= {(text, ins[at][0]) for dst, at, past in pending if past and dst & regs}
                if only_past and op.startswith(only_past):
                    pending = tuple((dst, at, True) for dst, at, _ in pending)
                if op.startswith(("ds_", "s_load", "s_buffer_load")):
                    read = inline and op.startswith("ds_read")
                    dst = _regs(text.split(None, 1)[1].split(",")[0]) if read else frozenset()
                    pending += ((dst, i, read and not only_past),)
            if op == "s_endpgm":
                break
            if op.startswith(("s_branch", "s_cbranch")):
                nexts = [labels[text.split()[1]]] + ([i + 1] if op != "s_branch" else [])
                for n in nexts:
                    key = (n, tuple((at, past) for _, at, past in pending))
                    if key not in seen:
                        seen.add(key)
                        work.append((n, pending))
                break
            i += 1
    return sorted(found)


def test_the_scan_sees_reads_left_in_flight():
    read = [";;#ASMSTART", "ds_read_b128 v[4:7], v1", ";;#ASMEND"]
    wait = [";;#ASMSTART", "s_waitcnt lgkmcnt(0)", ";;#ASMEND"]
    use = ["v_add_f32_e32 v0, v4, v5", "s_endpgm"]
    assert touched_in_flight(read + wait + use) == []
    assert touched_in_flight(read + use) == [("v_add_f32_e32 v0, v4, v5", "ds_read_b128 v[4:7], v1")]
    # the register given to another value on a path that skips the wait
    branch = read + ["s_cbranch_scc0 .LBB0_2"] + wait + use + [".LBB0_2:", "v_mov_b32_e32 v6, v9", "s_endpgm"]
    assert [t for t, _ in touched_in_flight(branch)] == ["v_mov_b32_e32 v6, v9"]
    assert touched_in_flight(branch, only_past="global_atomic_swap") == []
    # in order: one younger read may stay
    two = read + [";;#ASMSTART", "ds_read_b128 v[8:11], v1", ";;#ASMEND", "s_waitcnt lgkmcnt(1)"]
    assert touched_in_flight(two + use) == []
    assert touched_in_flight(two + ["v_mov_b32_e32 v0, v8", "s_endpgm"]) != []


@pytest.mark.skipif(not shutil.which(HIPCC) and not Path(HIPCC).exists(), reason="hipcc not available")
@pytest.mark.parametrize("source,kernels", [
    ("attention_packed", [("packed_kernel", 4, None)]),
    ("attention_tiled", [("mla_rows_kernel", 2, None)]),
    # the prefill's fast pass gives an item up (an atomic marks it) while value reads are in flight
    ("attention", [("paged_decode_kernel", 6, None), ("paged_decode8_kernel", 12, None), ("mla_decode", 4, None),
                   ("prefill_kernel", 8, "global_atomic_swap")]),
])
def test_no_register_of_a_read_in_flight_is_touched(tmp_path, source, kernels):
    out = tmp_path / f"{source}.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fhip-fp32-correctly-rounded-divide-sqrt",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wno-unused-result",
                    "--cuda-device-only", "-S", str(CSRC / f"{source}.hip"), "-o", str(out)], check=True, capture_output=True)
    text = out.read_text()
    for name, count, past in kernels:
        starts = [m.start() for m in re.finditer(rf"^_ZN3tai\w*{name}\w*:", text, re.M)]
        assert len(starts) == count, name
        for start in starts:
            body = text[start:text.index(".section", start)].splitlines()
            assert any("ds_read" in line for line in body)
            assert touched_in_flight(body, only_past=past) == [], body[0]
