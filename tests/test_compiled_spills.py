"""The compiled kernels hold no vector-register spill that lanes can miss.

The register allocator can put the store of a spilled value at the head of the block that follows a
divergent loop or branch, before the instruction that switches the block's lanes on again
(s_or_b64 exec, exec, ...): lanes that are off there keep what the slot held before, and read it back
later.  A build of the fused FP32 kernel (by the compiler option -disable-promote-alloca-to-vector)
lost the sum of the convergence error over a model's blocks in this way: other Newton counts,
wrong states and NaN, the same in every run.  Which builds are hit depends on code far from the spill,
so the built library is looked at: a spill store (to scratch, or to an accumulation register) of a
value from before its block, under lanes that the same block widens afterwards."""

import re
import struct
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
LIB = ROOT / "openturbine_amd" / "libkynema_amd.so"
LLVM = Path("/opt/rocm/llvm/bin")

RESTORE = re.compile(r"s_or_b64 exec, exec, s\[")
SPILL = re.compile(r"(scratch_store|v_accvgpr_write)")
NO_DEST = re.compile(r"(ds_write|global_store|scratch_store|buffer_store|s_)")


def _registers(text):
    out = {c + n for c, n in re.findall(r"\b([va])(\d+)\b", text)}
    for c, a, b in re.findall(r"\b([va])\[(\d+):(\d+)\]", text):
        out |= {c + str(i) for i in range(int(a), int(b) + 1)}
    return out


def _operands(ins):
    parts = re.split(r",\s*(?![^\[]*\])", ins.split(None, 1)[1]) if " " in ins else []
    return (set(), _registers(ins)) if NO_DEST.match(ins) else (_registers(parts[0]) if parts else set(),
                                                                _registers(",".join(parts[1:])))


def missed_spills(blocks):
    """Blocks: lists of instructions, in program order.  Returns the spills that lanes can miss."""
    found = []
    for block in blocks:
        widen = next((k for k, i in enumerate(block) if RESTORE.match(i)), None)
        if widen is None:
            continue
        defined = set()
        for ins in block[:widen]:
            dst, src = _operands(ins)
            if SPILL.match(ins) and src and not src & defined:
                found.append(ins)
            defined |= dst
    return found


def _images(lib, tmp_path):
    """The gfx950 code objects bundled in the library."""
    fat = tmp_path / "fat.bin"
    subprocess.run([LLVM / "llvm-objcopy", f"--dump-section=.hip_fatbin={fat}", lib, tmp_path / "copy.so"], check=True)
    data, at = fat.read_bytes(), 0
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        (count,), p = struct.unpack_from("<Q", data, at + 24), at + 32
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            if size and b"gfx950" in data[p + 24: p + 24 + n]:
                yield data[at + off: at + off + size]
            p += 24 + n
        at += 24


def _blocks(listing):
    """Basic blocks of a disassembly: split at branches, at their targets and at symbols."""
    code, targets, symbols, base = [], set(), {}, None
    for line in listing.splitlines():
        if m := re.match(r"([0-9a-f]{16}) <(\S+)>:", line):
            symbols[m[2]] = int(m[1], 16)
            targets.add(int(m[1], 16))
            continue
        m = re.match(r"\s+(\S.*?)\s*// ([0-9A-F]{12}):(?:.*<(\S+?)(?:\+0x([0-9a-f]+))?>)?", line)
        if not m:
            continue
        ins, addr = m[1], int(m[2], 16)
        code.append((addr, ins))
        if m[3] and ins.startswith(("s_branch", "s_cbranch")):
            targets.add(symbols[m[3]] + int(m[4] or "0", 16))
        if ins.startswith("s_getpc_b64"):
            base = addr + 4
        elif base is not None and (k := re.match(r"s_add_u32 s\d+, s\d+, (0x[0-9a-f]+|-?\d+)$", ins)):
            off = int(k[1], 0)
            targets.add(base + (off - (1 << 32) if off >= 1 << 31 else off))
            base = None
    block = []
    for addr, ins in code:
        if addr in targets and block:
            yield block
            block = []
        block.append(ins)
        if ins.startswith(("s_branch", "s_cbranch", "s_setpc", "s_endpgm")):
            yield block
            block = []
    if block:
        yield block


def test_detector():
    lost = ["v_writelane_b32 v254, s24, 18", "s_mov_b32 s30, 0x812dea11",
            "scratch_store_dwordx4 off, v[20:23], off offset:8", "s_or_b64 exec, exec, s[8:9]"]
    assert missed_spills([lost]) == [lost[2]]
    assert missed_spills([["v_accvgpr_write_b32 a3, v7", "s_or_b64 exec, exec, s[0:1]"]])
    assert not missed_spills([[lost[0], lost[3], lost[2]]])                               # after the lanes are back
    assert not missed_spills([["v_add_f64 v[20:21], v[2:3], v[4:5]", lost[2], lost[3]]])   # the block's own value
    assert not missed_spills([lost[:3]])                                                   # no lanes come back here


def test_no_compiled_kernel_spills_a_value_some_lanes_miss(tmp_path):
    if not LIB.exists():
        subprocess.run(["make", "-s", "-C", str(ROOT / "openturbine_amd")], check=True)
    if not (LLVM / "llvm-objdump").exists():
        pytest.skip("no llvm-objdump")
    kernels = 0
    for k, image in enumerate(_images(LIB, tmp_path)):
        path = tmp_path / f"{k}.elf"
        path.write_bytes(image)
        listing = subprocess.run([LLVM / "llvm-objdump", "-d", "--no-show-raw-insn", path], check=True,
                                 capture_output=True, text=True).stdout
        kernels += len(re.findall(r"^[0-9a-f]{16} <_ZN3kyn\d+k_", listing, re.M))
        assert missed_spills(_blocks(listing)) == []
    assert kernels > 30
