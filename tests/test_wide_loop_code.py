"""The built wide-loop kernels (PipeMainWide), read back from the library: their
MFMAs are inline asm whose wait states the compiler does not place, so the
sums are right only where the generated code keeps what the source counts on.
Every one works in place on accumulation registers; between the first and the
last of a stretch nothing else touches an accumulator and nothing spills; no
vector instruction writes an operand of an MFMA right before it; an
accumulator comes back only after many others; and the fences' wait states
stand between the MFMAs and any other access to the accumulators."""

import re
import shutil
import struct
import subprocess
from pathlib import Path

import pytest

from kernrelay_amd import build

LLVM = Path("/opt/rocm/llvm/bin")
APART = 3   # instructions between a vector write and the MFMA that reads it
BACK = 16   # MFMAs between two on one accumulator


def code_objects(lib, tmp):
    """The gfx950 code objects of a host library."""
    fat = tmp / "fatbin"
    subprocess.run([LLVM / "llvm-objcopy", "--dump-section", ".hip_fatbin=%s" % fat, lib, tmp / "unused"], check=True)
    data = fat.read_bytes()
    for m in re.finditer(rb"__CLANG_OFFLOAD_BUNDLE__", data):
        at = m.start()
        (n,), o = struct.unpack_from("<Q", data, at + 24), at + 32
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", data, o)
            triple = data[o + 24:o + 24 + length]
            o += 24 + length
            if b"gfx950" in triple and size:
                f = tmp / ("%d_%d.elf" % (at, off))
                f.write_bytes(data[at + off:at + off + size])
                yield f


def registers(operand):
    m = re.match(r"([va])\[(\d+):(\d+)\]$", operand)
    if m:
        return {(m.group(1), i) for i in range(int(m.group(2)), int(m.group(3)) + 1)}
    m = re.match(r"([va])(\d+)$", operand)
    return {(m.group(1), int(m.group(2)))} if m else set()


def operands(ins):
    return [o.strip() for o in ins.split(None, 1)[1].split(",")] if " " in ins else []


def faults(code):
    """What is wrong with a kernel's instructions."""
    bad = []
    at = [i for i, ins in enumerate(code) if ins.startswith("v_mfma")]
    if not at:
        return ["no MFMA"]
    seen = {}
    for n, i in enumerate(at):
        d, a, b, c = operands(code[i])[:4]
        if d != c or not d.startswith("a["):
            bad.append("not in place: " + code[i])
        for back in range(1, APART + 1):
            q = code[i - back]
            if q.startswith("v_") and not q.startswith("v_mfma") and registers(operands(q)[0]) & (
                    registers(a) | registers(b) | registers(c)):
                bad.append("%s right before %s" % (q, code[i]))
        if d in seen and n - seen[d] < BACK:
            bad.append("%d MFMAs apart: %s" % (n - seen[d], code[i]))
        seen[d] = n
    for ins in code[at[0]:at[-1]]:
        if ins.startswith(("v_accvgpr", "scratch_")) or (
                not ins.startswith("v_mfma") and any(k == "a" for o in operands(ins) for k, _ in registers(o))):
            bad.append("among the MFMAs: " + ins)

    def fenced(stretch):  # two s_nop 15 before the accumulators are touched
        nops = 0
        for ins in stretch:
            nops += ins == "s_nop 15"
            if nops >= 2:
                return True
            if any(k == "a" for o in operands(ins) for k, _ in registers(o)):
                return False
        return False

    if not fenced(code[at[-1] + 1:]):
        bad.append("no wait states after the last MFMA")
    if not fenced(reversed(code[:at[0]])):
        bad.append("no wait states before the first MFMA")
    return bad


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Instructions of every wide-loop kernel of the library, by name."""
    if not (LLVM / "llvm-objdump").exists() or not build.LIB.exists():
        pytest.skip("needs the ROCm LLVM tools and the built library")
    tmp = tmp_path_factory.mktemp("code")
    found = {}
    for elf in code_objects(build.LIB, tmp):
        table = subprocess.run([LLVM / "llvm-objdump", "-t", elf], check=True, capture_output=True, text=True).stdout
        names = sorted(set(re.findall(r"_ZN2kr\S*GemmPipeKernel\S*Lb0ELi3E\S*GemmParamsE$", table, re.M)))
        if not names:
            continue
        text = subprocess.run([LLVM / "llvm-objdump", "-d", "--no-show-raw-insn", "--no-leading-addr",
                               "--disassemble-symbols=" + ",".join(names), elf], check=True, capture_output=True,
                              text=True).stdout
        name = None
        for line in text.splitlines():
            m = re.match(r"^<(\S+)>:$", line.strip())
            if m:
                name = m.group(1) if m.group(1) in names else name
                found.setdefault(name, [])
            elif name and line.startswith("\t"):
                found[name].append(line.split("//")[0].strip())
    shutil.rmtree(tmp)
    return found


def test_wide_loop_code(kernels):
    assert len(kernels) == 6  # two types, three tiles
    for name, code in kernels.items():
        assert sum(ins.startswith("v_mfma") for ins in code) >= 128, name
        assert not faults(code), (name, faults(code)[:5])


def test_the_reading_finds_planted_faults():
    fence = ["s_nop 15", "s_nop 15"]
    loop = ["v_mfma_f32_16x16x32_bf16 a[%d:%d], v[0:3], v[4:7], a[%d:%d]" % (4 * i, 4 * i + 3, 4 * i, 4 * i + 3)
            for i in range(32)] * 2
    head = ["v_accvgpr_write_b32 a0, 0"] + fence + ["s_barrier"]
    good = head + loop + fence + ["v_accvgpr_read_b32 v0, a0"]
    assert faults(good) == []
    for planted in ("v_accvgpr_read_b32 v9, a3", "v_mov_b32_e32 v4, v9", "scratch_load_dword v9, off, s0", good[19]):
        assert faults(good[:20] + [planted] + good[20:]), planted
    assert faults(head + [loop[0].replace("a[0:3], v", "a[4:7], v")] + good[len(head) + 1:])
    assert faults(good[:-3] + good[-1:]) and faults(good[:1] + good[3:])
