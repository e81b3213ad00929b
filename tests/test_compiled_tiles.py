"""What the compiler made of bfaintb_prefill_wreg_kernel, whose accumulators are accumulation registers by name (acc_reserve in
bfaintb_prefill_wreg.hpp) and whose matrix instructions are assembly that its bookkeeping does not see into: that nothing else uses those
registers, that no ordinary instruction writes a matrix instruction's operands in the two wait states before it, and that a step waits for memory where
it says so and nowhere else."""
import os
import re
import shutil
import struct
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
KERNEL = b"bfaintb_prefill_wreg_kernelILi"


def code_objects(library):
    """The gfx950 code objects of a library built from several sources, one bundle each."""
    data = open(library, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        (count,), pos = struct.unpack_from("<Q", data, at + len(MAGIC)), at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            if data[pos + 24:pos + 24 + length].endswith(b"gfx950") and size:
                yield data[at + offset:at + offset + size]
            pos += 24 + length
        at = data.find(MAGIC, at + 1)


def registers(operand):
    m = re.fullmatch(r"([va])\[(\d+):(\d+)\]", operand) or re.fullmatch(r"([va])(\d+)()", operand)
    return {(m[1], i) for i in range(int(m[2]), int(m[3] or m[2]) + 1)} if m else set()


def check_listing(lines):
    """(matrix instructions, what is wrong) of a kernel's instructions."""
    count, wrong, before = 0, [], []
    for line in lines:
        op, _, rest = line.partition(" ")
        args = [a.split()[0] for a in re.split(r",(?![^\[]*\])", rest) if a.strip()]
        if op.startswith("v_mfma"):
            count += 1
            if args[0] != args[3] or {r[0] for r in registers(args[0])} != {"a"} or "a" in {r[0] for x in args[1:3] for r in registers(x)}:
                wrong.append(line)
            operands, states = registers(args[1]) | registers(args[2]), 0
            for was, was_args in reversed(before):
                if states >= 2:
                    break
                if was.startswith("v_") and not was.startswith("v_mfma") and was_args and registers(was_args[0]) & operands:
                    wrong.append("%s %s, then %s" % (was, was_args, line))
                states += int(was_args[0], 0) + 1 if was == "s_nop" else 1
        elif any(r[0] == "a" for x in args for r in registers(x)):
            if not (op == "v_accvgpr_write_b32" and args[1] == "0") and op != "v_accvgpr_read_b32":
                wrong.append(line)
        before = (before + [(op, args)])[-3:]
    return count, wrong


def memory_waits(lines, instructions):
    """What the waits for memory among the first so many matrix instructions leave in flight."""
    count, left = 0, []
    for line in lines:
        count += line.startswith("v_mfma")
        m = re.search(r"vmcnt\((\d+)\)", line)
        if m and 0 < count < instructions:
            left.append(int(m[1]))
    return left


def test_the_checks_see_what_they_are_for():
    mfma = "v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]"
    assert check_listing(["v_accvgpr_write_b32 a0, 0", "v_mov_b32_e32 v4, v9", "s_nop 1", mfma, "v_accvgpr_read_b32 v1, a2"]) == (1, [])
    for listing in (["v_accvgpr_write_b32 a0, v7"], ["v_accvgpr_mov_b32 a1, a0"], ["ds_read_b128 a[4:7], v3"], ["v_mov_b32_e32 v4, v9", "s_nop 0", mfma],
                    ["v_mfma_f32_16x16x32_bf16 a[4:7], v[0:3], v[4:7], a[0:3]"]):
        assert len(check_listing(listing)[1]) == 1, listing


@pytest.mark.skipif(not shutil.which(LLVM + "/llvm-objdump"), reason="no disassembler")
def test_nothing_but_the_matrix_instructions_uses_the_accumulators(tmp_path):
    import awesome_fusion_amd as af
    if not os.path.exists(af.library_path()):
        af.build_library(verbose=False)
    seen = {}
    for i, code in enumerate(c for c in code_objects(af.library_path()) if KERNEL in c):
        path = str(tmp_path / ("%d.co" % i))
        open(path, "wb").write(code)
        notes = subprocess.run([LLVM + "/llvm-readelf", "--notes", path], check=True, capture_output=True, text=True).stdout
        for entry in re.split(r"\n  - \.agpr_count:", notes)[1:]:
            name = re.search(r"\.name: +(\S+)", entry)[1]
            form = re.search(r"bfaintb_prefill_wreg_kernelILi(\d)ELb(\d)ELb(\d)ELi(\d+)E", name)
            if form:
                figures = {key: int(re.search(r"\.%s: +(\d+)" % key, entry)[1]) for key in ("vgpr_spill_count", "private_segment_fixed_size")}
                assert int(entry.split()[0]) == 16 * int(form[4]) and not any(figures.values()), (name, entry.split()[0], figures)
                seen[name] = None
        listing = subprocess.run([LLVM + "/llvm-objdump", "-d", "--no-show-raw-insn", "--no-leading-addr", path], check=True, capture_output=True, text=True).stdout
        for part in listing.split("\n<")[1:]:
            name, _, body = part.partition(">:\n")
            if name in seen:
                lines = [x.split("//")[0].strip() for x in body.split("\n") if x.strip()]
                packed, blocks = map(int, re.search(r"ILi\dELb\dELb(\d)ELi(\d+)E", name).groups())
                # twelve steps are written out (a loop of six, up to six behind it): one wait at a step's barrier and, of packed codes, one at its
                # start (the first step's stands before its first matrix instruction); none of them for the last copies
                waits = memory_waits(lines, 12 * 8 * blocks)
                seen[name] = check_listing(lines) + (len(waits) - (23 if packed else 12), min(waits))
    assert len(seen) == 40, sorted(seen)
    for name, (count, wrong, more_waits, least) in seen.items():
        assert count >= 12 * 8 * 8 and not wrong, (name, count, wrong[:5])
        assert more_waits == 0 and least >= 4, (name, more_waits, least)
