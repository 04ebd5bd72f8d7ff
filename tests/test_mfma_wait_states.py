"""The built kernels leave a matrix instruction the wait states its result needs before anything reads it, on every path.

The compiler fills straight-line code up; where paths of different lengths join between the matrix instruction and the reader
it may count along the longer one (csrc/conv_mfma_kernel.h, mfma_settle).  Runs on the disassembly of the library's own
gfx950 code objects; no GPU."""
import os
import re
import struct
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from cldnn_amd import hip

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
# a result of 4 passes (16 clocks) is ready after 4 + 4 wait states, one of 8 passes after 8 + 4
NEED = {"v_mfma_i32_16x16x64_i8": 8, "v_mfma_i32_32x32x32_i8": 12}
REG = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+))")


def code_objects():
    """the gfx950 ELF images inside the library (one offload bundle per translation unit)"""
    blob = open(hip.LIB_PATH, "rb").read()
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := blob.find(magic, at)) >= 0:
        count, = struct.unpack_from("<Q", blob, at + 24)
        p = at + 32
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", blob, p)
            if b"gfx950" in blob[p + 24:p + 24 + n] and size:
                yield blob[at + off:at + off + size]
            p += 24 + n
        at += len(magic)


def kernels(elf_path):
    """name -> [(instruction, operands, address)] in address order"""
    text = subprocess.run([OBJDUMP, "-d", elf_path], stdout=subprocess.PIPE, check=True, text=True).stdout
    out, ins = {}, None
    for line in text.splitlines():
        if line.startswith("\t") and "//" in line:
            body, _, tail = line.partition("//")
            op, _, operands = body.strip().partition(" ")
            ins.append((op, operands, int(tail.split(":")[0], 16)))
        elif line.endswith(">:"):
            ins = out.setdefault(line[line.index("<") + 1:-2], [])
    return out


def registers(operands):
    found = set()
    for kind, lo, hi, one in REG.findall(operands):
        found.update((kind, i) for i in (range(int(lo), int(hi) + 1) if lo else (int(one),)))
    return found


def too_early(ins):
    """[(wait states, matrix instruction, reader)] for readers that a path reaches before the result is ready"""
    index = {address: i for i, (_, _, address) in enumerate(ins)}
    used = {}

    def regs(i):
        if i not in used:
            used[i] = registers(ins[i][1])
        return used[i]

    bad = []
    for start, (op, operands, _) in enumerate(ins):
        if op not in NEED:
            assert not op.startswith("v_mfma"), "no wait states known for " + op
            continue
        result = registers(operands.split(",")[0])
        seen, work = {}, [(start + 1, 0)]
        while work:
            i, states = work.pop()
            while i < len(ins) and states < NEED[op] and seen.get(i, 99) > states:
                seen[i] = states
                name, args, address = ins[i]
                if name in NEED:
                    dst, a, b, c = (registers(x) for x in args.split(",")[:4])
                    # the next product may accumulate into the result; as an operand, or in part, it is read like by others
                    if (a | b) & result or (dst != result and dst & result) or (c != result and c & result):
                        bad.append((states, operands, " ".join(ins[i][:2])))
                    if dst & result:
                        break
                elif not name.startswith("s_") and regs(i) & result:
                    bad.append((states, operands, " ".join(ins[i][:2])))
                    break
                states += int(args, 0) + 1 if name == "s_nop" else 1
                if name == "s_endpgm":
                    break
                if name == "s_branch" or name.startswith("s_cbranch"):
                    offset = int(args.split()[0], 0)
                    target = index[address + 4 + 4 * (offset - 65536 if offset >= 32768 else offset)]
                    if name == "s_branch":
                        i = target
                        continue
                    work.append((target, states))
                i += 1
    return bad


def test_paths_are_followed():
    """the scan itself: a reader behind a join is as near as the shorter way to it"""
    mfma = ("v_mfma_i32_16x16x64_i8", "v[0:3], v[4:7], v[8:11], v[0:3]")
    put = lambda code: [(op, args, 4 * i) for i, (op, args) in enumerate(code)]
    read = ("v_add_u32_e32", "v20, v3, v21")
    assert too_early(put([mfma, ("s_cbranch_scc1", "7")] + [("s_nop", "0")] * 7 + [read, ("s_endpgm", "")])) == [(1, mfma[1], " ".join(read))]
    assert too_early(put([mfma, read, ("s_branch", "65533")])) == [(0, mfma[1], " ".join(read))]
    assert not too_early(put([mfma, ("s_nop", "7"), read, ("s_endpgm", "")]))
    assert not too_early(put([mfma, mfma, ("s_nop", "7"), read, ("s_endpgm", "")]))


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="needs the ROCm disassembler")
def test_no_result_is_read_before_its_wait_states(tmp_path):
    products, paths = 0, []
    for n, elf in enumerate(code_objects()):
        paths.append(str(tmp_path / ("%d.elf" % n)))
        with open(paths[-1], "wb") as f:
            f.write(elf)
    with ThreadPoolExecutor(4) as pool:  # four disassemblers at a time
        for found in pool.map(kernels, paths):
            for name, ins in found.items():
                products += sum(op in NEED for op, _, _ in ins)
                bad = too_early(ins)
                assert not bad, "%s: %s" % (name, bad[:3])
    assert products > 10000  # the library's kernels were found
