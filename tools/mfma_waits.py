"""Results of matrix instructions that are read too early, in the assembly of this package's own libraries (CPU only).

    python tools/mfma_waits.py                                   # every kernel of the three libraries: a minute
    python tools/mfma_waits.py --lib path.so --kernels REGEX

The vector unit may read what a matrix instruction writes a fixed number of wait states behind it, and it is the compiler that counts them.  Where
paths meet behind matrix instructions of different lengths it has counted the shorter one's: the K = 16 product of fp8 numbers on one path, the K = 64
one, eight states longer, on the other.  Such a read comes too early now and then, with no error.

From every matrix instruction all paths are followed until its result is whole; every other instruction is a state (s_nop its own number), a branch that is
taken five and one that is not two, which is less than either takes.  Products that read or replace the result end a path: the hardware waits."""
import argparse
import os
import re
import struct
import subprocess
import sys
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIBS = [os.path.join(ROOT, "nano-vllm-hw3_amd", "nanovllm", "_lib", f"lib{n}.so") for n in ("qlinear", "seqmix", "hymix")]
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
REGISTER = re.compile(r"\b([av])(?:(\d+)\b|\[(\d+):(\d+)\])")


def code_objects(path):
    """The gfx950 code objects inside a library."""
    with open(path, "rb") as f:
        data = f.read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        count, p = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(count):
            offset, size, n = struct.unpack_from("<QQQ", data, p)
            if size and b"gfx950" in data[p + 24:p + 24 + n]:
                yield data[at + offset:at + offset + size]
            p += 24 + n
        at = data.find(magic, at + 24)


def kernels(code, names):
    """(name, instructions) of a code object's kernels and functions whose name matches; an instruction is (op, operands, index a branch goes to)."""
    with tempfile.NamedTemporaryFile(suffix=".o") as f:
        f.write(code)
        f.flush()
        symbols = subprocess.run([OBJDUMP, "-t", f.name], capture_output=True, text=True, check=True).stdout
        wanted = [s for s in re.findall(r"F \.text\s+\S+(?:\s+\.\w+)?\s+(\S+)", symbols) if re.search(names, s)]
        if not wanted:
            return
        text = subprocess.run([OBJDUMP, "-d", "--disassemble-symbols=" + ",".join(wanted), f.name], capture_output=True, text=True, check=True).stdout
    for part in re.split(r"\n(?=[0-9a-f]{16} <)", text)[1:]:
        instructions, place = [], {}
        for line in part.split("\n")[1:]:
            m = re.match(r"\t(\S+)\s*(.*?)\s*// ([0-9A-F]+): ([0-9A-F]{8})", line)
            if m:
                place[int(m[3], 16)] = len(instructions)
                offset = int(m[4][4:], 16)
                instructions.append((m[1], m[2], int(m[3], 16) + 4 + 4 * (offset - (offset >> 15 << 16))))
        yield re.search(r"<(\S+)>", part)[1], [(op, r, place.get(to) if op.startswith(("s_branch", "s_cbranch")) else None) for op, r, to in instructions]


def passes(op):
    """Passes of four cycles."""
    if "f8f6f4" in op:
        return 16 if "32x32x64" in op else 8
    if "_f64" in op:
        return 16
    m = re.search(r"(\d+)x\d+x(\d+)", op)
    rows, k = int(m[1]), int(m[2])
    if rows == 32:
        return 8 if k >= 8 else 16
    return 4 if k >= 16 else 8


def registers(text):
    found = set()
    for kind, one, first, last in REGISTER.findall(text):
        found.update((kind, i) for i in (range(int(first), int(last) + 1) if first else (int(one),)))
    return found


def early_reads(code):
    """(matrix instruction, reader, states between them, states needed) of a kernel."""
    found = []
    for i, (op, rest, _) in enumerate(code):
        if not op.startswith(("v_mfma", "v_smfmac")):
            continue
        result = registers(rest.split(",")[0])
        need = passes(op) + 3 - (re.search(r"x[24]_f32", op) is not None)
        best, paths = {}, [(i + 1, 0)]
        while paths:
            j, states = paths.pop()
            if j is None or j >= len(code) or states >= need or best.get(j, need) <= states:
                continue
            best[j] = states
            o, r, to = code[j]
            if o.startswith(("v_mfma", "v_smfmac")):
                if not registers(r) & result:
                    paths.append((j + 1, states + 1))
            elif o == "s_nop":
                paths.append((j + 1, states + int(r, 0) + 1))
            elif o == "s_branch":
                paths.append((to, states + 5))
            elif o.startswith("s_cbranch"):
                paths += [(to, states + 5), (j + 1, states + 2)]
            elif o != "s_endpgm":
                reads = registers(r.partition(",")[2] if o[0] == "v" else r) & result
                if o[0] in "vdgb" and (reads or (states < need - 1 and registers(r) & result)):
                    found.append((op, f"{o} {r}", states, need))
                else:
                    paths.append((j + 1, states + 1))
    return found


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--lib", action="append")
    ap.add_argument("--kernels", default="")
    args = ap.parse_args()
    short = count = 0
    for lib in args.lib or LIBS:
        for code in code_objects(lib):
            for name, instructions in kernels(code, args.kernels):
                count += 1
                for op, reader, states, need in early_reads(instructions):
                    short += 1
                    print(f"{name}: {op} is read by '{reader}' after {states} states, {need} are needed", flush=True)
        print(f"{lib}: {count} kernels so far", flush=True)
    sys.exit(1 if short else 0)


if __name__ == "__main__":
    main()
