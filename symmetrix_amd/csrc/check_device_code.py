"""Wait states that the gfx950 instruction set leaves to the program, checked in the built library.

The compiler keeps them in code of its own; the instructions that this library writes as inline assembly are opaque to it.
The device code objects of the library (built from the sources beside this file) are listed with llvm-objdump, and every
instruction of a kind below is followed backwards, over all branches into it, through the instructions that may run right
before it:

  m0      a load from memory into LDS needs one wait state after a write of m0, which holds its LDS address
  dpp     an instruction that takes its first source from other lanes (DPP) needs two wait states after the vector
          instruction that wrote that source, and five after one that wrote the execution mask; where it is the
          double-precision multiply-add, one after a reciprocal, root or the like wrote any of its sources

Usage: check_device_code.py libsymmetrix_amd.so [llvm-objdump].  The build runs it and fails on a violation.
"""
import re
import struct
import subprocess
import sys
import tempfile

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(library):
    """The gfx950 code objects of a library's offload bundles."""
    data = open(library, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            name = data[entry + 24:entry + 24 + length]
            entry += 24 + length
            if size and b"gfx950" in name:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + len(MAGIC))


class Kernel:
    """Instructions of one function: (mnemonic, operands), and the places from which control reaches each."""

    def __init__(self, name):
        self.name, self.code, self.address, self.branches = name, [], [], []

    def add(self, mnemonic, operands, address, target):
        self.code.append((mnemonic, operands))
        self.address.append(address)
        self.branches.append(target)

    def close(self):
        index = {a: i for i, a in enumerate(self.address)}
        self.before = [[] for _ in self.code]
        for i, (mnemonic, _) in enumerate(self.code):
            if i and self.code[i - 1][0] not in ("s_branch", "s_endpgm", "s_setpc_b64"):
                self.before[i].append(i - 1)
        for i, target in enumerate(self.branches):
            if target is not None:
                self.before[index[target]].append(i)


LINE = re.compile(r"^\s+(\S+)\s*(.*?)\s*// ([0-9A-F]{12}):")
HEAD = re.compile(r"^([0-9a-f]+) <(.*)>:$")
TARGET = re.compile(r"<([^>]*?)(?:\+0x([0-9a-f]+))?>\s*$")


def kernels(listing):
    """Functions of an llvm-objdump listing."""
    found, base = [], 0
    for line in listing.splitlines():
        head = HEAD.match(line)
        if head:
            base = int(head.group(1), 16)
            found.append(Kernel(head.group(2)))
            continue
        m = LINE.match(line)
        if not m or not found:
            continue
        target = None
        if m.group(1).startswith(("s_cbranch", "s_branch")):
            t = TARGET.search(line)
            if not t or t.group(1) != found[-1].name:
                raise ValueError("branch out of its function: " + line)
            target = base + int(t.group(2) or "0", 16)
        found[-1].add(m.group(1), m.group(2), int(m.group(3), 16), target)
    for k in found:
        k.close()
    return found


def wait_states(mnemonic, operands):
    return int(operands, 0) + 1 if mnemonic == "s_nop" else 1


def reached_within(kernel, at, states, hit):
    """The nearest instructions for which hit(mnemonic, operands) holds with fewer than `states` wait states up to `at`."""
    todo, seen, out = [(b, 0) for b in kernel.before[at]], {}, []
    while todo:
        i, passed = todo.pop()
        if passed >= states or seen.get(i, states) <= passed:
            continue
        seen[i] = passed
        if hit(*kernel.code[i]):
            out.append(i)
            continue
        todo += [(b, passed + wait_states(*kernel.code[i])) for b in kernel.before[i]]
    return out


def writes_m0(mnemonic, operands):
    return operands.split(",")[0].strip() == "m0" and mnemonic.startswith("s_") and not mnemonic.startswith("s_cmp")


REGISTERS = re.compile(r"v\[(\d+):(\d+)\]|v(\d+)")


def vector_registers(operand):
    m = REGISTERS.match(operand.strip())
    if not m:
        return set()
    return {int(m.group(3))} if m.group(3) else set(range(int(m.group(1)), int(m.group(2)) + 1))


def written_by_vector(mnemonic, operands):
    """Vector registers that a vector arithmetic instruction writes."""
    if not mnemonic.startswith("v_") or mnemonic.startswith(("v_cmp", "v_readlane", "v_readfirstlane")):
        return set()
    parts = operands.split(",")
    out = vector_registers(parts[0])
    if "swap" in mnemonic and len(parts) > 1:      # (both operands change)
        out |= vector_registers(parts[1])
    return out


TRANSCENDENTAL = ("v_rcp", "v_rsq", "v_sqrt", "v_exp", "v_log", "v_sin", "v_cos")


def violations(kernel):
    """Texts, and how many instructions of the kinds above there are."""
    bad, looked_at = [], 0
    for i, (mnemonic, operands) in enumerate(kernel.code):
        if "load_lds" in mnemonic or (mnemonic.startswith("buffer_load") and operands.endswith(" lds")):
            looked_at += 1
            for j in reached_within(kernel, i, 1, writes_m0):
                bad.append(f"{kernel.name}: {mnemonic} at {kernel.address[i]:x} right after m0 was written at {kernel.address[j]:x}")
        if "_dpp" in mnemonic:
            looked_at += 1
            parts = operands.split(",")
            source = vector_registers(parts[1])
            rules = [(2, lambda m, o: written_by_vector(m, o) & source, "its first source was written"),
                     (5, lambda m, o: m.startswith("v_cmpx"), "the execution mask was written")]
            if mnemonic.startswith("v_fmac_f64"):
                sources = set().union(*(vector_registers(p) for p in parts[:3]))
                rules.append((1, lambda m, o: m.startswith(TRANSCENDENTAL) and written_by_vector(m, o) & sources, "a source was written"))
            for states, hit, what in rules:
                for j in reached_within(kernel, i, states, hit):
                    bad.append(f"{kernel.name}: {mnemonic} at {kernel.address[i]:x} too soon after {what} at {kernel.address[j]:x}")
    return bad, looked_at


def check(library, objdump="llvm-objdump"):
    bad, looked_at = [], 0
    for image in code_objects(library):
        with tempfile.NamedTemporaryFile(suffix=".elf") as f:
            f.write(image)
            f.flush()
            listing = subprocess.run([objdump, "-d", f.name], check=True, capture_output=True, text=True).stdout
        for kernel in kernels(listing):
            b, n = violations(kernel)
            bad += b
            looked_at += n
    return bad, looked_at


if __name__ == "__main__":
    bad, looked_at = check(*sys.argv[1:3])
    for line in bad[:20]:
        print(line, file=sys.stderr)
    if bad or not looked_at:
        sys.exit(f"{len(bad)} of {looked_at} instructions lack their wait states" if looked_at else "no device code found")
