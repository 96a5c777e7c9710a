"""The built library's gfx950 code as the tests read it: its kernels' instructions and what their metadata say of registers."""
import os
import re
import struct
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LLVM = "/opt/rocm/llvm/bin"
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(library):
    """The device code objects in the library's offload bundles, as bytes."""
    data = open(library, "rb").read()
    at = data.find(BUNDLE)
    while at >= 0:
        entries, = struct.unpack_from("<Q", data, at + len(BUNDLE))
        pos = at + len(BUNDLE) + 8
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            triple = data[pos + 24:pos + 24 + length]
            pos += 24 + length
            if triple.startswith(b"hip") and triple.endswith(b"gfx950") and size:
                yield data[at + offset:at + offset + size]
        at = data.find(BUNDLE, at + len(BUNDLE))


def _tool(name, *args):
    return subprocess.check_output([os.path.join(LLVM, name), *args], text=True)


def kernels(library):
    """(name, [(mnemonic, operands)]) of every function of the library's device code."""
    with tempfile.TemporaryDirectory() as folder:
        for n, image in enumerate(code_objects(library)):
            path = os.path.join(folder, f"{n}.elf")
            with open(path, "wb") as f:
                f.write(image)
            name, body = None, []
            for line in _tool("llvm-objdump", "-d", "--no-show-raw-insn", path).splitlines():
                if line.startswith("\t"):
                    mnemonic, _, rest = line.split("//", 1)[0].strip().partition(" ")
                    body.append((mnemonic, rest.strip()))
                elif line.endswith(">:"):
                    if name is not None:
                        yield name, body
                    name, body = line.split("<", 1)[1][:-2], []
            if name is not None:
                yield name, body


def addresses(library, pattern):
    """[(address, mnemonic, operands)] of the one function of the library's device code whose name the pattern matches."""
    found = []
    with tempfile.TemporaryDirectory() as folder:
        for n, image in enumerate(code_objects(library)):
            path = os.path.join(folder, f"{n}.elf")
            with open(path, "wb") as f:
                f.write(image)
            names = {line.split()[-1] for line in _tool("llvm-readelf", "-sW", path).splitlines() if " FUNC " in line}
            for name in (x for x in names if re.match(pattern, x)):
                body = []
                for line in _tool("llvm-objdump", "-d", "--no-show-raw-insn", "--disassemble-symbols=" + name, path).splitlines():
                    text, _, place = line.partition("//")
                    if line.startswith("\t") and place.strip():
                        mnemonic, _, rest = text.strip().partition(" ")
                        body.append((int(place.split(":")[0], 16), mnemonic, rest.strip()))
                found.append(body)
    assert len(found) == 1, pattern
    return found[0]


def metadata(library):
    """Per kernel of the library: the integer fields of its metadata (vgpr_count, private_segment_fixed_size, ...)."""
    out = {}
    with tempfile.TemporaryDirectory() as folder:
        for n, image in enumerate(code_objects(library)):
            path = os.path.join(folder, f"{n}.elf")
            with open(path, "wb") as f:
                f.write(image)
            fields = {}
            for line in _tool("llvm-readelf", "--notes", path).splitlines():
                m = re.match(r"\s+(?:- )?\.(\w+):\s+(\S+)$", line)
                if not m:
                    continue
                if m[1] == "symbol":
                    out[m[2].removesuffix(".kd")] = fields
                elif m[1] == "agpr_count":  # the first field of a kernel's record
                    fields = {"agpr_count": int(m[2])}
                elif m[2].isdigit():
                    fields[m[1]] = int(m[2])
    return out


_REGISTERS = re.compile(r"\b(vcc_lo|vcc_hi|vcc|([vs])(?:(\d+)\b|\[(\d+):(\d+)\]))")


def registers(operand):
    """The registers that an operand names: ("v", 3), ("s", 10), vcc as ("s", "vcc_lo") and ("s", "vcc_hi")."""
    out = set()
    for whole, kind, one, first, last in _REGISTERS.findall(operand):
        if whole == "vcc":
            out |= {("s", "vcc_lo"), ("s", "vcc_hi")}
        elif whole in ("vcc_lo", "vcc_hi"):
            out.add(("s", whole))
        else:
            lo, hi = (int(one), int(one)) if one else (int(first), int(last))
            out |= {(kind, r) for r in range(lo, hi + 1)}
    return out
