"""The device code of the built kernel library: its code objects, taken out of the library's offload bundles, and what the compiler's own tools say of them."""
import os
import re
import shutil
import struct
import subprocess

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _tool(name):
    found = shutil.which(name) or os.path.join("/opt/rocm/llvm/bin", name)
    assert os.path.exists(found), f"{name} not found"
    return found


def code_objects(library, folder):
    """Paths of the library's gfx950 code objects, one a source file, written into `folder`."""
    with open(library, "rb") as handle:
        data = handle.read()
    paths = []
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            target = data[entry + 24:entry + 24 + length]
            entry += 24 + length
            if b"gfx950" in target and size > 0:
                paths.append(os.path.join(str(folder), f"{len(paths)}.co"))
                with open(paths[-1], "wb") as out:
                    out.write(data[at + offset:at + offset + size])
        at = data.find(MAGIC, at + len(MAGIC))
    return paths


def kernels(path):
    """{mangled name: {field: number}} of a code object's kernels: vgpr_count, vgpr_spill_count, private_segment_fixed_size and the like."""
    notes = subprocess.run([_tool("llvm-readelf"), "--notes", path], capture_output=True, text=True, check=True).stdout
    found, fields = {}, {}
    for line in notes.splitlines():
        field = re.match(r"  ([- ]) \.(\w+):\s+(\S+)$", line)         # (a kernel's own fields; those of its arguments stand further in)
        if field is None:
            continue
        if field[1] == "-":
            fields = {}
        if field[2] == "symbol":
            found[field[3].strip("'").removesuffix(".kd")] = fields
        elif field[3].isdigit():
            fields[field[2]] = int(field[3])
    return found


def instructions(path):
    """(kernel's mangled name, instruction) of every line of a code object's disassembly."""
    kernel = None
    with subprocess.Popen([_tool("llvm-objdump"), "-d", "--no-show-raw-insn", "--no-leading-addr", path], stdout=subprocess.PIPE, text=True) as listing:
        for line in listing.stdout:
            head = re.match(r"(?:[0-9a-f]+ )?<(\w+)>:", line)
            if head is not None:
                kernel = head[1]
            elif line[:1].isspace():
                yield kernel, line.split(None, 1)[0] if line.strip() else ""
    assert listing.returncode == 0
