"""Check of the built device code for one mistake of the compiler.

Where a divergent branch joins, the code restores the execution mask (s_or_b64 exec) before
anything is done for all lanes of a wavefront.  The register allocator of this toolchain puts a
copy that it inserts at the start of the joined block (v_mov, v_accvgpr, a scratch access) in front
of that restore when a scalar copy already stands there: the lanes that did not take the branch
then lose the value.  k_fused<0, true, kRulesOff, kDeliverAny> delivered wrong inputs that way
while its lanes' LDS addresses stayed live across the delivery (fused.hpp, the `lt` of the group
loop).  Register pressure decides whether a copy lands there, so any edit can bring one about and
no source form excludes it; the build disassembles what it has made and refuses such a block.
"""
from __future__ import annotations

import os
import re
import struct
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor

OBJDUMP = os.environ.get("LLVM_OBJDUMP", "/opt/rocm/llvm/bin/llvm-objdump")
_MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"

_FUNCTION = re.compile(r"^[0-9a-f]+ <([^>]+)>:$")
_LINE = re.compile(r"^\t(\S+)\s*(.*?)\s*// ([0-9A-F]{12}):")
_TARGET = re.compile(r"<(.+?)(?:\+0x([0-9a-f]+))?>$")
# lane copies; v_readlane and its like move between scalar registers and lanes whatever the mask
_COPY = re.compile(r"^(v_mov_b(32|64)|v_accvgpr|scratch_)")
_LANE_FREE = ("v_readlane_b32", "v_writelane_b32", "v_readfirstlane_b32", "v_nop")
_VECTOR = ("v_", "ds_", "global_", "flat_", "buffer_", "scratch_", "image_")


def code_objects(lib_path: str):
    """The gfx950 code objects in a library's bundles."""
    with open(lib_path, "rb") as f:
        data = f.read()
    out, at = [], data.find(_MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + len(_MAGIC))
        p = at + len(_MAGIC) + 8
        for _ in range(count):
            offset, size, n = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + n]:
                out.append(data[at + offset:at + offset + size])
            p += 24 + n
        at = data.find(_MAGIC, at + len(_MAGIC))
    return out


def copies_before_exec_restore(listing: str):
    """(function, address, copies) of every block of a disassembly that copies lane registers
    between its start and the s_or_b64 exec that restores the mask."""
    lines, starts, function, base = [], set(), None, {}
    for text in listing.splitlines():
        m = _FUNCTION.match(text)
        if m:
            function = m.group(1)
            base[function] = int(text.split()[0], 16)
            continue
        m = _LINE.match(text)
        if not m:
            continue
        op, args, address = m.group(1), m.group(2), int(m.group(3), 16)
        lines.append((function, op, args, address))
        if op.startswith(("s_cbranch", "s_branch")):
            t = _TARGET.search(text)
            if t and t.group(1) in base:
                starts.add(base[t.group(1)] + int(t.group(2) or "0", 16))
    found, block, copies = [], False, []
    for function, op, args, address in lines:
        if address in starts:
            block, copies = True, []
        if not block:
            continue
        if op == "s_or_b64" and args.startswith("exec, exec"):
            if copies:
                found.append((function, address, copies))
            block = False
        elif _COPY.match(op):
            copies.append(f"{op} {args}")
        elif op in _LANE_FREE:
            pass
        elif op.startswith(_VECTOR) or op.startswith(("s_cbranch", "s_branch")) or "saveexec" in op or \
                args.startswith("exec"):
            block = False
    return found


def check(lib_path: str) -> int:
    """Raises when a kernel of the library holds such a block; returns the kernels' count."""
    def one(code):
        with tempfile.NamedTemporaryFile(suffix=".co") as f:
            f.write(code)
            f.flush()
            r = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", f.name], check=True, capture_output=True, text=True)
        return copies_before_exec_restore(r.stdout), len(re.findall(r"^[0-9a-f]+ <[^>]+>:$", r.stdout, re.M))

    with ThreadPoolExecutor(max(1, min(8, os.cpu_count() or 1))) as pool:
        results = list(pool.map(one, code_objects(lib_path)))
    bad = [b for found, _ in results for b in found]
    if bad:
        raise RuntimeError(f"{lib_path}: lane registers copied in front of an exec restore (see {__name__}):\n" + "\n".join(
            f"  {fn} at 0x{at:x}: {'; '.join(c)}" for fn, at, c in bad))
    return sum(n for _, n in results)
