"""What the compiler wrote about the kernels of a built libtdvmc.so: registers,
scratch, static LDS (its code objects' metadata notes)."""
import os
import re
import struct
import subprocess
import tempfile

READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def kernels(path):
    """{demangled name: {vgpr_count, vgpr_spill_count, private_segment_fixed_size, group_segment_fixed_size}}"""
    data = open(path, "rb").read()
    out = {}
    at = data.find(MAGIC)
    while at >= 0:
        p = at + len(MAGIC)
        (n,) = struct.unpack_from("<Q", data, p)
        p += 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen].decode()
            p += 24 + idlen
            if "gfx" not in name or size == 0:
                continue
            with tempfile.NamedTemporaryFile(suffix=".co") as f:
                f.write(data[at + off:at + off + size])
                f.flush()
                notes = subprocess.run([READELF, "--notes", f.name], capture_output=True, text=True, check=True).stdout
            for block in re.split(r"\n\s+- (?=\.(?:agpr_count|args):)", notes)[1:]:
                sym = re.search(r"^\s*\.name:\s+(_Z\S+)$", block, re.M)
                if sym:
                    out[sym.group(1)] = {k: int(v) for k, v in re.findall(r"\.(vgpr_count|vgpr_spill_count|private_segment_fixed_size|"
                                                                           r"group_segment_fixed_size):\s+(\d+)", block)}
        at = data.find(MAGIC, at + 1)
    names = list(out)
    plain = subprocess.run(["c++filt"], input="\n".join(names), capture_output=True, text=True, check=True).stdout.splitlines()
    return {d: out[m] for m, d in zip(names, plain)}
