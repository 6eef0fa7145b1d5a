"""Scratch memory of the built gfx950 kernels, read from the library's own code objects: the
contact and pair-test kernels are chains of dependent work on few waves, and every register that
they spill lengthens the chain. The power of the cohesive separation depth, inlined, took 68
registers of them, the rim point of a cylinder (an arc tangent, a sine and a cosine) 59."""
import os
import re
import shutil
import struct
import subprocess
import tempfile

import pytest

import xdynamics_dll_amd._lib as _lib

TOOLS = [p for p in ("/opt/rocm/llvm/bin", "/opt/rocm/lib/llvm/bin") if os.path.exists(p + "/llvm-readelf")]
READELF = TOOLS[0] + "/llvm-readelf" if TOOLS else shutil.which("llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    """The gfx950 code objects of the offload bundles in a library."""
    blob = open(path, "rb").read()
    at = blob.find(MAGIC)
    while at >= 0:
        n = struct.unpack_from("<Q", blob, at + 24)[0]
        p = at + 32
        for _ in range(n if n < 16 else 0):   # not a bundle: the string alone
            off, size, tl = struct.unpack_from("<QQQ", blob, p)
            triple = blob[p + 24: p + 24 + tl]
            if b"gfx950" in triple and size:
                yield blob[at + off: at + off + size]
            p += 24 + tl
        at = blob.find(MAGIC, at + len(MAGIC))


def kernels():
    """Scratch bytes a lane of every kernel, by demangled name."""
    out = {}
    for obj in code_objects(_lib.LIB_PATH):
        with tempfile.NamedTemporaryFile(suffix=".o") as f:
            f.write(obj)
            f.flush()
            notes = subprocess.run([READELF, "--notes", f.name], capture_output=True, text=True).stdout
        for block in notes.split("- .agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\S+)", block).group(1)
            out[name] = int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", block).group(1))
    names = subprocess.run(["c++filt"], input="\n".join(out), capture_output=True, text=True).stdout.splitlines()
    return {n.replace("(anonymous namespace)::", "").replace("xdem::", "").replace("void ", "").split("(")[0]: v
            for n, v in zip(names, out.values())}


@pytest.mark.skipif(not READELF or not shutil.which("c++filt"), reason="needs llvm-readelf and c++filt")
def test_scratch_of_the_contact_kernels():
    k = kernels()
    collide = {n: v for n, v in k.items() if n.startswith("k_collide<")}
    assert len(collide) == 64
    plain = {n: v for n, v in collide.items() if n.endswith("false>")}   # no cylinder bodies
    assert max(plain.values()) <= 16, plain
    one = {n: v for n, v in plain.items() if n.split(", ")[1] == "false"}   # one scene
    assert len(one) == 16 and max(one.values()) == 0, one
    cyl = {n: v for n, v in collide.items() if n not in plain}   # three slots by index: 144
    assert len(cyl) == 32 and max(cyl.values()) <= 256, cyl
    for name in ("k_p2p<", "k_touch<"):
        some = {n: v for n, v in k.items() if n.startswith(name)}
        assert some and max(some.values()) == 0, some
