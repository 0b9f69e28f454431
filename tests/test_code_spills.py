"""The compiler has placed the spill of a vector register at the head of a block that joins divergent lanes, before the
lanes of the other side are switched on again: their values are lost, and come back from scratch memory as whatever it
held (central detector rows of the intensity projection, where one lane of a wave had skipped a branch).  The kernels of
the built library are disassembled and searched for blocks that hold nothing but spills and scalar work ahead of the
exec mask's restore."""
import os
import re
import shutil
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "virtualcbct_amd", "libvcbct.so")
LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    """The gfx950 ELF images of the bundles in a host library's .hip_fatbin."""
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + idlen] and size:
                yield data[at + off:at + off + size]
            p += 24 + idlen
        at = data.find(MAGIC, at + 24)


def lost_spills(lines):
    """(function, block) of every join whose first vector instructions are spills, ahead of the exec restore."""
    found, fn, block, spills, clean = [], "", "", 0, True
    for line in lines:
        m = re.match(r"^[0-9a-f]* ?<(.+)>:$", line)
        if m:
            if not re.match(r"^L\d+$", m.group(1)):
                fn = m.group(1)
            block, spills, clean = m.group(1), 0, True
            continue
        t = line.split("//")[0].strip()
        if not t:
            continue
        if re.match(r"s_or_b64 exec, exec", t):
            if clean and spills:
                found.append((fn, block))
            clean = False
        elif t.startswith("scratch_store"):
            spills += 1
        elif t.startswith(("s_cbranch", "s_branch")) or "saveexec" in t or not t.startswith(
                ("s_", "v_writelane", "v_readlane")):
            clean = False
            if t.startswith(("s_cbranch", "s_branch")):  # the fall-through starts a block
                block, spills, clean = block + "+", 0, True
    return found


def test_the_search_finds_a_lost_spill():
    good = ["0 <k>:", "\tv_mov_b32 v0, 0", "\ts_cbranch_execz 9 <L0>", "\tv_mov_b32 v1, 0", "00 <L0>:",
            "\ts_or_b64 exec, exec, s[0:1]", "\tscratch_store_dword off, v0, off", "\ts_endpgm"]
    bad = good[:5] + ["\tv_writelane_b32 v9, s3, 1", good[6], good[5]]
    assert not lost_spills(good) and lost_spills(bad) == [("k", "L0")]


def test_no_spill_ahead_of_an_exec_restore(tmp_path):
    objdump = shutil.which("llvm-objdump", path=LLVM)
    if not objdump or not os.path.exists(LIB):
        pytest.skip("no disassembler or library")
    images = list(code_objects(LIB))
    assert images
    for i, image in enumerate(images):
        f = tmp_path / f"{i}.co"
        f.write_bytes(image)
        text = subprocess.run([objdump, "-d", "--symbolize-operands", str(f)], capture_output=True, text=True,
                              check=True).stdout
        found = lost_spills(text.split("\n"))
        assert not found, found
