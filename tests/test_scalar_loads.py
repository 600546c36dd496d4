"""Scalar loads and the vector stores that replace what they read.

A word of uniform address may be read through the scalar cache.  Such a load is
not ordered with vector stores, and the compiler has been seen to store to the
same word without waiting for it first (a one-thread kernel then reads its own
new value).  The library's device code is disassembled and searched for that:
a scalar load still outstanding when a store through the same base overlaps
it.  CPU only."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "gpugraph_amd", "csrc")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"

LOAD = re.compile(r"s_load_dword(?:x(\d+))? (s\d+|s\[\d+:\d+\]), s\[(\d+):(\d+)\], (0x[0-9a-f]+)$")
STORE = re.compile(r"global_(?:store|atomic)_\w+ .*\bs\[(\d+):\d+\](?: offset:(-?\d+))?(?: .*)?$")
WIDTH = {"byte": 1, "short": 2, "dword": 4, "dwordx2": 8, "dwordx3": 12, "dwordx4": 16}
DEST = re.compile(r"(?:s_\w+|v_readfirstlane_b32|v_readlane_b32) (s\d+|s\[\d+:\d+\])")


def registers(text):
    a = [int(x) for x in re.findall(r"\d+", text)]
    return range(a[0], a[-1] + 1)


def hazards(listing):
    """(kernel, load, store) for every store that overlaps an outstanding load."""
    found, kernel, pending, version = [], "", [], {}
    for line in listing.splitlines():
        head = re.match(r"^[0-9a-f]+ <(.+)>:$", line)
        if head:
            kernel, pending, version = head.group(1), [], {}
            continue
        ins = line.split("//")[0].strip()
        if ins.startswith("s_waitcnt") and ("lgkmcnt(0)" in ins or re.search(r"s_waitcnt (0x0|0)$", ins)):
            pending = []
            continue
        load = LOAD.match(ins)
        store = STORE.match(ins)
        if store:
            kind = ins.split()[0]
            width = max((w for k, w in WIDTH.items() if kind.endswith("_" + k)), default=8)
            base, off = int(store.group(1)), int(store.group(2) or 0)
            for b, v, lo, hi, text in pending:
                if b == base and v == version.get(base, 0) and lo < off + width and off < hi:
                    found.append((kernel, text, ins))
        if load:
            lo = int(load.group(5), 16)
            base = int(load.group(3))
            pending.append((base, version.get(base, 0), lo, lo + 4 * int(load.group(1) or 1), ins))
        dest = DEST.match(ins)
        if dest:
            for r in registers(dest.group(1)):
                version[r] = version.get(r, 0) + 1
    return found


def test_the_search_finds_an_overlap():
    text = """0000000000001000 <k>:
	s_load_dwordx2 s[4:5], s[0:1], 0x0   // 0
	s_waitcnt lgkmcnt(0)   // 8
	s_load_dwordx2 s[6:7], s[4:5], 0x40   // 10
	global_store_dword v0, v1, s[4:5] offset:72   // 18
	global_store_dwordx2 v0, v[2:3], s[4:5] offset:{}   // 20
"""
    assert len(hazards(text.format(64))) == 1
    assert len(hazards(text.format(68))) == 1
    assert not hazards(text.format(56))
    assert not hazards(text.format(64).replace("\tglobal_store_dwordx2", "\ts_waitcnt lgkmcnt(0)\n\tglobal_store_dwordx2"))
    assert not hazards(text.format(64).replace("\tglobal_store_dwordx2", "\ts_mov_b64 s[4:5], s[8:9]\n\tglobal_store_dwordx2"))


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
@pytest.mark.parametrize("binary", ["libgasgraph.so", "drivers/gas_bfs", "drivers/gas_pagerank"])
def test_no_store_overtakes_a_scalar_load(binary, tmp_path):
    src = os.path.join(CSRC, binary)
    if not os.path.exists(src):
        pytest.skip("not built")
    copy = shutil.copy(src, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", copy], cwd=tmp_path, check=True, capture_output=True, timeout=60)
    objects = [f for f in os.listdir(tmp_path) if f.endswith("gfx950")]
    assert objects
    loads = 0
    for f in objects:
        text = subprocess.run([OBJDUMP, "-d", f], cwd=tmp_path, check=True, capture_output=True, text=True,
                              timeout=60).stdout
        loads += text.count("s_load_dword")
        assert not hazards(text)
    assert loads > 100
