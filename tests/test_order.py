"""The red-black passes of one launch hand maps from block to block, across the
XCDs' caches: the built propagation kernels have to acquire at device scope
between taking a ring entry and the block's first read of a map, and to release
between a tile's last barrier and its announcement.  Read from the library's own
device code (no GPU)."""
import os
import re
import shutil
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "patchmatch_amd", "libpmp.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    d = tmp_path_factory.mktemp("code")
    shutil.copy(LIB, d / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=d, check=True, capture_output=True, timeout=60)
    out = {}
    for f in sorted(os.listdir(d)):
        if not f.endswith("gfx950"):
            continue
        text = subprocess.run([OBJDUMP, "-d", f], cwd=d, check=True, capture_output=True, text=True, timeout=120).stdout
        for name, body in re.findall(r"^[0-9a-f]+ <(_ZN3pmp13k_propagate_q\w+)>:\n(.*?)(?=^[0-9a-f]+ <|\Z)", text, re.M | re.S):
            out[name] = [line.split("//")[0].strip() for line in body.splitlines()]
    return out


def test_handed_over_maps_are_ordered(kernels):
    assert len(kernels) == 16   # edge modes x tile sizes x forms (the wide form has two tile sizes)
    for name, code in kernels.items():
        swap = max(k for k, c in enumerate(code) if c.startswith("global_atomic_swap "))
        barrier = next(k for k in range(swap, len(code)) if code[k].startswith("s_barrier"))
        assert "buffer_inv sc1" in code[swap:barrier], f"{name}: no acquire between the ring and the block's reads"
        announce = max(k for k, c in enumerate(code) if c.startswith("global_atomic_cmpswap "))
        barrier = max(k for k in range(announce) if code[k].startswith("s_barrier"))
        stores = max(k for k in range(barrier) if code[k].startswith("global_store"))
        assert any(re.match(r"s_waitcnt .*vmcnt\(0\)", c) for c in code[stores:barrier]), f"{name}: stores in flight"
        tail = code[barrier:announce]
        arrival = next(k for k, c in enumerate(tail) if c.startswith("global_atomic_add "))
        assert "buffer_wbl2 sc1" in tail[:arrival], f"{name}: arrivals do not release"
        written = tail.index("buffer_wbl2 sc1")
        assert any(re.match(r"s_waitcnt .*vmcnt\(0\)", c) for c in tail[written:arrival]), f"{name}: write-back not waited for"
        assert "buffer_inv sc1" in tail[arrival:], f"{name}: the last arrival does not acquire the others'"
        assert "buffer_wbl2 sc1" in tail[arrival:], f"{name}: the ring entry does not release"
