"""The map from a launch's workgroups to blocks of particles
(jax-sph_amd/csrc/block_map.h, compiled on its own with g++): every block is
served once, by the XCD that serves it in a launch without the workgroups that
reduce for an earlier one."""
import ctypes
import os
import subprocess

import pytest

HDR = os.path.join(os.path.dirname(__file__), os.pardir, "jax-sph_amd", "csrc", "block_map.h")
XCDS = 8  # workgroup b of a launch runs on XCD b mod 8


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("block_map")
    src = d / "wrap.cpp"
    src.write_text('#include "%s"\nextern "C" {\n'
                   "int tail_blocks() { return sph::kTailBlocks; }\n"
                   "unsigned grid(long long b, int r) { return sph::xcd_grid(b, r); }\n"
                   "int block(int b, int g, int t, int r) "
                   "{ return sph::sweep_block_of(b, g, t != 0, r); }\n}\n" % os.path.abspath(HDR))
    so = d / "wrap.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", str(so), str(src)],
                   check=True)
    lib = ctypes.CDLL(str(so))
    lib.grid.argtypes = [ctypes.c_longlong, ctypes.c_int]
    return lib


@pytest.mark.parametrize("remap", [0, 1])
@pytest.mark.parametrize("blocks", [1, 7, 8, 9, 79, 704, 4096])
def test_tail_keeps_each_block_on_its_xcd(lib, blocks, remap):
    grid, extra = lib.grid(blocks, remap), lib.tail_blocks()
    plain = {lib.block(b, grid, 0, remap): b % XCDS for b in range(grid)}
    assert sorted(plain) == list(range(grid))
    tail = [lib.block(b, grid + extra, 1, remap) for b in range(grid + extra)]
    assert tail[:extra] == [grid] * extra     # past the last particle
    assert {l: (extra + k) % XCDS for k, l in enumerate(tail[extra:])} == plain
    assert len(tail) - extra == len(plain)
