"""Registers of the sweeps in the built library: no scratch memory, and no more
registers than the wavefronts a SIMD they are meant to run with allow, also
with the workgroup that reduces an earlier launch's partials compiled in."""
import os
import re
import shutil
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "jax-sph_amd", "jax_sph_amd", "libsph.so")
READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(path):
    """The gfx950 code objects of the library's offload bundles, one a source."""
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, name = struct.unpack_from("<QQQ", data, p)
            triple = data[p + 24:p + 24 + name]
            p += 24 + name
            if b"gfx950" in triple and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(LIB) or not os.path.exists(READELF):
        pytest.skip("needs the built library and llvm-readelf")
    out, d = {}, tmp_path_factory.mktemp("code")
    for k, code in enumerate(_code_objects(LIB)):
        f = d / f"{k}.o"
        f.write_bytes(code)
        notes = subprocess.run([READELF, "--notes", str(f)], check=True, capture_output=True,
                               text=True).stdout
        for part in notes.split(".agpr_count:")[1:]:
            name = re.search(r"\.name: +(\S+)", part).group(1)
            out[name] = {key: int(re.search(rf"\.{key}: +(\d+)", part).group(1))
                         for key in ("private_segment_fixed_size", "vgpr_count")}
    assert out, "no code object found"
    return out


# kernels and the registers their wavefronts a SIMD allow: density, walls and the
# standard force without extras at eight wavefronts, the Riemann force of any
# kernel function at seven (2D) and six, the delta-SPH force with extras at six
LIMITS = {rf"k_{name}ILi{dim}E": 64 for name in ("density", "walls") for dim in (2, 3)}
LIMITS.update({rf"k_forceILi{dim}ELi{kind}ELi0ELb{tvf}ELb0E": 64
               for dim in (2, 3) for kind in (1, 2) for tvf in (0, 1)})
LIMITS.update({r"k_forceILi2ELin1ELi1ELb0ELb0E": 72, r"k_forceILi3ELin1ELi1ELb0ELb0E": 80,
               r"k_forceILi3ELi[12]ELi2ELb1ELb1E": 80})


@pytest.mark.parametrize("pattern", list(LIMITS))
def test_registers(kernels, pattern):
    found = {k: v for k, v in kernels.items() if re.search(pattern, k) and "_ens" not in k}
    assert found, "kernel missing from the library"
    for name, r in found.items():
        assert r["private_segment_fixed_size"] == 0, name
        assert r["vgpr_count"] <= LIMITS[pattern], name
