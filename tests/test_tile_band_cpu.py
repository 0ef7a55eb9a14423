"""The bounds of the matrix-core pair build (jax-sph_amd/csrc/tile_band.h,
compiled on its own with g++): for every particle that passes as inside its
cell, what the expanded square can lose fits in the band that is left to the
exact filter, by the worst case and by pairs near the cutoff evaluated as the
kernel does."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HDR = os.path.join(os.path.dirname(__file__), os.pardir, "jax-sph_amd", "csrc", "tile_band.h")
F = np.float32


@pytest.fixture(scope="module")
def band(tmp_path_factory):
    d = tmp_path_factory.mktemp("tile_band")
    src = d / "wrap.cpp"
    src.write_text('#include "%s"\nextern "C" void band(const float* box, const float* cell, '
                   "int dim, float reach, float cutoff_sq, float* out) {\n"
                   "  const sph::TileBand t = sph::tile_band(box, cell, dim, reach, cutoff_sq);\n"
                   "  out[0] = t.lo; out[1] = t.hi;\n"
                   "  for (int k = 0; k < 3; ++k) out[2 + k] = t.inside[k];\n}\n"
                   % os.path.abspath(HDR))
    so = d / "wrap.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", str(so), str(src)],
                   check=True)
    lib = ctypes.CDLL(str(so))

    def call(box, cell, reach):
        box, cell = np.asarray(box, F), np.asarray(cell, F)
        out = np.zeros(5, F)
        p = [x.ctypes.data_as(ctypes.c_void_p) for x in (box, cell, out)]
        lib.band(p[0], p[1], len(box), ctypes.c_float(reach), ctypes.c_float(F(reach) * F(reach)),
                 p[2])
        return float(out[0]), float(out[1]), out[2:2 + len(box)].astype(np.float64)
    return call


GRIDS = [([1.0, 1.0], 5), ([1.0, 1.0, 1.0], 5), ([2 * np.pi] * 3, 21), ([2 * np.pi] * 3, 200),
         ([0.9, 1.7, 1.2], 7), ([0.999] * 3, 5), ([7.99] * 3, 5), ([1.0, 1.0], 900), ([5.4, 2.1], 40)]


def _grid(box, cells):
    box = np.asarray(box, F)
    reach = F(box.min() / F(cells) * F(0.999))
    return box, (box / np.floor(box / reach)).astype(F), reach


@pytest.mark.parametrize("box,cells", GRIDS)
def test_worst_case(band, box, cells):
    box, cell, reach = _grid(box, cells)
    lo, hi, inside = band(box, cell, reach)
    ulp_box = float(np.nextafter(box.max(), F(np.inf)) - box.max())
    # particles within the grid pass as inside
    assert np.all(inside >= 0.5 * cell + 2 * ulp_box)
    loss = 15 * 2.0 ** -24 * (2 * np.sqrt((inside ** 2).sum()) + float(reach)) ** 2
    metric = 2 * float(reach) * np.sqrt(3) * 3 * ulp_box
    r_sq = float(F(reach) * F(reach))
    rounding = float(np.spacing(F(hi)))   # of the band's own ends
    assert r_sq - lo >= loss + metric - rounding and hi - r_sq >= loss + metric - rounding


def _fma(a, b, c):
    return (a.astype(np.float64) * b + c).astype(F)


@pytest.mark.parametrize("box,cells", GRIDS)
def test_pairs_at_the_cutoff(band, box, cells):
    box, cell, reach = _grid(box, cells)
    lo, hi, inside = band(box, cell, reach)
    dim, n = len(box), 200_000
    rng = np.random.default_rng(cells)
    o = ((rng.integers(0, np.floor(box / cell).astype(int), (n, dim)) + F(0.5)).astype(F) * cell)
    # up to the edge of `inside`, many in its corners; the other particle at the cutoff
    s = rng.uniform(-1, 1, (n, dim))
    s = np.where(rng.random((n, dim)) < 0.5, np.sign(s), s)
    pa = (o + s * inside).astype(F)
    v = rng.normal(size=(n, dim))
    v *= (float(reach) * (1 + rng.uniform(-1e-6, 1e-6, (n, 1)))) / np.linalg.norm(v, axis=1,
                                                                               keepdims=True)
    pb = (pa + v).astype(F)
    a, b = (pa - o).astype(F), (pb - o).astype(F)
    ok = np.all(np.abs(a) <= inside.astype(F), axis=1)
    assert ok.mean() > 0.1

    def square(x):
        t = (x[:, 0] * x[:, 0]).astype(F)
        for k in range(1, dim):
            t = _fma(x[:, k], x[:, k], t)
        return t
    mid = F(0.5) * (F(lo) + F(hi))
    width = 0.5 * (F(hi) - F(lo))
    d = _fma(square(a), np.ones(n, F), (square(b) - mid).astype(F))
    for k in range(dim):
        d = _fma(F(-2) * a[:, k], b[:, k], d)
    true = ((pa.astype(np.float64) - pb) ** 2).sum(1) - float(F(reach) * F(reach))
    decided = ok & (np.abs(d) >= width)
    assert np.all((d < 0)[decided] == (true < 0)[decided])
    # and the loss itself is within the band
    assert np.abs(d - true)[ok].max() < float(width)
