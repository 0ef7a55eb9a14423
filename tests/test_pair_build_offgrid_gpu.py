"""Exact lists of positions that are not in their cell: outside the box (clamped
into its outer cells), not finite, or both next to pairs at the cutoff.  The
unordered list, from the matrix cores, holds for each sender the receivers of
one side of its id that the ordered list holds, whose build compares candidate by
candidate."""
import numpy as np
import pytest
import torch

from oracle import nl_oracle as nlo

pytestmark = pytest.mark.gpu

js = pytest.importorskip("jax_sph_amd")
from jax_sph_amd import partition  # noqa: E402
from jax_sph_amd.jax_md import space  # noqa: E402


def _positions(dim, cells, kind, seed):
    """Particles of a unit box, most of the outer ones at the cutoff from another."""
    rng = np.random.default_rng(seed)
    n = 1500 if dim == 3 else 900
    cutoff = np.float32(0.9995 / cells)
    r = rng.random((n, dim))
    v = rng.normal(size=(n // 2, dim))
    v *= cutoff * (1 + rng.uniform(-3e-7, 3e-7, (n // 2, 1))) / np.linalg.norm(v, axis=1,
                                                                             keepdims=True)
    out = rng.random((n // 2, dim)) < 0.4
    side = rng.random((n // 2, dim)) < 0.5
    beyond = rng.uniform(0, 0.6 / cells, (n // 2, dim))
    r[:n // 2] = np.where(out, np.where(side, -beyond, 1 + beyond), r[:n // 2])
    r[n // 2:2 * (n // 2)] = r[:n // 2] + v
    r = r.astype(np.float32)
    if kind == "not finite":
        bad = rng.integers(0, n, 12)
        r[bad[:4], 0] = np.nan
        r[bad[4:8], dim - 1] = np.inf
        r[bad[8:]] = -np.inf
    return r, cutoff


@pytest.mark.parametrize("kind", ["outside", "not finite"])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("cells", [5, 7])
def test_lists_agree(dim, cells, kind):
    r, cutoff = _positions(dim, cells, kind, 10 * dim + cells)
    n = len(r)
    disp, _ = space.periodic(side=np.ones(dim))
    t = torch.tensor(r, device="cuda")
    got = {}
    for fmt in (partition.Sparse, partition.OrderedSparse):
        fn = partition.neighbor_list(disp, np.ones(dim), r_cutoff=float(cutoff), format=fmt,
                                     capacity_multiplier=2.0)
        nb = fn.allocate(t)
        assert not bool(nb.did_buffer_overflow)
        got[fmt] = nlo.sorted_pairs(nb.idx.cpu().numpy(), n)
    full, half = got[partition.Sparse], got[partition.OrderedSparse]
    assert len(half[0]) > n
    # the format keeps the receivers of one side of the sender's id
    for keep in (full[0] < full[1], full[0] > full[1]):
        if np.array_equal(full[:, keep], half):
            break
    else:
        raise AssertionError("the ordered list is no half of the unordered one")
    bad = ~np.isfinite(r).all(1)
    assert not bad[full].any()
