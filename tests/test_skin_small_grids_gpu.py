"""Skin lists on grids of three and four cells a side, where every cell is next
to a face: pair sets, occupancy and error bits of each step, with rebuilds among
them, against the oracle's per-step search."""
import numpy as np
import pytest

from oracle import nl_oracle as nlo

pytestmark = pytest.mark.gpu

js = pytest.importorskip("jax_sph_amd")
from tests.test_step_gpu import _make  # noqa: E402


@pytest.mark.parametrize("dim,side,kernel", [(2, 11, "QSK"), (2, 13, "QSK"), (2, 9, "WC2K"),
                                             (3, 11, "QSK"), (3, 13, "QSK"), (3, 9, "WC2K")])
def test_skin_lists(dim, side, kernel):
    dx = 2 * np.pi / side if dim == 3 else 1 / side
    cfg, state, nb, adv, R, *_ = _make("tgv", {
        "case": {"dim": dim, "dx": dx, "r0_noise_factor": 0.2}, "kernel": {"name": kernel},
        "solver": {"dt": None}})
    assert nb.workspace.skin_on
    ref_nb = R.ns.allocate(state["r"].cpu().numpy())
    st, rebuilds = state, 0
    for k in range(16):
        if k % 5 == 4:
            nb.workspace.tune("skin_rebuild", 1)
        st, nb = adv(cfg.solver.dt, st, nb)
        r = st["r"].cpu().numpy()
        ref_nb = R.ns.update(r, ref_nb)
        info = nb.info.cpu().numpy()
        rebuilds += int(info[7] > 0)
        assert int(info[0]) == int(ref_nb.error) and int(info[1]) == ref_nb.occupancy, k
        if int(ref_nb.error):
            break   # the reference's pairs are then incomplete by design
        assert np.array_equal(nlo.sorted_pairs(nb.idx.cpu().numpy(), len(r)),
                              nlo.sorted_pairs(ref_nb.idx, len(r))), k
    assert rebuilds >= 1
