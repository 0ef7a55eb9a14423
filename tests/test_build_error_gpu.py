"""A build that ends early leaves nothing behind: after a call that returns an
error part of the way (here one that a call before it left in the runtime, found
at the first launch), the next build of the workspace gives the lists and the
occupancy of an undisturbed one."""
import numpy as np
import pytest
import torch

from oracle import nl_oracle as nlo

pytestmark = pytest.mark.gpu

js = pytest.importorskip("jax_sph_amd")
from jax_sph_amd import _lib, case_setup, partition  # noqa: E402
from jax_sph_amd.ensemble import Ensemble  # noqa: E402
from jax_sph_amd.jax_md import space  # noqa: E402
from tests.test_step_gpu import _make  # noqa: E402

FIELDS = ("r", "u", "v", "dudt", "dvdt", "rho", "p")


def _leave_an_error():
    """A refused call: the runtime keeps its error for whoever asks next."""
    torch.cuda.synchronize()
    assert _lib.lib().hipSetDevice(1 << 20) != 0


@pytest.mark.parametrize("dim,n", [(2, 9000), (3, 9000), (3, 700)])
def test_list(dim, n):
    r = np.random.default_rng(dim).random((n, dim)).astype(np.float32)
    cutoff = 0.02 if dim == 2 else 0.09
    disp, _ = space.periodic(side=np.ones(dim))
    fn = partition.neighbor_list(disp, np.ones(dim), r_cutoff=cutoff, format=partition.Sparse)
    t = torch.tensor(r, device="cuda")
    nb = fn.allocate(t)
    want = nlo.sorted_pairs(nb.idx.cpu().numpy(), n)
    _leave_an_error()
    with pytest.raises(_lib.SphError):
        nb.update(t)
    after = nb.update(t)
    assert torch.equal(after.info[:4], nb.info[:4])
    assert np.array_equal(nlo.sorted_pairs(after.idx.cpu().numpy(), n), want)


@pytest.mark.parametrize("skin", ["auto", 0.0])
@pytest.mark.parametrize("dx", [0.01, 0.02])
def test_step(dx, skin):
    case = ("tgv", {"case": {"dim": 2, "dx": dx}}, "jaxmd_vmap", skin)
    cfg, state, nb, adv, *_ = _make(*case)
    ref, ref_nb = adv(cfg.solver.dt, state, nb)
    ref, ref_nb = adv(cfg.solver.dt, ref, ref_nb)
    _, state, nb, adv, *_ = _make(*case)
    _leave_an_error()
    with pytest.raises(_lib.SphError):
        adv(cfg.solver.dt, state, nb)
    st, nb = adv(cfg.solver.dt, state, nb)
    st, nb = adv(cfg.solver.dt, st, nb)
    assert torch.equal(nb.info[:4], ref_nb.info[:4])
    for k in FIELDS:
        assert torch.equal(st[k], ref[k]), k


def test_ensemble():
    def members():
        return Ensemble.from_configs([
            case_setup.load_config("tgv", {"case": {"dim": 2, "dx": dx}}) for dx in (0.02, 0.0125)])
    ref, ens = members(), members()
    ref.step(2)
    _leave_an_error()
    with pytest.raises(_lib.SphError):
        ens.step()
    ens.step(2)
    for k in range(2):
        assert torch.equal(ens.error_info(k)[:4], ref.error_info(k)[:4])
        for f in FIELDS:
            assert torch.equal(ens.state(k)[f], ref.state(k)[f]), (k, f)
