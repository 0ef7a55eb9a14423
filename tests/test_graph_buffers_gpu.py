"""StepGraph: one, two and three steps a replay end in the held buffers as the
eager steps do, and the list keeps the positions it was built at when the
caller writes other ones into the held state."""
import numpy as np
import pytest
import torch

from oracle import nl_oracle as nlo

pytestmark = pytest.mark.gpu

js = pytest.importorskip("jax_sph_amd")
from jax_sph_amd.graph import StepGraph  # noqa: E402
from tests.test_step_gpu import _make  # noqa: E402

KEYS = ("r", "u", "v", "dudt", "dvdt", "rho", "p", "drhodt")


@pytest.mark.parametrize("steps", [1, 2, 3])
def test_replays_and_list(steps):
    case = ("tgv", {"case": {"dim": 2, "dx": 0.04}})
    cfg, state, nb, adv, *_ = _make(*case)
    st = state
    for _ in range(2 * steps):
        st, nb = adv(cfg.solver.dt, st, nb)
    _, state2, nb2, adv2, *_ = _make(*case)
    g = StepGraph(adv2, state2, nb2, cfg.solver.dt, steps_per_replay=steps)
    held = {k: v.data_ptr() for k, v in g.state.items()}
    g.replay(2)
    assert {k: v.data_ptr() for k, v in g.state.items()} == held
    for k in KEYS:
        assert torch.equal(g.state[k], st[k]), k
    n = len(state["r"])
    want = nlo.sorted_pairs(nb.idx.cpu().numpy(), n)
    g.state["r"].copy_(torch.flip(g.state["r"], [0]))
    assert np.array_equal(nlo.sorted_pairs(g.neighbors.idx.cpu().numpy(), n), want)
