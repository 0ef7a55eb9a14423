"""HIP-graph replay of fused si_euler steps.

At small particle counts a step is a dozen short kernels, and the host-side
launch cost dominates.  :class:`StepGraph` captures ``k`` fused steps once
(``torch.cuda.graph`` records every kernel the library launches on the
capture stream) and replays them as one graph launch.  Each replay advances
the held state by ``k`` steps in place: the last step leaves its results in
the held buffers and its error block in the one the first step reads, so the
error bits stay sticky from replay to replay.  Only the positions are copied
there (the list keeps those it was built at, whatever the caller then does
with the held ones); a single step, which would write what it reads, copies
everything.  Five steps of 10,000 particles took 242 us with nine copies a
replay and take 228.

The step itself allocates nothing and makes no host decisions, so the graph
replays exactly the eager computation.  The Verlet-skin rebuild test runs on
the device.  The library records no memset node: fills are kernels.  The
results are bitwise those of the eager steps (tested).  A list overflow
inside a replay shows in :attr:`did_buffer_overflow`; the caller then
re-allocates and redoes the steps eagerly, as after any overflow.
"""
from __future__ import annotations

from typing import Dict

import torch

from . import _lib
from .jax_md.partition import NeighborList


class StepGraph:
    def __init__(self, advance, state: Dict[str, torch.Tensor], neighbors: NeighborList,
                 dt: float, steps_per_replay: int = 1):
        if getattr(advance, "_sph_fusable", None) is None or \
                advance._sph_fusable(neighbors) is None:
            raise ValueError("StepGraph needs the fused step (see integrator.si_euler)")
        self.k = int(steps_per_replay)
        if self.k < 1:
            raise ValueError("steps_per_replay must be >= 1")
        self.state = {key: v.clone() for key, v in state.items()}
        self._info0 = neighbors.info
        torch.cuda.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            st, nb = self.state, neighbors
            out = {key: self.state[key] for key in advance._sph_solver.output_keys()}
            # held buffers the library can write (others are converted by the copy)
            direct = self.k > 1 and all(_lib.as_f32(v) is v for v in out.values())
            for _ in range(self.k - 1 if direct else self.k):
                st, nb = advance(dt, st, nb)
            if direct:
                st, nb = advance._sph_fused(dt, st, nb, advance._sph_fusable(nb), out=out,
                                            info=self._info0)
            for key, v in self.state.items():
                if st[key] is not v:
                    v.copy_(st[key])
            if nb.info is not self._info0:
                self._info0.copy_(nb.info)
        self.neighbors = nb
        self.replays = 0

    def replay(self, n: int = 1):
        """Advances the held state by n * steps_per_replay steps."""
        for _ in range(n):
            self.graph.replay()
        self.replays += n

    @property
    def did_buffer_overflow(self) -> bool:
        return bool(self._info0[0] & 3)
