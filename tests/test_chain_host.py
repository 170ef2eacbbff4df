"""Chains of launches as the host side forms them (enqueue_chain), on the CPU: launches are recorded
instead of run (hip_stub)."""

import numpy as np

import hip_stub
import workloads as W
from pto_wsp import Dense, In, Out, P, Tile, kernel, pto, workload

F32 = W.F32


def _scale_kernel(R, C):
    @kernel
    def scale(x: In[Tile[R, C, F32]], y: Out[Tile[R, C, F32]]):
        pto.store(y, pto.mul(x, pto.constant(2.0, F32)))

    return scale


def test_eight_grid_loops_and_every_slot():
    """A nest of the most loops has no variable left for a loop of the launches; twelve views fill
    the slots, and each keeps its strides."""
    R, C = 4, 8
    X, Y = ([W.T(np.zeros((2, R, C), np.float32)) for _ in range(6)] for _ in range(2))
    scale = _scale_kernel(R, C)
    one, two = Dense[1](), Dense[2]()

    @workload
    def wl():
        for a in P(two):
            for b in P(one):
                for c in P(one):
                    for d in P(one):
                        for e in P(one):
                            for f in P(one):
                                for g in P(one):
                                    for h in P(one):
                                        for i in range(6):
                                            scale[a, b, c, d, e, f, g, h](x=X[i][a], y=Y[i][a])

    launches, _ = hip_stub.run(W.rr4(wl()))
    assert len(launches) == 1
    assert launches[0].s3 == [C] * 12 and launches[0].s4 == [1] * 12
    assert launches[0].coef == [[R * C] + [0] * 7] * 12
