"""Chains of launches as the host side forms them (enqueue_chain), on the CPU: launches are recorded
instead of run (hip_stub)."""

import mmap

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


def _view(shape, strides):
    """A float32 array over reserved addresses, which nothing touches: launches are only recorded."""
    n = 4 * (1 + sum((e - 1) * s for e, s in zip(shape, strides)))
    buf = mmap.mmap(-1, n, flags=mmap.MAP_PRIVATE | mmap.MAP_ANONYMOUS | 0x4000)  # MAP_NORESERVE
    return np.lib.stride_tricks.as_strided(np.frombuffer(buf, np.float32, 1), shape, [4 * s for s in strides])


def test_more_work_items_than_a_launch_takes():
    """Rows that need 2^32 lanes or more run as the launches themselves, which loop over their rows;
    fewer as one chain."""
    R, C = 64, 40  # columns that are not unit: a lane for each, 64 to a row

    def launches(tasks):
        X, Y, Z = (W.T(_view((tasks, R, C), (R * C, 1, R))) for _ in range(3))
        scale = _scale_kernel(R, C)

        @workload
        def wl():
            for t in P(Dense[tasks]()):
                scale[t](x=X[t], y=Y[t])
                scale[t](x=Y[t], y=Z[t])

        return hip_stub.run(W.rr4(wl()))[0]

    assert len(launches((1 << 20) - 1)) == 1
    over = launches(1 << 20)
    assert len(over) == 2
    assert all(x.blocks * x.threads < 1 << 32 for x in over)


def test_more_row_blocks_than_a_launch_takes():
    """The same for row blocks: 64 lanes for 16 rows."""
    R, K, N = 64, 32, 32

    def launches(tasks):
        X, Y = W.T(_view((tasks, R, K), (R * K, K, 1))), W.T(_view((tasks, R, N), (R * N, N, 1)))
        Wt = W.T(np.zeros((K, N), np.float32))

        @kernel
        def proj(x: In[Tile[R, K, F32]], w: In[Tile[K, N, F32]], y: Out[Tile[R, N, F32]]):
            pto.store(y, pto.max(pto.matmul(x, w), pto.constant(0.0, F32)))

        @workload
        def wl():
            for t in P(Dense[tasks]()):
                proj[t](x=X[t], w=Wt, y=Y[t])

        return hip_stub.run(W.rr4(wl()))[0]

    assert [x.entry.split("_")[1] for x in launches((1 << 24) - 1)] == ["block"]
    over = launches(1 << 24)
    assert [x.entry.split("_")[1] for x in over] == ["tile"]
    assert over[0].blocks * over[0].threads < 1 << 32
