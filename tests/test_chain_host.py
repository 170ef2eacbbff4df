"""Chains of launches as the host side forms them (enqueue_chain), on the CPU: launches are recorded
instead of run (hip_stub)."""

import math
import mmap

import numpy as np

import hip_stub
import pytest
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


def _llama_blocks(n, d, mlp, st=128, ts=64):
    """n llama blocks (attention, add, rmsnorm, MLP, add), each reading what the one before it wrote."""
    def new(*shape):
        return np.zeros(shape, np.float32)

    xs = [new(st, ts, d) for _ in range(n + 1)]
    X, KT = [W.T(x) for x in xs], [W.T(x.transpose(0, 2, 1)) for x in xs]
    W1, W2 = ([W.T(new(*s)) for _ in range(n)] for s in ((d, mlp), (mlp, d)))
    Attn, Res, Xn, Mlp = (W.T(new(st, ts, d)) for _ in range(4))

    @kernel
    def attn(q: In[Tile[ts, d, F32]], k_t: In[Tile[d, ts, F32]], v: In[Tile[ts, d, F32]], out: Out[Tile[ts, d, F32]]):
        s = pto.mul(pto.matmul(q, k_t), pto.constant(1.0 / math.sqrt(d), F32))
        e = pto.exp(pto.sub(s, pto.rowmax(s)))
        pto.store(out, pto.matmul(pto.div(e, pto.rowsum(e)), v))

    @kernel
    def add(a: In[Tile[ts, d, F32]], b: In[Tile[ts, d, F32]], out: Out[Tile[ts, d, F32]]):
        pto.store(out, pto.add(a, b))

    @kernel
    def rmsnorm(x: In[Tile[ts, d, F32]], out: Out[Tile[ts, d, F32]]):
        pto.store(out, pto.mul(x, pto.rsqrt(pto.rowmean(pto.mul(x, x)))))

    @kernel
    def mlp_relu(x: In[Tile[ts, d, F32]], w1: In[Tile[d, mlp, F32]], w2: In[Tile[mlp, d, F32]], out: Out[Tile[ts, d, F32]]):
        pto.store(out, pto.matmul(pto.max(pto.matmul(x, w1), pto.constant(0.0, F32)), w2))

    @workload
    def wl():
        for s in P(Dense[st]()):
            for i in range(n):
                attn[s](q=X[i][s], k_t=KT[i][s], v=X[i][s], out=Attn[s])
                add[s](a=X[i][s], b=Attn[s], out=Res[s])
                rmsnorm[s](x=Res[s], out=Xn[s])
                mlp_relu[s](x=Xn[s], w1=W1[i], w2=W2[i], out=Mlp[s])
                add[s](a=Res[s], b=Mlp[s], out=X[i + 1][s])

    return W.rr4(wl())


def _norms(n, C):
    X = [W.T(np.zeros((4, 16, C), np.float32)) for _ in range(n + 1)]

    @kernel
    def rmsnorm(x: In[Tile[16, C, F32]], out: Out[Tile[16, C, F32]]):
        pto.store(out, pto.mul(x, pto.rsqrt(pto.rowmean(pto.mul(x, x)))))

    @workload
    def wl():
        for s in P(Dense[4]()):
            for i in range(n):
                rmsnorm[s](x=X[i][s], out=X[i + 1][s])

    return W.rr4(wl())


# Chained whole, in part (the MLP's width refused), not at all (a row's registers), and by as many
# views as a chain has slots.
@pytest.mark.parametrize("make,per_8", [(lambda n: _llama_blocks(n, 64, 128), 8), (lambda n: _llama_blocks(n, 256, 512), 16),
                                        (lambda n: _norms(n, 4096), 8), (lambda n: _norms(n, 128), 1)])
def test_host_time_is_linear_in_launches(make, per_8):
    """Eight times the launches cost about eight times the host time (the search that tried every
    length from every start: 50 times and more)."""
    few, t_few = hip_stub.run(make(8), passes=20)
    many, t_many = hip_stub.run(make(64), passes=20)
    assert len(few) == per_8
    assert t_many <= 20 * t_few


def test_error_comes_after_the_launches_before_it():
    """A launch whose tiles leave their tensor is an error at its own turn: those before it run."""
    R, C = 16, 32
    X, Y, Z = (W.T(np.zeros((4, R, C), np.float32)) for _ in range(3))
    scale = _scale_kernel(R, C)

    @workload
    def wl():
        for t in P(Dense[4]()):
            scale[t](x=X[t], y=Y[t])
        for t in P(Dense[4]()):
            scale[t](x=Y[t], y=Z[t])
        for t in P(Dense[4]()):
            scale[t](x=Z[t], y=Y[t + 1])

    with pytest.raises(RuntimeError, match="tiles of param y"):
        hip_stub.run(W.rr4(wl()))
    assert hip_stub.recorded() == ["ptowsp_rows_scale"]  # the first two, chained
