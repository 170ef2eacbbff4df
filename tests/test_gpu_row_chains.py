"""Chains of row-program launches run as one kernel: reads forwarded in registers, loops unrolled,
stores made once.  Against the oracle, which runs the launches one after the other.

Elementwise results, maxima and copies are exact; sums of n terms in another order are within
n * 2^-24 relative for positive terms (rtol 2^-23 * n covers both sides)."""

import numpy as np
import pytest

import workloads as W
from oracle.runner import run_workload
from pto_wsp import Dense, In, InOut, Out, P, Tile, kernel, pto, workload

pytestmark = pytest.mark.gpu
F32 = W.F32


def _both(make, arrs, launches):
    ga, ca = ({k: v.copy() for k, v in arrs.items()} for _ in range(2))
    prog = make(ga).compile(target="hip_gfx950")
    prog.execute()
    prog.synchronize()
    ref = run_workload(make(ca))
    assert prog.stats.total_cycles == ref.total_cycles and prog.stats.task_count == ref.task_count
    assert prog.stats.launches == launches
    return ga, ca


@pytest.mark.parametrize("B,S,V,launches", [(1, 8, 512, 1), (2, 72, 512, 1), (3, 40, 256, 3)])
def test_three_phase_softmax(gpu, B, S, V, launches):
    """Two P.seq launches and a P() launch over the same views are one pass; overlapping views
    (V = 256) are not."""
    lg = np.random.default_rng(V + S).standard_normal((B, S, V)).astype(np.float32)
    ga, ca = _both(lambda a: W.rr4(W.softmax3(a)), W.softmax3_arrays(lg), launches)
    np.testing.assert_array_equal(ga["rmax"], ca["rmax"])
    np.testing.assert_allclose(ga["rsum"], ca["rsum"], rtol=V * 2.0 ** -23)
    np.testing.assert_allclose(ga["probs"], ca["probs"], rtol=V * 2.0 ** -22, atol=1e-9)


def _three(a, R, C, dt=F32):
    """t = x * g; u = t - rowmax(t); out = u / m (m [R, 1]); a [1, C] vector g; t and u are stored."""
    X, G, M, T_, U, O = W.T(a["x"]), W.T(a["g"]), W.T(a["m"]), W.T(a["t"]), W.T(a["u"]), W.T(a["out"], dt)
    n, nt = a["x"].shape[:2]

    @kernel
    def k1(x: In[Tile[R, C, F32]], g: In[Tile[1, C, F32]], t: Out[Tile[R, C, F32]]):
        pto.store(t, pto.mul(x, g))

    @kernel
    def k2(t: In[Tile[R, C, F32]], u: Out[Tile[R, C, F32]]):
        pto.store(u, pto.sub(t, pto.rowmax(t)))

    @kernel
    def k3(u: In[Tile[R, C, F32]], m: In[Tile[R, 1, F32]], out: Out[Tile[R, C, dt]]):
        pto.store(out, pto.div(u, m))

    @workload
    def wl():
        for b in P(Dense[n]()):
            for i in P(Dense[nt]()):
                k1[b, i](x=X[b][i], g=G, t=T_[b][i])
                k2[b, i](t=T_[b][i], u=U[b][i])
                k3[b, i](u=U[b][i], m=M[b][i], out=O[b][i])

    return W.rr4(wl())


# Even and masked widths, rows that do not fill a wave, many rows per lane team, a 16-bit store.
@pytest.mark.parametrize("R,C,dt", [(3, 64, F32), (8, 19, F32), (4, 101, F32), (5, 512, F32), (1, 1001, F32), (16, 8, F32),
                                    (4, 96, W.BF16), (2, 33, W.F16)])
def test_row_chain(gpu, R, C, dt):
    rng = np.random.default_rng(C)
    a = {"x": rng.standard_normal((2, 3, R, C)), "g": rng.uniform(0.5, 2, (1, C)), "m": rng.uniform(0.5, 2, (2, 3, R, 1)),
         "t": np.zeros((2, 3, R, C)), "u": np.zeros((2, 3, R, C)), "out": np.zeros((2, 3, R, C))}
    a = {k: v.astype(np.float32) for k, v in a.items()}
    if dt != F32:
        a["out"] = a["out"].astype(np.float16 if dt == W.F16 else np.uint16)
    ga, ca = _both(lambda x: _three(x, R, C, dt), a, 1)
    for k in ("t", "u", "out"):
        np.testing.assert_array_equal(ga[k].view(np.uint8), ca[k].view(np.uint8))


def test_row_chain_that_would_cross_rows(gpu):
    """A launch that reads another row's tile of what the launch before it wrote is not chained."""
    n, R, C = 6, 4, 32
    x = np.random.default_rng(0).standard_normal((n, R, C)).astype(np.float32)

    def make(a):
        X, T_, O = W.T(a["x"]), W.T(a["t"]), W.T(a["out"])

        @kernel
        def copy(s: In[Tile[R, C, F32]], d: Out[Tile[R, C, F32]]):
            pto.store(d, pto.mul(s, s))

        @workload
        def wl():
            for i in P(Dense[n - 1]()):
                copy[i](s=X[i], d=T_[i + 1])
            for i in P(Dense[n - 1]()):
                copy[i](s=T_[i], d=O[i])

        return W.rr4(wl())

    ga, ca = _both(make, {"x": x, "t": x.copy(), "out": np.zeros_like(x)}, 2)
    np.testing.assert_array_equal(ga["out"], ca["out"])


def test_row_chain_loop_accumulators(gpu):
    """Two loops over the same steps, the second reading what the first wrote in every step and the
    accumulator it left, in place; then a launch without the loop."""
    n, L, R, C = 3, 5, 4, 48
    rng = np.random.default_rng(2)
    a = {"x": rng.uniform(0.5, 1.5, (n, L, R, C)), "y": np.zeros((n, L, R, C)), "s": rng.uniform(0, 1, (n, R, 1)), "z": np.zeros((n, R, 1))}
    a = {k: v.astype(np.float32) for k, v in a.items()}

    def make(t):
        X, Y, S, Z = (W.T(t[k]) for k in ("x", "y", "s", "z"))

        @kernel
        def first(x: In[Tile[R, C, F32]], y: Out[Tile[R, C, F32]], s: InOut[Tile[R, 1, F32]]):
            pto.store(y, pto.mul(x, pto.constant(2.0, F32)))
            pto.store(s, pto.max(s, pto.rowmax(x)))

        @kernel
        def second(y: InOut[Tile[R, C, F32]], s: In[Tile[R, 1, F32]]):
            pto.store(y, pto.sub(y, s))

        @kernel
        def third(s: In[Tile[R, 1, F32]], z: Out[Tile[R, 1, F32]]):
            pto.store(z, pto.mul(s, pto.constant(3.0, F32)))

        @workload
        def wl():
            for i in P(Dense[n]()):
                for j in P.seq(Dense[L]()):
                    first[i, j](x=X[i][j], y=Y[i][j], s=S[i])
            for i in P(Dense[n]()):
                for j in P(Dense[L]()):
                    second[i, j](y=Y[i][j], s=S[i])
            for i in P(Dense[n]()):
                third[i](s=S[i], z=Z[i])

        return W.rr4(wl())

    ga, ca = _both(make, a, 2)  # third's tiles have one column: not the same rows
    for k in ("y", "s", "z"):
        np.testing.assert_array_equal(ga[k], ca[k])
