"""Row programs at widths that do not split evenly over a lane team: the layout whose last
chunks reach past the row's end (row_layout, row_load_m and its companions).

Every kernel runs on the GPU and on the oracle.  Elementwise results, maxima and stores are
exact; a row sum of n terms in another order is within n * 2^-24 of its terms' magnitudes
(rtol 2^-23 * n covers both sides' orders for the positive terms used here)."""

import numpy as np
import pytest

import workloads as W
from oracle.runner import run_workload
from pto_wsp import Dense, In, InOut, Out, P, Tile, kernel, pto, workload

pytestmark = pytest.mark.gpu
F32 = W.F32
NP_OUT = {W.F32: np.float32, W.F16: np.float16, W.BF16: np.uint16}


def _stats(arrs, R, C):
    """mx = rowmax(x), sm = rowsum(x), y = x * g - m (a [1, C] column vector, a [R, 1] row vector)."""
    X, G, M = W.T(arrs["x"]), W.T(arrs["g"]), W.T(arrs["m"])
    MX, SM, Y = W.T(arrs["mx"]), W.T(arrs["sm"]), W.T(arrs["y"])
    n = arrs["x"].shape[0]

    @kernel
    def stats(x: In[Tile[R, C, F32]], g: In[Tile[1, C, F32]], m: In[Tile[R, 1, F32]], mx: Out[Tile[R, 1, F32]],
              sm: Out[Tile[R, 1, F32]], y: Out[Tile[R, C, F32]]):
        pto.store(mx, pto.rowmax(x))
        pto.store(sm, pto.rowsum(x))
        pto.store(y, pto.sub(pto.mul(x, g), m))

    @workload
    def wl():
        for i in P(Dense[n]()):
            stats[i](x=X[i], g=G, m=M[i], mx=MX[i], sm=SM[i], y=Y[i])

    return W.rr4(wl())


def _run(make, arrs):
    ga, ca = ({k: v.copy(order="K") if v.flags.c_contiguous else v for k, v in arrs.items()} for _ in range(2))
    prog = make(ga).compile(target="hip_gfx950")
    prog.execute()
    prog.synchronize()
    ref = run_workload(make(ca))
    assert prog.stats.total_cycles == ref.total_cycles
    return prog, ga, ca


# Even split (4, 96), one chunk past the end, one element past a chunk, a full team and its
# neighbours, several chunks per lane, and one row per tile (tasks that share a wave).
@pytest.mark.parametrize("R,C", [(4, 5), (8, 19), (3, 24), (2, 63), (2, 65), (8, 96), (5, 100), (1, 255), (4, 257), (1, 1001),
                                 (3, 1025), (2, 2047)])
def test_row_width(gpu, R, C):
    rng = np.random.default_rng(C)
    n = 7
    arrs = {"x": rng.uniform(0.5, 2.0, (n, R, C)).astype(np.float32), "g": rng.uniform(-1, 1, (1, C)).astype(np.float32),
            "m": rng.standard_normal((n, R, 1)).astype(np.float32), "mx": np.zeros((n, R, 1), np.float32),
            "sm": np.zeros((n, R, 1), np.float32), "y": np.zeros((n, R, C), np.float32)}
    prog, ga, ca = _run(lambda a: _stats(a, R, C), arrs)
    assert prog._native.kernel_family("stats") == "row_program"
    np.testing.assert_array_equal(ga["mx"], ca["mx"])
    np.testing.assert_array_equal(ga["y"], ca["y"])
    np.testing.assert_allclose(ga["sm"], ca["sm"], rtol=C * 2.0 ** -23)


def test_row_width_special_values(gpu):
    """NaN, infinities, the lowest finite value and signed zeros: as the oracle's sequential
    maximum (a NaN sticks only as the first element) and sum."""
    R, C = 8, 37
    x = np.random.default_rng(0).uniform(-2, -1, (2, R, C)).astype(np.float32)
    low = np.finfo(np.float32).min
    x[0, 0, 0] = np.nan
    x[0, 1, 20] = np.nan
    x[0, 2, 36] = np.nan
    x[0, 3, :] = -np.inf
    x[0, 4, 35] = np.inf
    x[0, 5, :] = low
    x[0, 6, :] = -0.0
    x[0, 7, 4] = np.nan
    x[0, 7, 0] = -3.0
    arrs = {"x": x, "g": np.ones((1, C), np.float32), "m": np.zeros((2, R, 1), np.float32), "mx": np.zeros((2, R, 1), np.float32),
            "sm": np.zeros((2, R, 1), np.float32), "y": np.zeros((2, R, C), np.float32)}
    _, ga, ca = _run(lambda a: _stats(a, R, C), arrs)
    np.testing.assert_array_equal(ga["mx"], ca["mx"])
    np.testing.assert_array_equal(ga["y"], ca["y"])
    np.testing.assert_allclose(ga["sm"], ca["sm"], rtol=C * 2.0 ** -23)
    assert np.signbit(ga["sm"][0, 6, 0]) == np.signbit(ca["sm"][0, 6, 0])


@pytest.mark.parametrize("dt", [W.F16, W.BF16], ids=["f16", "bf16"])
@pytest.mark.parametrize("C", [19, 101, 1001])
def test_row_width_cast_store(gpu, C, dt):
    x = np.random.default_rng(C).standard_normal((2, 3, 4, C)).astype(np.float32)
    arrs = {"x": x, "out": np.zeros(x.shape, NP_OUT[dt])}
    _, ga, ca = _run(lambda a: W.rr4(W.store_cast(a, dt)), arrs)
    np.testing.assert_array_equal(ga["out"].view(np.uint16), ca["out"].view(np.uint16))


@pytest.mark.parametrize("layout", ["pitched", "offset", "transposed"])
def test_row_width_views(gpu, layout):
    """Rows inside a wider buffer, rows that start one element off alignment, and columns with a
    stride: the elements around the tiles stay as they were."""
    import torch

    R, C, n = 4, 101, 6
    rng = np.random.default_rng(1)
    x = rng.standard_normal((n, R, C)).astype(np.float32)

    def place(buf):
        if layout == "transposed":
            return buf.reshape(n, 120, R + 2).permute(0, 2, 1)[:, 1:R + 1, 5:5 + C]
        return buf.reshape(n, R + 2, 120)[:, 1:R + 1, (5 if layout == "offset" else 8):][:, :, :C]

    xb, yb = (torch.full((n * (R + 2) * 120,), 7.0, device=gpu) for _ in range(2))
    xv, yv = place(xb), place(yb)
    xv.copy_(torch.from_numpy(x))
    w = W.rmsnorm({"x": xv.unsqueeze(0), "y": yv.unsqueeze(0)})
    prog = W.rr4(w).compile(target="hip_gfx950")
    prog.execute()
    prog.synchronize()
    want = W.rmsnorm_ref(x)
    np.testing.assert_allclose(yv.cpu().numpy(), want, rtol=C * 2.0 ** -23)
    yv.fill_(7.0)
    assert bool((yb == 7.0).all())


@pytest.mark.parametrize("C", [19, 100, 257])
def test_row_width_loop_accumulators(gpu, C):
    """A P.seq loop whose accumulators stay in a masked row's registers."""
    R, n, L = 3, 4, 5
    x = np.random.default_rng(C).uniform(0.5, 1.5, (n, L, R, C)).astype(np.float32)
    arrs = {"x": x, "m": np.full((n, R, 1), -np.inf, np.float32), "acc": np.zeros((n, R, C), np.float32)}

    def make(a):
        X, M, A = W.T(a["x"]), W.T(a["m"]), W.T(a["acc"])

        @kernel
        def step(x: In[Tile[R, C, F32]], m: InOut[Tile[R, 1, F32]], acc: InOut[Tile[R, C, F32]]):
            pto.store(m, pto.max(m, pto.rowmax(x)))
            pto.store(acc, pto.add(acc, x))

        @workload
        def wl():
            for i in P(Dense[n]()):
                for j in P.seq(Dense[L]()):
                    step[i, j](x=X[i][j], m=M[i], acc=A[i])

        return W.rr4(wl())

    _, ga, ca = _run(make, arrs)
    np.testing.assert_array_equal(ga["m"], ca["m"])
    np.testing.assert_array_equal(ga["acc"], ca["acc"])
