"""Random programs of several launches over few tensors, against the oracle, which runs them one
after the other: what is chained, and what only looks as if it could be (views shifted by a tile,
right operands and broadcast vectors that an earlier launch wrote, tensors written twice).

Every launch keeps its values near 1 (means, halves, products over 1/sqrt(K)).  A product sums K <= 64
terms in another order, within K * 2^-24 = 4e-6 of its magnitude and with random signs within
sqrt(K) * 2^-24 = 5e-7; seven launches stay within 1e-5 relative Frobenius."""

import numpy as np
import pytest

import workloads as W
from oracle.runner import run_workload
from pto_wsp import Dense, In, InOut, Out, P, Tile, kernel, pto, workload

pytestmark = pytest.mark.gpu
F32 = W.F32
R = 32


def _make(seed, arrs):
    """The program of `seed` over arrs: t0..t4 [n + 1, R, C], w [C, C], v [1, C], s0, s1 [n + 1, R, 1]."""
    rng = np.random.default_rng(seed)
    n, C = arrs["t0"].shape[0] - 1, arrs["t0"].shape[2]
    T_, TT = [W.T(arrs[f"t{i}"]) for i in range(5)], [W.T(arrs[f"t{i}"].swapaxes(1, 2)) for i in range(5)]
    Wt, V, S = W.T(arrs["w"]), W.T(arrs["v"]), [W.T(arrs["s0"]), W.T(arrs["s1"])]

    @kernel
    def halve(x: In[Tile[R, C, F32]], y: Out[Tile[R, C, F32]]):
        pto.store(y, pto.add(pto.mul(x, pto.constant(0.5, F32)), pto.constant(0.25, F32)))

    @kernel
    def mean2(x: In[Tile[R, C, F32]], z: In[Tile[R, C, F32]], y: Out[Tile[R, C, F32]]):
        pto.store(y, pto.mul(pto.add(x, z), pto.constant(0.5, F32)))

    @kernel
    def update(x: In[Tile[R, C, F32]], y: InOut[Tile[R, C, F32]]):
        pto.store(y, pto.max(pto.mul(y, pto.constant(0.75, F32)), x))

    @kernel
    def norm(x: In[Tile[R, C, F32]], v: In[Tile[1, C, F32]], y: Out[Tile[R, C, F32]]):
        pto.store(y, pto.mul(pto.mul(x, pto.rsqrt(pto.add(pto.rowmean(pto.mul(x, x)), pto.constant(0.5, F32)))), v))

    @kernel
    def rows(x: In[Tile[R, C, F32]], s: Out[Tile[R, 1, F32]]):
        pto.store(s, pto.rowmax(x))

    @kernel
    def shift(x: In[Tile[R, C, F32]], s: In[Tile[R, 1, F32]], y: Out[Tile[R, C, F32]]):
        pto.store(y, pto.mul(pto.sub(x, s), pto.constant(0.5, F32)))

    @kernel
    def proj(x: In[Tile[R, C, F32]], w: In[Tile[C, C, F32]], y: Out[Tile[R, C, F32]]):
        pto.store(y, pto.max(pto.matmul(x, w), pto.constant(-1.0, F32)))

    @kernel
    def scores(x: In[Tile[R, C, F32]], k_t: In[Tile[C, R, F32]], v: In[Tile[R, C, F32]], y: Out[Tile[R, C, F32]]):
        e = pto.exp(pto.mul(pto.matmul(x, k_t), pto.constant(1.0 / C, F32)))
        pto.store(y, pto.matmul(pto.div(e, pto.rowsum(e)), v))

    steps = []
    for _ in range(int(rng.integers(3, 8))):
        x, z, y = (int(i) for i in rng.integers(0, 5, 3))
        if x == y:
            y = (y + 1) % 5
        # One launch in six reads its neighbour's tile; the plain ones that then race on their own are left out.
        off = int(rng.random() < 1 / 6 and x != y and z != y)
        steps.append((str(rng.choice(["halve", "mean2", "update", "norm", "rows", "shift", "proj", "proj", "scores"])), x, z, y, off,
                      int(rng.integers(0, 2))))

    @workload
    def wl():
        for op, x, z, y, o, s in steps:
            for i in P(Dense[n]()):  # a loop of its own: the launches of one would be promised not to meet
                j = i + 1 if o else i
                X, Z, Y = T_[x][j], T_[z if z != y else x][i], T_[y][i]
                if op == "halve":
                    halve[i](x=X, y=Y)
                elif op == "mean2":
                    mean2[i](x=X, z=Z, y=Y)
                elif op == "update":
                    update[i](x=X, y=Y)
                elif op == "norm":
                    norm[i](x=X, v=V, y=Y)
                elif op == "rows":
                    rows[i](x=X, s=S[s][i])
                elif op == "shift":
                    shift[i](x=X, s=S[s][j], y=Y)
                elif op == "proj":
                    proj[i](x=X, w=Wt, y=Y)
                else:
                    scores[i](x=X, k_t=TT[x][j], v=Z, y=Y)

    return W.rr4(wl())


@pytest.mark.parametrize("seed", range(20))
def test_random_chain(gpu, seed):
    import torch

    n, C = 5, (64, 32, 48, 64)[seed % 4]
    rng = np.random.default_rng(1000 + seed)
    base = {f"t{i}": rng.standard_normal((n + 1, R, C)) for i in range(5)}
    base |= {"w": rng.standard_normal((C, C)) / np.sqrt(C), "v": rng.uniform(0.5, 1.5, (1, C))}
    base |= {f"s{i}": rng.standard_normal((n + 1, R, 1)) for i in range(2)}
    base = {k: v.astype(np.float32) for k, v in base.items()}
    want = {k: v.copy() for k, v in base.items()}
    ref = run_workload(_make(seed, want))

    got = {k: torch.from_numpy(v.copy()).to(gpu) for k, v in base.items()}
    prog = _make(seed, got).compile(target="hip_gfx950")
    prog.execute()
    prog.synchronize()
    assert prog.stats.total_cycles == ref.total_cycles and prog.stats.task_count == ref.task_count
    for k, v in want.items():
        x = got[k].cpu().numpy().astype(np.float64)
        assert np.linalg.norm(x - v) <= 1e-5 * np.linalg.norm(v), (k, prog.stats.launches)


def _make_loops(seed, arrs):
    """Launches over a grid and in-kernel loops of the same extents, over arrs: t0..t3 [n, L, R, C],
    v [1, C], accumulators s0, s1 [n, R, 1]."""
    rng = np.random.default_rng(seed)
    n, L, R, C = arrs["t0"].shape
    T_, S, V = [W.T(arrs[f"t{i}"]) for i in range(4)], [W.T(arrs["s0"]), W.T(arrs["s1"])], W.T(arrs["v"])

    @kernel
    def halve(x: In[Tile[R, C, F32]], y: Out[Tile[R, C, F32]]):
        pto.store(y, pto.add(pto.mul(x, pto.constant(0.5, F32)), pto.constant(0.25, F32)))

    @kernel
    def mean2(x: In[Tile[R, C, F32]], z: In[Tile[R, C, F32]], y: Out[Tile[R, C, F32]]):
        pto.store(y, pto.mul(pto.add(x, z), pto.constant(0.5, F32)))

    @kernel
    def scale(x: In[Tile[R, C, F32]], v: In[Tile[1, C, F32]], y: InOut[Tile[R, C, F32]]):
        pto.store(y, pto.mul(pto.add(x, y), v))

    @kernel
    def shift(x: In[Tile[R, C, F32]], s: In[Tile[R, 1, F32]], y: Out[Tile[R, C, F32]]):
        pto.store(y, pto.mul(pto.sub(x, s), pto.constant(0.5, F32)))

    @kernel
    def fold_max(x: In[Tile[R, C, F32]], s: InOut[Tile[R, 1, F32]]):
        pto.store(s, pto.max(s, pto.rowmax(x)))

    @kernel
    def fold_mean(x: In[Tile[R, C, F32]], s: InOut[Tile[R, 1, F32]]):
        pto.store(s, pto.add(pto.mul(s, pto.constant(0.5, F32)), pto.rowmean(x)))

    steps = []
    for _ in range(int(rng.integers(2, 7))):
        x, z, y = (int(i) for i in rng.integers(0, 4, 3))
        if x == y:
            y = (y + 1) % 4
        op = str(rng.choice(["halve", "mean2", "scale", "shift", "fold_max", "fold_mean"]))
        seq = op.startswith("fold") or rng.random() < 0.5
        steps.append((op, x, z if z != y else x, y, seq, bool(rng.random() < 0.1), int(rng.integers(0, 2))))

    def call(i, j, op, x, z, y, seq, first, s):
        X, Y = T_[x][i][0 if first else j], T_[y][i][j]
        if op == "halve":
            halve[i, j](x=X, y=Y)
        elif op == "mean2":
            mean2[i, j](x=X, z=T_[z][i][j], y=Y)
        elif op == "scale":
            scale[i, j](x=X, v=V, y=Y)
        elif op == "shift":
            shift[i, j](x=X, s=S[s][i], y=Y)
        elif op == "fold_max":
            fold_max[i, j](x=X, s=S[s][i])
        else:
            fold_mean[i, j](x=X, s=S[s][i])

    @workload
    def wl():
        for st in steps:
            for i in P(Dense[n](), names=["outer"]):
                for j in P.seq(Dense[L](), name="step") if st[4] else P(Dense[L](), names=["step"]):
                    call(i, j, *st)

    return W.rr4(wl())


@pytest.mark.parametrize("seed", range(20))
def test_random_loops(gpu, seed):
    """Grid loops and in-kernel loops in turn over the same tiles, with accumulators in place."""
    import torch

    n, L, R, C = 3, (3, 5, 2, 1)[seed % 4], (4, 16, 3)[seed % 3], (32, 48, 19, 64)[seed % 4]
    rng = np.random.default_rng(5000 + seed)
    base = {f"t{i}": rng.standard_normal((n, L, R, C)) for i in range(4)}
    base |= {f"s{i}": rng.standard_normal((n, R, 1)) for i in range(2)}
    base["v"] = rng.uniform(0.3, 0.6, (1, C))
    base = {k: v.astype(np.float32) for k, v in base.items()}
    want = {k: v.copy() for k, v in base.items()}
    ref = run_workload(_make_loops(seed, want))
    got = {k: torch.from_numpy(v.copy()).to(gpu) for k, v in base.items()}
    prog = _make_loops(seed, got).compile(target="hip_gfx950")
    prog.execute()
    prog.synchronize()
    assert prog.stats.total_cycles == ref.total_cycles and prog.stats.task_count == ref.task_count
    for k, v in want.items():
        x = got[k].cpu().numpy().astype(np.float64)
        assert np.linalg.norm(x - v) <= 1e-5 * np.linalg.norm(v), (k, prog.stats.launches)
