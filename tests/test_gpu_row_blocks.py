"""Row-block chains: kernels with matmuls whose rows are independent, run as waves of 16 rows with
their values in registers, alone or chained with the launches before and after them.

Against float64 (and the oracle for the chains).  fp32 products summed in another order over K
terms differ by at most K * 2^-24 of the sum of magnitudes, the softmax weights by a few roundings:
the tests' 1e-5 relative Frobenius, as for the tile programs, holds at K <= 256."""

import math

import numpy as np
import pytest

import workloads as W
from oracle.runner import run_workload
from pto_wsp import Dense, In, InOut, Out, P, Tile, kernel, pto, workload

pytestmark = pytest.mark.gpu
F32 = W.F32


def _rel(x, y):
    return np.linalg.norm(np.asarray(x, np.float64) - y) / np.linalg.norm(y)


def _run(w):
    prog = w.compile(target="hip_gfx950")
    for _ in range(2):
        prog.execute()
        prog.synchronize()
    return prog


# 1, 2 and 4 waves per workgroup, several workgroups per task, score tiles wider than the rows.
@pytest.mark.parametrize("ts,D", [(32, 32), (64, 64), (64, 128), (96, 64), (128, 128), (256, 64)])
def test_attention_row_blocks(gpu, ts, D):
    rng = np.random.default_rng(ts + D)
    q, k, v = (rng.standard_normal((2, 3, 2 * ts, D), dtype=np.float32) for _ in range(3))
    a = W.attention_arrays(q, k, v, ts)
    w = W.rr4(W.tiled_attention(a, ts))
    prog = _run(w)
    assert prog.stats.launches == 1
    assert "row-block program" in prog._native.precompile(0, row_blocks=True)
    q64, k64, v64 = (x.astype(np.float64).reshape(2, 3, 2, ts, D) for x in (q, k, v))
    s = q64 @ k64.transpose(0, 1, 2, 4, 3) / math.sqrt(D)
    e = np.exp(s - s.max(-1, keepdims=True))
    assert _rel(a["o"], ((e / e.sum(-1, keepdims=True)) @ v64).reshape(q.shape)) <= 1e-5


def _attention_error(B, S, D, ts):
    rng = np.random.default_rng(S + D)
    q, k, v = (rng.standard_normal((B, 4, S, D), dtype=np.float32) for _ in range(3))
    a = W.attention_arrays(q, k, v, ts)
    assert _run(W.rr4(W.tiled_attention(a, ts))).stats.launches == 1
    q, k, v = (x.reshape(B, 4, S // ts, ts, D).astype(np.float64) for x in (q, k, v))
    s = q @ k.swapaxes(-1, -2) / math.sqrt(D)
    e = np.exp(s - s.max(-1, keepdims=True))
    return _rel(a["o"], ((e / e.sum(-1, keepdims=True)) @ v).reshape(B, 4, S, D))


# From 1024 workgroups the right operands take turns in one LDS buffer; 128 rows are two workgroups.
@pytest.mark.parametrize("B,S,D,ts", [(4, 4096, 64, 64), (4, 4032, 128, 64), (4, 4096, 128, 64), (3, 11008, 64, 128)])
def test_attention_operands_in_turn(gpu, B, S, D, ts):
    assert _attention_error(B, S, D, ts) <= 1e-5


# Products below 32^3 from 256 tasks (fewer in the first case: the scalar loop).
@pytest.mark.parametrize("B,S,D,ts", [(5, 192, 64, 16), (4, 256, 64, 16), (4, 272, 32, 16), (1, 1040, 16, 16)])
def test_attention_small_products(gpu, B, S, D, ts):
    assert _attention_error(B, S, D, ts) <= 1e-5


@pytest.mark.parametrize("seq,d,mlp,ts,launches", [(256, 64, 128, 64, 1), (96, 32, 128, 32, 1), (192, 128, 256, 64, 1), (160, 64, 256, 16, 2)])
def test_llama_chain(gpu, seq, d, mlp, ts, launches):
    """The five launches of the llama block: one chain, also where the right operands do not fit in
    LDS whole; the attention of ten tasks with products below 32^3 stays a tile program before the
    chain of the other four.  All intermediate tensors are written."""
    rng = np.random.default_rng(seq)
    x = rng.standard_normal((seq, d), dtype=np.float32)
    w1 = (rng.standard_normal((d, mlp)) / math.sqrt(d)).astype(np.float32)
    w2 = (rng.standard_normal((mlp, d)) / math.sqrt(mlp)).astype(np.float32)
    out = np.zeros_like(x)
    prog = _run(W.llama_block(x, w1, w2, out, ts, 1e-6))
    assert prog.stats.launches == launches
    assert _rel(out, W.llama_block_ref(x, w1, w2, ts, 1e-6)) <= 1e-5
    if seq <= 256 and d <= 64:
        ref = np.zeros_like(x)
        res = run_workload(W.llama_block(x, w1, w2, ref, ts, 1e-6))
        assert prog.stats.total_cycles == res.total_cycles
        assert _rel(out, ref) <= 1e-5


def _proj(arrs, R, K, N, first=None):
    """h = x + b (b: [1, K] scaled by g through a mul), y = relu(h @ w) * r - r with r [R, 1]; h stored."""
    X, Wt, G, RV, H, Y = (W.T(arrs[k]) for k in ("x", "w", "g", "r", "h", "y"))
    n = arrs["x"].shape[0]

    @kernel
    def scale(x: In[Tile[R, K, F32]], g: In[Tile[1, K, F32]], h: Out[Tile[R, K, F32]]):
        pto.store(h, pto.mul(x, g))

    @kernel
    def proj(h: In[Tile[R, K, F32]], w: In[Tile[K, N, F32]], r: In[Tile[R, 1, F32]], y: InOut[Tile[R, N, F32]]):
        z = pto.max(pto.matmul(h, w), pto.constant(0.0, F32))
        pto.store(y, pto.add(y, pto.sub(pto.mul(z, r), r)))

    @workload
    def wl():
        for i in P(Dense[n]()):
            scale[i](x=X[i], g=G, h=H[i])
            proj[i](h=H[i], w=Wt, r=RV[i], y=Y[i])

    return W.rr4(wl())


@pytest.mark.parametrize("layout", ["plain", "transposed", "offset", "alias_right", "alias_rows"])
def test_chain_views(gpu, layout):
    """Broadcast vectors, an InOut output and strided or unaligned views; a chain that would read as
    a right operand, or through another view, what it writes stays separate launches."""
    import torch

    R, K, N, n = 32, 64, 96, 5
    rng = np.random.default_rng(7)
    a = {"x": rng.standard_normal((n, R, K)), "w": rng.standard_normal((K, N)) / 8, "g": rng.uniform(0.5, 1.5, (1, K)),
         "r": rng.standard_normal((n, R, 1)), "h": np.zeros((n, R, K)), "y": rng.standard_normal((n, R, N))}
    a = {k: v.astype(np.float32) for k, v in a.items()}
    t = {k: torch.from_numpy(v).to(gpu) for k, v in a.items()}
    if layout == "transposed":
        t["w"] = t["w"].t().contiguous().t()
        t["x"] = t["x"].permute(0, 2, 1).contiguous().permute(0, 2, 1)
    elif layout == "offset":
        for k in ("x", "h", "w"):
            buf = torch.zeros(t[k].numel() + 1, device=gpu)
            v = buf[1:].reshape(t[k].shape)
            v.copy_(t[k])
            t[k] = v
    elif layout == "alias_right":
        buf = torch.zeros(n * R * K, device=gpu)   # w lies inside h's memory (R * K >= K * N / 2 rows)
        t["h"] = buf.reshape(n, R, K)
        t["w"] = buf[:K * N].reshape(K, N)
        t["w"].copy_(torch.from_numpy(a["w"]).to(gpu))
    elif layout == "alias_rows":
        buf = torch.zeros(n * R * K + K, device=gpu)  # x is h one row further
        t["x"], t["h"] = buf[:n * R * K].reshape(n, R, K), buf[K:].reshape(n, R, K)
        t["x"].copy_(torch.from_numpy(a["x"]).to(gpu))
    prog = _proj(t, R, K, N).compile(target="hip_gfx950")
    prog.execute()
    prog.synchronize()
    assert prog.stats.launches == (2 if layout.startswith("alias") else 1)
    if layout == "alias_rows":
        return  # the first launch itself races on its rows; only the route is checked
    h = a["x"].astype(np.float64) * a["g"]
    w = a["w"].astype(np.float64) if layout != "alias_right" else h.astype(np.float32).reshape(-1)[:K * N].reshape(K, N).astype(np.float64)
    want = a["y"] + (np.maximum(h @ w, 0) * a["r"] - a["r"])
    np.testing.assert_allclose(t["h"].cpu().numpy(), h, rtol=1e-6)
    assert _rel(t["y"].cpu().numpy(), want) <= 1e-5


def test_row_blocks_special_values(gpu):
    """NaN and infinities in q: rows stay apart, as in the oracle."""
    ts = D = 32
    rng = np.random.default_rng(3)
    q, k, v = (rng.standard_normal((1, 1, 2 * ts, D), dtype=np.float32) for _ in range(3))
    q[0, 0, 3, 5] = np.nan
    q[0, 0, 40, 0] = np.inf
    ga, ca = W.attention_arrays(q, k, v, ts), W.attention_arrays(q, k, v, ts)
    _run(W.rr4(W.tiled_attention(ga, ts)))
    run_workload(W.rr4(W.tiled_attention(ca, ts)))
    np.testing.assert_array_equal(np.isnan(ga["o"]), np.isnan(ca["o"]))
    ok = ~np.isnan(ca["o"])
    assert np.isnan(ga["o"][0, 0, 3]).all() and ok[0, 0, 4].all()
    np.testing.assert_allclose(ga["o"][ok], ca["o"][ok], rtol=2e-4, atol=1e-6)
