"""Workloads that a user of this framework has it run, for timing.

Every case is one compiled program over device-resident tensors, called the way a user's
program calls it: ``execute()`` and ``synchronize()``.  The kinds are the framework's
examples and benchmark workloads:

* ``rows``      the quickstart's rmsnorm tile and the row softmax tile over X[B, T, R, C];
* ``softmax3``  the three-phase softmax example (running max, exp + running sum, rescale);
* ``gemm``      the bgemm example's C[b] += A[b] @ B[b] with a P.seq K loop;
* ``attention`` the attention example (fused q k^T / sqrt(d), softmax, v per sequence tile);
* ``llama``     the llama example block (attention, residual, rmsnorm, ReLU MLP, residual);
* ``decode``    paged grouped-query decode with a normalisation launch.
"""

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pto-wsp_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from pto_wsp import (DType, Dense, DenseDyn, DispatchPolicy, In, InOut, Out, P, TaskWindow, Tensor, Tile,  # noqa: E402
                     WindowMode, kernel, pto, workload)

F32, I32 = DType.F32, DType.I32
DTYPES = {"f32": (DType.F32, torch.float32, 4), "f16": (DType.F16, torch.float16, 2), "bf16": (DType.BF16, torch.bfloat16, 2)}


def _rows(name, op, B, T, R, C, out="f32"):
    return {"name": name, "kind": "rows", "op": op, "B": B, "T": T, "R": R, "C": C, "out": out}


def _gemm(name, dtype, B, M, N, K, tm, tn, tk):
    return {"name": name, "kind": "gemm", "dtype": dtype, "B": B, "M": M, "N": N, "K": K, "tm": tm, "tn": tn, "tk": tk}


def _decode(name, dtype, batch, hkv, G, D, page, lmin, lmax):
    return {"name": name, "kind": "decode", "dtype": dtype, "batch": batch, "hkv": hkv, "G": G, "D": D, "page": page,
            "lmin": lmin, "lmax": lmax}


def listed():
    return [
        # The README quickstart: two 16x128 tiles.  What a first program and a small step of a
        # larger one cost: launch and host latency.
        _rows("rmsnorm_quickstart", "rmsnorm", 1, 2, 16, 128),
        # The benchmark's headline: rmsnorm of 2M rows of 128, 1 GiB in and 1 GiB out.
        _rows("rmsnorm_large", "rmsnorm", 16, 8192, 16, 128),
        # The benchmark's softmax: 1M rows of 512.
        _rows("softmax_large", "softmax", 8, 4096, 32, 512),
        # Scores over a ragged number of classes: 32k rows of an odd width.
        _rows("softmax_odd", "softmax", 4, 1024, 8, 1001),
        # The three-phase softmax example at the benchmark's size.
        {"name": "softmax_phases", "kind": "softmax3", "B": 8, "S": 4096, "V": 512},
        # The benchmark's batched bf16 GEMM: the largest compute-bound call.
        _gemm("bgemm_large", "bf16", 64, 2048, 2048, 2048, 128, 128, 64),
        # The bgemm example's own 16x16x16 f16 tiles at an ordinary layer size.
        _gemm("bgemm_example", "f16", 4, 1024, 1024, 1024, 16, 16, 16),
        # A decode step's projection: 32 tokens against a 4096 x 4096 weight.
        _gemm("gemm_tokens", "bf16", 1, 32, 4096, 4096, 32, 128, 64),
        # The attention example over [4, 16, 2048, 64] with 64-token tiles (prefill in local windows).
        {"name": "attention_tiles", "kind": "attention", "B": 4, "H": 16, "S": 2048, "D": 64, "tile": 64},
        # The llama example's block over 8192 tokens: a whole small model step of five launches.
        {"name": "llama_block", "kind": "llama", "S": 8192, "d": 64, "mlp": 128, "tile": 64},
        # The benchmark's paged decode: 64 sequences of up to 8192 tokens.
        _decode("decode_batch", "bf16", 64, 8, 4, 128, 16, 512, 8192),
        # The same model serving two sequences: little work, many CUs to spread it over.
        _decode("decode_small", "bf16", 2, 8, 4, 128, 16, 512, 8192),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rows", "rows", "rows", "gemm", "gemm", "gemm", "decode", "decode", "attention", "llama", "softmax3"])
    if kind == "rows":
        # Widths: multiples of 64 up to 8192, or any width up to 1024 (odd ones among them).
        regular = rng.random() < 0.5
        C = 64 * _log_int(rng, 1, 128) if regular else _log_int(rng, 17, 1024)
        R = rng.choice([1, 2, 4, 8, 16, 32])
        tiles = max(1, _log_int(rng, 1 << 12, (1 << 28) if regular else (1 << 25)) // (R * C))
        B = min(tiles, rng.choice([1, 2, 4, 8, 16]))
        c = _rows("", rng.choice(["rmsnorm", "softmax"]), B, max(1, tiles // B), R, C, rng.choice(["f32", "f32", "bf16", "f16"]))
    elif kind == "softmax3":
        c = {"kind": kind, "B": rng.randint(1, 8), "S": 8 * _log_int(rng, 8, 512), "V": rng.choice([512, 512, 512, 256])}
    elif kind == "gemm":
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        tm, tn, tk = rng.choice([(16, 16, 16), (32, 64, 32), (64, 64, 64), (128, 128, 64), (32, 128, 64)])
        B = _log_int(rng, 1, 16)
        M = tm * max(1, _log_int(rng, 16, 4096) // tm)
        N = tn * max(1, _log_int(rng, 64, 8192) // tn)
        K = tk * max(1, _log_int(rng, 64, 4096) // tk)
        cap = 1.2e11 if dtype == "f32" else 1.0e12
        if (M // tm) % max(1, 64 // tm) or (N // tn) % max(1, 64 // tn):
            cap = 2.0e10  # neither side a multiple of 64: smaller calls
        while 2.0 * B * M * N * K > cap and B > 1:
            B = (B + 1) // 2
        while 2.0 * B * M * N * K > cap and N > tn:
            N = tn * max(1, N // tn // 2)
        while 2.0 * B * M * N * K > cap and M > tm:
            M = tm * max(1, M // tm // 2)
        c = _gemm("", dtype, B, M, N, K, tm, tn, tk)
    elif kind == "attention":
        D, tile = rng.choice([32, 64, 64, 128]), rng.choice([16, 32, 64, 64])
        B, H = rng.choice([1, 2, 4]), _log_int(rng, 1, 32)
        S = tile * max(1, _log_int(rng, 128, 4096) // tile)
        while B * H * S * D > (1 << 23) and H > 1:
            H = (H + 1) // 2
        c = {"kind": kind, "B": B, "H": H, "S": S, "D": D, "tile": tile}
    elif kind == "llama":
        d, tile = rng.choice([32, 64, 64, 128]), rng.choice([16, 32, 64])
        c = {"kind": kind, "S": tile * max(1, _log_int(rng, 128, 16384) // tile), "d": d, "mlp": d * rng.choice([2, 4]), "tile": tile}
    else:
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        page = rng.choice([8, 16, 16, 32, 64])
        G = rng.choice([g for g in (1, 2, 4, 7, 8, 16) if g != page])
        D, hkv = rng.choice([64, 128, 128, 256]), rng.choice([1, 2, 4, 8])
        lmax = _log_int(rng, 64, 16384)
        lmin = max(1, lmax // rng.choice([1, 2, 4, 16]))
        batch = _log_int(rng, 1, 128)
        es = DTYPES[dtype][2]
        while batch > 1 and batch * lmax * hkv * D * es * 2 > 1.0e9:
            batch = (batch + 1) // 2
        c = _decode("", dtype, batch, hkv, G, D, page, lmin, lmax)
    c.pop("name", None)
    return c


# ------------------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device="cuda:0")
    g.manual_seed(seed)
    return g


def _randn(g, shape, dtype=torch.float32, scale=1.0):
    x = torch.randn(shape, generator=g, device="cuda:0", dtype=torch.float32)
    if scale != 1.0:
        x *= scale
    return x.to(dtype)


def _lengths(case, seed):
    return np.random.default_rng(seed).integers(case["lmin"], case["lmax"] + 1, size=case["batch"])


def _inputs(case, seed):
    """The tensors a user's program holds before the call."""
    g, kind = _gen(seed), case["kind"]
    if kind == "rows":
        x = _randn(g, (case["B"], case["T"], case["R"], case["C"]), scale=3.0 if case["op"] == "softmax" else 1.0)
        return {"x": x, "y": torch.empty_like(x, dtype=DTYPES[case["out"]][1])}
    if kind == "softmax3":
        B, S, V = case["B"], case["S"], case["V"]
        x = _randn(g, (B, S, V))
        return {"x": x, "y": torch.zeros_like(x), "rmax": torch.full((B, S // 8, 8, 1), float("-inf"), device=x.device),
                "rsum": torch.zeros((B, S // 8, 8, 1), device=x.device)}
    if kind == "gemm":
        B, M, N, K, dt = case["B"], case["M"], case["N"], case["K"], DTYPES[case["dtype"]][1]
        return {"a": _randn(g, (B, M, K), dt), "b": _randn(g, (B, K, N), dt, 1.0 / math.sqrt(K)), "c": _randn(g, (B, M, N))}
    if kind == "attention":
        B, H, S, D, ts = (case[k] for k in ("B", "H", "S", "D", "tile"))
        q, kt, v = _randn(g, (B, H, S // ts, ts, D)), _randn(g, (B, H, S // ts, D, ts)), _randn(g, (B, H, S // ts, ts, D))
        return {"q": q, "k_t": kt, "v": v, "o": torch.empty_like(q)}
    if kind == "llama":
        S, d, mlp = case["S"], case["d"], case["mlp"]
        return {"x": _randn(g, (S, d)), "w1": _randn(g, (d, mlp), scale=1.0 / math.sqrt(d)),
                "w2": _randn(g, (mlp, d), scale=1.0 / math.sqrt(mlp)), "out": torch.empty((S, d), device="cuda:0")}
    batch, hkv, G, D, page = (case[k] for k in ("batch", "hkv", "G", "D", "page"))
    lengths = _lengths(case, seed)
    npages = (lengths + page - 1) // page
    max_pages = (case["lmax"] + page - 1) // page
    total = int(npages.sum())
    phys = np.random.default_rng(seed + 1).permutation(total).astype(np.int32)
    pt = np.zeros((batch, max_pages), np.int32)
    off = 0
    for b in range(batch):
        pt[b, :npages[b]] = phys[off:off + npages[b]]
        off += npages[b]
    tok = torch.arange(max_pages * page, device="cuda:0").reshape(1, max_pages, 1, page)
    mask = torch.where(tok < torch.from_numpy(lengths).to("cuda:0").reshape(batch, 1, 1, 1), 0.0, 1e30).to(torch.float32)
    dt = DTYPES[case["dtype"]][1]
    acc = (batch, hkv, G)
    return {"q": _randn(g, acc + (D,), dt), "k_cache": _randn(g, (total, hkv, page, D), dt), "v_cache": _randn(g, (total, hkv, page, D), dt),
            "page_table": torch.from_numpy(pt).to("cuda:0"), "npages": torch.from_numpy(npages.astype(np.int32)).to("cuda:0"),
            "mask": mask.contiguous(), "m": torch.full(acc + (1,), float("-inf"), device="cuda:0"),
            "l": torch.zeros(acc + (1,), device="cuda:0"), "o": torch.zeros(acc + (D,), device="cuda:0"),
            "out": torch.zeros(acc + (D,), device="cuda:0")}


# ------------------------------------------------------------------------------ workloads
def _T(x, dtype=F32):
    return Tensor(data=x, shape=tuple(x.shape), dtype=dtype)


def _rows_workload(case, t):
    B, NT, R, C = t["x"].shape
    odt = DTYPES[case["out"]][0]
    X, Y = _T(t["x"]), _T(t["y"], odt)
    if case["op"] == "rmsnorm":
        @kernel
        def rmsnorm_tile(x: In[Tile[R, C, F32]], out: Out[Tile[R, C, odt]]):
            inv = pto.rsqrt(pto.rowmean(pto.mul(x, x)))
            pto.store(out, pto.mul(x, inv))

        body = rmsnorm_tile
    else:
        @kernel
        def softmax_tile(x: In[Tile[R, C, F32]], out: Out[Tile[R, C, odt]]):
            e = pto.exp(pto.sub(x, pto.rowmax(x)))
            pto.store(out, pto.div(e, pto.rowsum(e)))

        body = softmax_tile

    @workload
    def rows_wl():
        for b in P(Dense[B]()):
            for i in P(Dense[NT]()):
                body[b, i](x=X[b][i], out=Y[b][i])

    return rows_wl()


def _softmax3_workload(t):
    B, S, V = t["x"].shape
    tr, tc = 8, 64
    st, vt = S // tr, V // tc
    L, PR = _T(t["x"].reshape(B, st, tr, vt, tc)), _T(t["y"].reshape(B, st, tr, vt, tc))
    RM, RS = _T(t["rmax"]), _T(t["rsum"])

    @kernel
    def update_rowmax(x_tile: In[Tile[tr, tc, F32]], m_acc: InOut[Tile[tr, 1, F32]]):
        pto.store(m_acc, pto.max(m_acc, pto.rowmax(x_tile)))

    @kernel
    def exp_and_accumulate(x_tile: In[Tile[tr, tc, F32]], m_tile: In[Tile[tr, 1, F32]],
                           y_tile: Out[Tile[tr, tc, F32]], l_acc: InOut[Tile[tr, 1, F32]]):
        e = pto.exp(pto.sub(x_tile, m_tile))
        pto.store(l_acc, pto.add(l_acc, pto.rowsum(e)))
        pto.store(y_tile, e)

    @kernel
    def rescale(y_tile: InOut[Tile[tr, tc, F32]], l_tile: In[Tile[tr, 1, F32]]):
        pto.store(y_tile, pto.div(y_tile, l_tile))

    bb, ss, vv = Dense[B](), Dense[st](), Dense[vt]()

    @workload
    def softmax_workload():
        for b in P(bb):
            for s in P(ss):
                for v in P.seq(vv):
                    update_rowmax[b, s, v](x_tile=L[b][s][v], m_acc=RM[b][s])
        for b in P(bb):
            for s in P(ss):
                for v in P.seq(vv):
                    exp_and_accumulate[b, s, v](x_tile=L[b][s][v], m_tile=RM[b][s], y_tile=PR[b][s][v], l_acc=RS[b][s])
        for b in P(bb):
            for s in P(ss):
                for v in P(vv):
                    rescale[b, s, v](y_tile=PR[b][s][v], l_tile=RS[b][s])

    return softmax_workload()


def _gemm_workload(case, t):
    B, M, N, K, tm, tn, tk = (case[k] for k in ("B", "M", "N", "K", "tm", "tn", "tk"))
    dt = DTYPES[case["dtype"]][0]
    A = _T(t["a"].reshape(B, M // tm, tm, K // tk, tk).permute(0, 1, 3, 2, 4), dt)
    Bm = _T(t["b"].reshape(B, K // tk, tk, N // tn, tn).permute(0, 3, 1, 2, 4), dt)
    C = _T(t["c"].reshape(B, M // tm, tm, N // tn, tn).permute(0, 1, 3, 2, 4))

    @kernel
    def gemm_tile(a_tile: In[Tile[tm, tk, dt]], b_tile: In[Tile[tk, tn, dt]], c_tile: InOut[Tile[tm, tn, F32]]):
        pto.store(c_tile, pto.add(c_tile, pto.matmul(a_tile, b_tile)))

    @workload
    def bgemm():
        for b in P(Dense[B]()):
            for m in P(Dense[M // tm]()):
                for n in P(Dense[N // tn]()):
                    for k in P.seq(Dense[K // tk]()):
                        gemm_tile[b, m, n, k](a_tile=A[b][m][k], b_tile=Bm[b][n][k], c_tile=C[b][m][n])

    return bgemm()


def _attention_workload(case, t):
    B, H, S, D, ts = (case[k] for k in ("B", "H", "S", "D", "tile"))
    Q, KT, V, O = _T(t["q"]), _T(t["k_t"]), _T(t["v"]), _T(t["o"])

    @kernel
    def attention_tile(q: In[Tile[ts, D, F32]], k_t: In[Tile[D, ts, F32]], v: In[Tile[ts, D, F32]], out: Out[Tile[ts, D, F32]]):
        s = pto.mul(pto.matmul(q, k_t), pto.constant(1.0 / math.sqrt(D), F32))
        e = pto.exp(pto.sub(s, pto.rowmax(s)))
        pto.store(out, pto.matmul(pto.div(e, pto.rowsum(e)), v))

    @workload
    def attention():
        for b, h in P(Dense[B](), Dense[H]()):
            for s in P(Dense[S // ts]()):
                attention_tile[b, h, s](q=Q[b][h][s], k_t=KT[b][h][s], v=V[b][h][s], out=O[b][h][s])

    return attention()


def _llama_workload(case, t):
    ts, d, mlp, eps = case["tile"], case["d"], case["mlp"], 1e-6
    st = case["S"] // ts
    x = t["x"].reshape(st, ts, d)
    X, KT, W1, W2, O = _T(x), _T(x.permute(0, 2, 1)), _T(t["w1"]), _T(t["w2"]), _T(t["out"].reshape(st, ts, d))
    Xn, Attn, Res1, Mlp = (_T(torch.empty_like(x)) for _ in range(4))

    @kernel
    def rmsnorm_tile(x: In[Tile[ts, d, F32]], out: Out[Tile[ts, d, F32]]):
        inv = pto.rsqrt(pto.add(pto.rowmean(pto.mul(x, x)), pto.constant(eps, F32)))
        pto.store(out, pto.mul(x, inv))

    @kernel
    def attn_tile(q: In[Tile[ts, d, F32]], k_t: In[Tile[d, ts, F32]], v: In[Tile[ts, d, F32]], out: Out[Tile[ts, d, F32]]):
        s = pto.mul(pto.matmul(q, k_t), pto.constant(1.0 / math.sqrt(d), F32))
        e = pto.exp(pto.sub(s, pto.rowmax(s)))
        pto.store(out, pto.matmul(pto.div(e, pto.rowsum(e)), v))

    @kernel
    def add_tile(a: In[Tile[ts, d, F32]], b: In[Tile[ts, d, F32]], out: Out[Tile[ts, d, F32]]):
        pto.store(out, pto.add(a, b))

    @kernel
    def mlp_tile(x: In[Tile[ts, d, F32]], w1: In[Tile[d, mlp, F32]], w2: In[Tile[mlp, d, F32]], out: Out[Tile[ts, d, F32]]):
        h = pto.matmul(x, w1)
        pto.store(out, pto.matmul(pto.max(h, pto.constant(0.0, F32)), w2))

    @workload
    def block():
        for s in P(Dense[st]()):
            attn_tile[s](q=X[s], k_t=KT[s], v=X[s], out=Attn[s])
            add_tile[s](a=X[s], b=Attn[s], out=Res1[s])
            rmsnorm_tile[s](x=Res1[s], out=Xn[s])
            mlp_tile[s](x=Xn[s], w1=W1, w2=W2, out=Mlp[s])
            add_tile[s](a=Res1[s], b=Mlp[s], out=O[s])

    return block()


def _decode_workload(case, t):
    batch, hkv, G, D, page = (case[k] for k in ("batch", "hkv", "G", "D", "page"))
    dt, sc = DTYPES[case["dtype"]][0], 1.0 / math.sqrt(D)
    max_pages = t["page_table"].shape[1]
    Q, KT, V = _T(t["q"], dt), _T(t["k_cache"].permute(0, 1, 3, 2), dt), _T(t["v_cache"], dt)
    PT, NP, MASK = _T(t["page_table"], I32), _T(t["npages"], I32), _T(t["mask"])
    M, L, O, OUT = _T(t["m"]), _T(t["l"]), _T(t["o"]), _T(t["out"])

    @kernel
    def decode_page(q: In[Tile[G, D, dt]], k_t: In[Tile[D, page, dt]], v: In[Tile[page, D, dt]], mask: In[Tile[1, page, F32]],
                    m_acc: InOut[Tile[G, 1, F32]], l_acc: InOut[Tile[G, 1, F32]], o_acc: InOut[Tile[G, D, F32]]):
        s = pto.sub(pto.mul(pto.matmul(q, k_t), pto.constant(sc, F32)), mask)
        m_new = pto.max(m_acc, pto.rowmax(s))
        p = pto.exp(pto.sub(s, m_new))
        alpha = pto.exp(pto.sub(m_acc, m_new))
        pto.store(l_acc, pto.add(pto.mul(l_acc, alpha), pto.rowsum(p)))
        pto.store(o_acc, pto.add(pto.mul(o_acc, alpha), pto.matmul(p, v)))
        pto.store(m_acc, m_new)

    @kernel
    def normalize(o_acc: In[Tile[G, D, F32]], l_acc: In[Tile[G, 1, F32]], out: Out[Tile[G, D, F32]]):
        pto.store(out, pto.div(o_acc, l_acc))

    @workload
    def paged_decode():
        for b in P(Dense[batch]()):
            for g in P(Dense[hkv]()):
                for pg in P.seq(DenseDyn(max_pages, extent=NP[b]), name="pg"):
                    decode_page[b, g, pg](q=Q[b][g], k_t=KT[PT[b][pg]][g], v=V[PT[b][pg]][g], mask=MASK[b][pg],
                                          m_acc=M[b][g], l_acc=L[b][g], o_acc=O[b][g])
        for b in P(Dense[batch]()):
            for g in P(Dense[hkv]()):
                normalize[b, g](o_acc=O[b][g], l_acc=L[b][g], out=OUT[b][g])

    return paged_decode()


def prepare(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "softmax3":
        wl = _softmax3_workload(t)
    elif kind == "rows":
        wl = _rows_workload(case, t)
    else:
        wl = {"gemm": _gemm_workload, "attention": _attention_workload, "llama": _llama_workload, "decode": _decode_workload}[kind](case, t)
    wl = wl.dispatch(DispatchPolicy.round_robin(num_aicpus=4)).task_graph(window=TaskWindow(8192, "tasks", WindowMode.STALL))
    return {"kind": kind, "t": t, "prog": wl.compile(target="hip_gfx950")}


OUTPUTS = {"rows": ("y",), "softmax3": ("y", "rmax", "rsum"), "gemm": ("c",), "attention": ("o",), "llama": ("out",),
           "decode": ("out", "m", "l", "o")}


def run(state):
    t, kind = state["t"], state["kind"]
    # The accumulators of a decode step or a phased softmax start afresh; a GEMM adds to its C.
    if kind == "decode":
        t["m"].fill_(float("-inf"))
        t["l"].zero_()
        t["o"].zero_()
    elif kind == "softmax3":
        t["rmax"].fill_(float("-inf"))
        t["rsum"].zero_()
    state["prog"].execute()
    state["prog"].synchronize()
    return {k: t[k] for k in OUTPUTS[kind]}


# ------------------------------------------------------------------------------ work and accuracy
def work(case):
    kind = case["kind"]
    if kind == "rows":
        n = case["B"] * case["T"] * case["R"] * case["C"]
        return {"bytes": n * (4 + DTYPES[case["out"]][2]), "flops": 4 * n}
    if kind == "softmax3":
        n = case["B"] * case["S"] * case["V"]
        return {"bytes": 8 * n + 16 * case["B"] * case["S"], "flops": 5 * n}
    if kind == "gemm":
        B, M, N, K, es = case["B"], case["M"], case["N"], case["K"], DTYPES[case["dtype"]][2]
        return {"bytes": B * ((M * K + K * N) * es + 8 * M * N), "flops": 2 * B * M * N * K}
    if kind == "attention":
        n = case["B"] * case["H"] * case["S"]
        return {"bytes": 16 * n * case["D"], "flops": 4 * n * case["tile"] * case["D"]}
    if kind == "llama":
        S, d, mlp = case["S"], case["d"], case["mlp"]
        return {"bytes": 8 * S * d + 8 * d * mlp, "flops": 4 * S * d * (case["tile"] + mlp)}
    # Paged decode: K and V of the tokens (the mean length: the lengths come from the seed), q, out and accumulators.
    tok = case["batch"] * (case["lmin"] + case["lmax"]) / 2.0
    rows, D, es = case["batch"] * case["hkv"] * case["G"], case["D"], DTYPES[case["dtype"]][2]
    return {"bytes": tok * case["hkv"] * D * es * 2 + rows * (D * (es + 12) + 16), "flops": 4 * tok * case["hkv"] * case["G"] * D}


def tolerance(case):
    # About four times the error against 64 bits that each kind shows (its sums in another order
    # move by as much): 6e-7 for a row of 1001 added one by one, 7e-8 in short rows, 2e-7 in a
    # GEMM, 3e-7 in attention, 2.3e-6 where 16-bit decode multiplies p as two 16-bit parts.  A
    # 16-bit output may round a few values to the neighbour.
    kind = case["kind"]
    if kind == "rows" and case["out"] != "f32":
        return {"rel": 1e-3, "max": 1e-2}
    if kind == "decode":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 2.5e-6, "max": 5e-5}


def exact(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "rows":
        y = torch.empty_like(t["x"], dtype=torch.float64)
        for b in range(case["B"]):
            x = t["x"][b].double()
            y[b] = x / x.square().mean(-1, keepdim=True).sqrt() if case["op"] == "rmsnorm" else torch.softmax(x, -1)
        return {"y": y}
    if kind == "softmax3":
        return _softmax3_exact(case, t)
    if kind == "gemm":
        c = t["c"].double()
        for b in range(case["B"]):
            c[b] += t["a"][b].double() @ t["b"][b].double()
        return {"c": c}
    if kind == "attention":
        s = t["q"].double() @ t["k_t"].double() / math.sqrt(case["D"])
        return {"o": torch.softmax(s, -1) @ t["v"].double()}
    if kind == "llama":
        x = t["x"].double().reshape(case["S"] // case["tile"], case["tile"], case["d"])
        s = x @ x.transpose(1, 2).contiguous() / math.sqrt(case["d"])
        res = x + torch.softmax(s, -1) @ x
        xn = res / (res.square().mean(-1, keepdim=True) + 1e-6).sqrt()
        out = res + torch.relu(xn @ t["w1"].double()) @ t["w2"].double()
        return {"out": out.reshape(case["S"], case["d"])}
    batch, hkv, G, D, page = (case[k] for k in ("batch", "hkv", "G", "D", "page"))
    shape = (batch, hkv, G)
    r = {"out": torch.empty(shape + (D,), dtype=torch.float64, device="cuda:0"), "o": torch.empty(shape + (D,), dtype=torch.float64, device="cuda:0"),
         "m": torch.empty(shape + (1,), dtype=torch.float64, device="cuda:0"), "l": torch.empty(shape + (1,), dtype=torch.float64, device="cuda:0")}
    scale = float(np.float32(1.0 / math.sqrt(D)))
    for b, n in enumerate(_lengths(case, seed)):
        n = int(n)
        pages = t["page_table"][b, :(n + page - 1) // page].long()
        k = t["k_cache"][pages].double().permute(1, 3, 0, 2).reshape(hkv, D, -1)[:, :, :n].contiguous()
        v = t["v_cache"][pages].double().permute(1, 0, 2, 3).reshape(hkv, -1, D)[:, :n].contiguous()
        s = (t["q"][b].double() @ k) * scale
        r["m"][b] = s.amax(-1, keepdim=True)
        e = (s - r["m"][b]).exp()
        r["l"][b] = e.sum(-1, keepdim=True)
        r["o"][b] = e @ v
        r["out"][b] = r["o"][b] / r["l"][b]
    return r


def _softmax3_exact(case, t):
    """The example's three phases over its [8, 64] tile views, in 64 bits and in program order.
    View v of sequence tile s starts at element V * v of the tile's 8 * V elements and its 8 rows
    are 64 elements apart: 512 elements in all, so with V = 256 neighbouring views overlap."""
    B, S, V = case["B"], case["S"], case["V"]
    tr, tc = 8, 64
    st, vt = S // tr, V // tc
    x = t["x"].double().reshape(B, st, tr * V)
    y = torch.zeros_like(x)
    idx = [vt * tc * v + tc * torch.arange(tr, device=x.device)[:, None] + torch.arange(tc, device=x.device)[None] for v in range(vt)]
    m = torch.stack([x[:, :, i].amax(-1) for i in idx]).amax(0)
    total = torch.zeros_like(m)
    for i in idx:
        e = (x[:, :, i] - m[..., None]).exp()
        total += e.sum(-1)
        y[:, :, i] = e
    for i in idx:
        y[:, :, i] = y[:, :, i] / total[..., None]
    return {"y": y.reshape(B, S, V), "rmax": m[..., None], "rsum": total[..., None]}
