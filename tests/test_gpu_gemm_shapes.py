"""GEMM blocks away from whole 256x256 ones: C cut into smaller blocks whatever the task tiles,
last blocks that are not whole, few rows, and K summed in parts by blocks of their own.

Against float64.  The products are exact in fp32 (f32: rounded once) and a sum of K terms in any
order and grouping is within K * 2^-24 of the sum of magnitudes; over random signs that is below
the GEMM tests' 1e-5 relative Frobenius at every K here."""

import numpy as np
import pytest

import workloads as W
from test_zz_no_alloc import AbiProgram, _lib

pytestmark = pytest.mark.gpu


def _data(gpu, dt, B, M, N, K, seed=0):
    import torch

    g = torch.Generator(device=gpu)
    g.manual_seed(seed)
    tdt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[dt]
    a = (torch.rand((B, M, K), generator=g, device=gpu) * 2 - 1).to(tdt)
    b = (torch.rand((B, K, N), generator=g, device=gpu) * 2 - 1).to(tdt)
    return {"a": a, "b": b, "c": torch.randn((B, M, N), generator=g, device=gpu)}


def _check(got, t, c0, plain_k=0):
    a, b = t["a"].double(), t["b"].double()
    want = a[:, :, -plain_k:] @ b[:, -plain_k:].contiguous() if plain_k else c0.double() + a @ b
    assert float((got.double() - want).norm() / want.norm()) <= 1e-5


SHAPES = [
    # dt, B, M, N, K, (tm, tn, tk)
    ("bf16", 1, 16, 512, 1024, (16, 128, 64)),    # 16 rows of a 32-row block, K in parts
    ("bf16", 1, 32, 4096, 4096, (32, 128, 64)),
    ("f16", 3, 48, 208, 528, (16, 16, 16)),       # edges both ways, 16-column stages
    ("bf16", 1, 80, 144, 2048, (16, 16, 16)),     # edges and K in parts
    ("f16", 1, 208, 1200, 528, (16, 16, 16)),
    ("bf16", 2, 144, 16, 512, (16, 16, 32)),      # fewer than 64 columns
    ("f32", 1, 32, 1024, 2048, (32, 64, 32)),
    ("f32", 2, 112, 176, 336, (16, 16, 16)),
    ("f32", 1, 1024, 1024, 256, (64, 64, 64)),
    ("bf16", 1, 1024, 1024, 128, (128, 128, 128)),  # a K step of two stages
    ("bf16", 4, 512, 256, 320, (256, 256, 64)),   # task tiles larger than the blocks
    ("f16", 1, 256, 256, 8192, (256, 256, 64)),   # one tile, K in many parts
]


@pytest.mark.parametrize("dt,B,M,N,K,tile", SHAPES, ids=[f"{s[0]}-{s[1]}x{s[2]}x{s[3]}x{s[4]}" for s in SHAPES])
def test_gemm_shape(gpu, dt, B, M, N, K, tile):
    import torch

    t = _data(gpu, dt, B, M, N, K)
    # The C matrix sits inside a larger buffer: what surrounds it stays as it is.
    buf = torch.full((B, M + 2, N), 5.0, device=gpu)
    c0 = t["c"]
    wdt = {"bf16": W.BF16, "f16": W.F16, "f32": W.F32}[dt]
    prog = None
    for _ in range(3):  # the split's counters return to zero
        buf[:, 1:M + 1].copy_(c0)
        if prog is None:
            c = buf[:, 1:M + 1]
            tm, tn, tk = tile
            # bgemm() reshapes C, which needs a contiguous one: B == 1 views are.
            c = c if B == 1 else c0.clone()
            prog = W.rr4(W.bgemm({"a": t["a"], "b": t["b"], "c": c}, tm, tn, tk, wdt)).compile(target="hip_gfx950")
        elif B > 1:
            c.copy_(c0)
        prog.execute()
        prog.synchronize()
        _check(c, t, c0)
    if B == 1:
        assert bool((buf[:, 0] == 5.0).all()) and bool((buf[:, M + 1] == 5.0).all())


# One, two and three stages: C is read ahead of the last two.
@pytest.mark.parametrize("dt,k", [("bf16", 64), ("bf16", 128), ("f16", 192), ("f32", 32), ("f32", 64), ("f32", 96)])
@pytest.mark.parametrize("B,M,N", [(3, 80, 144), (512, 64, 128), (64, 176, 208)])
def test_gemm_few_stages(gpu, dt, k, B, M, N):
    test_gemm_shape(gpu, dt, B, M, N, k, (16, 16, 32))


@pytest.mark.parametrize("dt,M,N,K", [("bf16", 80, 144, 320), ("f32", 80, 144, 320), ("bf16", 80, 144, 4096)])
def test_gemm_edges_special_values(gpu, dt, M, N, K):
    """Blocks with edges, K whole and in parts: what is not finite in A's last row or B's first column
    (which the rows and columns past the edges read again) stays in its own row and column."""
    import torch

    t = _data(gpu, dt, 1, M, N, K, seed=3)
    t["a"][0, M - 1, 5] = float("inf")
    t["a"][0, 3, K - 1] = float("nan")
    t["b"][0, 7, 0] = float("-inf")
    c = t["c"].clone()
    wdt = {"bf16": W.BF16, "f32": W.F32}[dt]
    prog = W.rr4(W.bgemm({"a": t["a"], "b": t["b"], "c": c}, 16, 16, 16, wdt)).compile(target="hip_gfx950")
    prog.execute()
    prog.synchronize()
    want = t["c"].double() + t["a"].double() @ t["b"].double()
    assert torch.equal(torch.isnan(c), torch.isnan(want)) and torch.equal(torch.isinf(c), torch.isinf(want))
    ok = torch.isfinite(want)
    assert int(ok.sum()) == (M - 2) * (N - 1)
    assert float((c[ok].double() - want[ok]).norm() / want[ok].norm()) <= 1e-5


@pytest.mark.parametrize("M,N,K,tk", [(48, 256, 512, 256), (160, 192, 1024, 1024), (32, 512, 1024, 512)])
def test_gemm_plain_last_step(gpu, M, N, K, tk):
    """store(c, matmul(a, b)) under a K loop: the last step's product, in stages and parts."""
    t = _data(gpu, "bf16", 1, M, N, K, seed=1)
    c = t["c"].clone()
    prog = W.rr4(W.bgemm({"a": t["a"], "b": t["b"], "c": c}, 16, 16, tk, W.BF16, plain=True)).compile(target="hip_gfx950")
    prog.execute()
    prog.synchronize()
    _check(c, t, None, plain_k=tk)


def test_split_k_no_allocation_run(gpu):
    """The no-allocation entry point runs the same split-K kernel in its fixed scratch, bit for bit."""
    import torch

    t = _data(gpu, "bf16", 1, 32, 2048, 4096, seed=2)
    c = t["c"].clone()
    p = AbiProgram(W.rr4(W.bgemm({"a": t["a"], "b": t["b"], "c": c}, 32, 128, 64, W.BF16)), "noalloc_gemm")
    p.run(_lib.ptowsp_hip_launch)
    first = c.clone()
    _check(first, t, t["c"])
    for _ in range(2):
        c.copy_(t["c"])
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info(gpu)[0]
        p.run(_lib.ptowsp_hip_launch_noalloc)
        torch.cuda.synchronize()
        assert torch.cuda.mem_get_info(gpu)[0] == free
        assert torch.equal(c, first)
