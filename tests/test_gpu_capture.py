"""Runs captured into graphs: a split-K GEMM takes K whole there, so that its graph holds no scratch
of the program.

Against float64 with the GEMM tests' 1e-5 relative Frobenius, every replay, with eager runs and
synchronisations between them."""

import gc

import pytest

import workloads as W
from test_gpu_gemm_shapes import _check, _data

pytestmark = pytest.mark.gpu


def _captured(gpu, dt, M, N, K, tile, seed):
    import torch

    t = _data(gpu, dt, 1, M, N, K, seed=seed)
    c0 = t["c"].clone()
    wdt = {"bf16": W.BF16, "f32": W.F32}[dt]
    prog = W.rr4(W.bgemm(t, *tile, wdt)).compile(target="hip_gfx950")
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        prog.execute()
        prog.synchronize()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        prog.execute()
    prog.synchronize()
    return prog, graph, t, c0


# A ring of two with edges, a ring of four, f32; C read ahead and not.
@pytest.mark.parametrize("dt,M,N,K,tile", [("bf16", 80, 144, 2048, (16, 16, 16)), ("bf16", 32, 4096, 4096, (32, 128, 64)),
                                           ("f32", 112, 176, 1344, (16, 16, 16))])
def test_captured_split_k(gpu, dt, M, N, K, tile):
    import torch

    prog, graph, t, c0 = _captured(gpu, dt, M, N, K, tile, 1)
    for _ in range(3):
        t["c"].copy_(c0)
        graph.replay()
        torch.cuda.synchronize()
        _check(t["c"], t, c0)
        t["c"].copy_(c0)
        prog.execute()
        prog.synchronize()
        _check(t["c"], t, c0)
    # Replays beside an eager run of another program, and after the program has gone.
    other, g2, t2, c2 = _captured(gpu, dt, M, N, K, tile, 2)
    for _ in range(4):
        t["c"].copy_(c0)
        t2["c"].copy_(c2)
        torch.cuda.synchronize()
        graph.replay()
        other.execute()
        other.synchronize()
        torch.cuda.synchronize()
        _check(t["c"], t, c0)
        _check(t2["c"], t2, c2)
    del prog, other
    gc.collect()
    junk = torch.full((1 << 22,), 7.0, device=gpu)
    for g, x, z in ((graph, t, c0), (g2, t2, c2)):
        x["c"].copy_(z)
        g.replay()
        torch.cuda.synchronize()
        _check(x["c"], x, z)
    assert bool((junk == 7.0).all())
