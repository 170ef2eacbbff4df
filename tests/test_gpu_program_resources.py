"""Programs made and dropped in turn: the error flag, events and launch scratch of one pass to the
next (ptowsp_program::take_resources), whatever kind of launch left its partials there.

Against float64 with the GEMM tests' 1e-5 relative Frobenius (exact products, fp32 sums of K terms),
and the error flag of a run that failed against the run after it."""

import gc

import pytest

import workloads as W
from test_gpu_decode_many_parts import test_many_partials as decode_many_partials
from test_gpu_gemm_shapes import _check, _data

pytestmark = pytest.mark.gpu


def _gemm(gpu, M, N, K):
    t = _data(gpu, "bf16", 1, M, N, K)
    c0 = t["c"].clone()
    prog = W.rr4(W.bgemm(t, 16, 16, 32, W.BF16)).compile(target="hip_gfx950")
    for _ in range(2):
        t["c"].copy_(c0)
        prog.execute()
        prog.synchronize()
        _check(t["c"], t, c0)
        assert prog.stats.device_time_ms > 0
    return prog


def test_scratch_passes_between_programs(gpu):
    """Split-K and decode programs of growing and shrinking scratch, one after the other."""
    for M, N, K in ((16, 512, 1024), (80, 144, 2048), (16, 64, 8192), (32, 2048, 2048)):
        prog = _gemm(gpu, M, N, K)
        del prog
        gc.collect()
        decode_many_partials(gpu, [2100], 1, 1, 128, 16, "bf16")
        gc.collect()


def test_live_programs_do_not_share(gpu):
    """Two programs alive at once, on streams of their own."""
    import torch

    del_me = _gemm(gpu, 16, 512, 1024)
    del del_me
    gc.collect()
    runs = []
    for i in range(2):
        t = _data(gpu, "bf16", 1, 16, 512, 4096, seed=i)
        runs.append((W.rr4(W.bgemm(t, 16, 16, 32, W.BF16)).compile(target="hip_gfx950"), t, t["c"].clone(), torch.cuda.Stream()))
    torch.cuda.synchronize()
    for _ in range(8):
        for prog, t, c0, st in runs:
            with torch.cuda.stream(st):
                t["c"].copy_(c0)
                prog.execute()
        for prog, t, c0, st in runs:
            prog.synchronize()
            _check(t["c"], t, c0)
