"""Programs made and dropped in turn: the error flag, events and launch scratch of one pass to the
next (ptowsp_program::take_resources), whatever kind of launch left its partials there.

Against float64 with the GEMM tests' 1e-5 relative Frobenius (exact products, fp32 sums of K terms).
A run that ended with an error leaves flag and counters clear for the program after it."""

import gc

import numpy as np
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


@pytest.mark.parametrize("fault", ["pages", "index"])
def test_resources_of_a_failed_run(gpu, fault):
    """A decode that ends with an error (a page count above its maximum, a page index out of range:
    both cut by the kernel's own checks) passes its flag and counters on; the runs after it find
    neither an error nor a count."""
    from pto_wsp import ExecutionError

    a = W.paged_decode_arrays([2100], 1, 1, 128, seed=1)
    if fault == "pages":
        a["npages"][0] = a["page_table"].shape[1] + 1
    else:
        a["page_table"][0, 70] = a["k_cache"].shape[0]
    prog = W.rr4(W.paged_decode(a)).compile(target="hip_gfx950")
    assert prog._native.kernel_family("decode_page") == "decode"
    prog.execute()
    with pytest.raises(ExecutionError, match="declared maximum" if fault == "pages" else "out of range"):
        prog.synchronize()
    del prog
    gc.collect()
    decode_many_partials(gpu, [2100], 1, 1, 128, 16, "bf16")
    gc.collect()
    _gemm(gpu, 16, 512, 1024)


def test_failed_run_then_the_same_program(gpu):
    """The program whose run failed runs again with its tensors put right."""
    from pto_wsp import ExecutionError

    a = W.paged_decode_arrays([2100], 1, 1, 128, seed=1)
    good = a["page_table"].copy()
    a["page_table"][0, 70] = a["k_cache"].shape[0]
    prog = W.rr4(W.paged_decode(a)).compile(target="hip_gfx950")
    prog.execute()
    with pytest.raises(ExecutionError, match="out of range"):
        prog.synchronize()
    a["page_table"][:] = good
    a["m"][:], a["l"][:], a["o"][:] = -np.inf, 0.0, 0.0
    prog.execute()
    prog.synchronize()
    ref = W.paged_decode_ref(a)
    assert np.linalg.norm(a["out"] - ref) <= 1e-5 * np.linalg.norm(ref)
