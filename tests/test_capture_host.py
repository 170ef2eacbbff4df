"""What a captured run puts into its graph, on the CPU: launches are recorded instead of run
(hip_stub).  A graph may be replayed beside others of the same program and after the program has run
with other sizes."""

import numpy as np
import pytest

import hip_stub
import workloads as W


def _gemm(dt, M, N, K):
    nd = np.float32 if dt == W.F32 else np.uint16
    a = {"a": np.zeros((1, M, K), nd), "b": np.zeros((1, K, N), nd), "c": np.zeros((1, M, N), np.float32)}
    return W.rr4(W.bgemm(a, 16, 16, 32, dt))


@pytest.mark.parametrize("dt", [W.BF16, W.F32])
def test_captured_gemm_holds_no_scratch(dt):
    """A kernel that takes K whole, loaded with the one that splits it: one workgroup per block, no scratch."""
    with hip_stub.program(_gemm(dt, 80, 144, 2048)) as once:
        (eager,) = once()
        (captured,) = once(capture=True)
        (again,) = once()
    assert eager.base[3] and again.base[3] and captured.base[3] is None
    assert captured.entry == eager.entry + "_whole" and captured.threads == eager.threads
    assert captured.blocks < eager.blocks == again.blocks and eager.blocks % captured.blocks == 0
