"""What a captured run puts into its graph, on the CPU: launches are recorded instead of run
(hip_stub).  A graph may be replayed beside others of the same program and after the program has run
with other sizes."""

import numpy as np
import pytest

import hip_stub
import workloads as W
from pto_wsp import Dense, DenseDyn, In, InOut, P, Tile, kernel, pto, sequential, workload


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


def test_captured_decode_keeps_its_scratch():
    """A later run of the same program, whose GEMM has grown, leaves a captured decode's scratch alone."""
    d = W.paged_decode_arrays([100, 30], 1, 1, 64)
    M, N, K = 16, 128, 8192
    A, B = W.T(np.zeros((64, K // 64, M, 64), np.uint16), W.BF16), W.T(np.zeros((K // 64, 64, N), np.uint16), W.BF16)
    C = W.T(np.zeros((64, M, N), np.float32))
    rows = DenseDyn(0)

    @kernel
    def gemm(a: In[Tile[M, 64, W.BF16]], b: In[Tile[64, N, W.BF16]], c: InOut[Tile[M, N, W.F32]]):
        pto.store(c, pto.add(c, pto.matmul(a, b)))

    @workload
    def gemms():
        for m in P(rows, names=["m"]):
            for k in P.seq(Dense[K // 64]()):
                gemm[m, k](a=A[m][k], b=B[k], c=C[m])

    with hip_stub.program(W.rr4(sequential(W.paged_decode(d), gemms()))) as once:
        once.prog.set_axis_sizes({"m": 1})
        once()
        captured = once(capture=True)
        scratch = captured[0].base[7]
        assert captured[0].entry == "ptowsp_decode_decode_page" and scratch and not hip_stub.freed(scratch)
        once.prog.set_axis_sizes({"m": 64})
        grown = once()
        assert grown[0].base[7] == scratch and grown[1].base[3] != scratch
        assert not hip_stub.freed(scratch)
        assert once()[0].base[7] == grown[1].base[3]
