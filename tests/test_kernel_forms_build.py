"""The kernel forms that precompile() does not choose, built for gfx950 on the CPU as a run emits
them: GEMM blocks with edges, of 32 rows, with rings of four stages and with K in parts,
row blocks whose right operands are streamed, staged late or shared by tasks, chains, masked rows
and decodes.  Launches are recorded instead of run (hip_stub)."""

import numpy as np
import pytest

import hip_stub
import workloads as W

DT = {"bf16": (W.BF16, np.uint16), "f16": (W.F16, np.float16), "f32": (W.F32, np.float32)}


# dtype, problem, task tile, block, workgroups (more than C has blocks: K in parts), threads
@pytest.mark.parametrize("dt,B,M,N,K,tile,blocks,threads", [
    ("bf16", 1, 80, 144, 2048, (16, 16, 16), 24, 256),      # 64x64, edges, 4 parts
    ("f16", 3, 48, 208, 528, (16, 16, 16), 12, 256),        # edges, K not of whole stages
    ("bf16", 1, 32, 4096, 4096, (32, 128, 64), 128, 256),   # 32x128, ring of four, 4 parts
    ("bf16", 4, 1024, 1024, 1024, (16, 16, 16), 512, 256),  # 64x128
    ("f32", 2, 112, 176, 336, (16, 16, 16), 48, 256),  # edges, 4 parts
    ("f32", 1, 32, 1024, 2048, (32, 64, 32), 64, 256),
])
def test_gemm_forms(dt, B, M, N, K, tile, blocks, threads):
    wdt, ndt = DT[dt]
    a = {"a": np.zeros((B, M, K), ndt), "b": np.zeros((B, K, N), ndt), "c": np.zeros((B, M, N), np.float32)}
    launches, _ = hip_stub.run(W.rr4(W.bgemm(a, *tile, wdt)))
    assert [(x.entry, x.blocks, x.threads) for x in launches] == [("ptowsp_gemm_gemm_tile", blocks, threads)]


@pytest.mark.parametrize("seq,d,mlp,ts", [(192, 128, 512, 64), (8192, 64, 128, 64), (4096, 64, 256, 16), (160, 128, 512, 32)])
def test_llama_block_forms(seq, d, mlp, ts):
    """Whole operands, streamed ones, and tasks that share a workgroup."""
    z = np.zeros
    launches, _ = hip_stub.run(W.llama_block(z((seq, d), np.float32), z((d, mlp), np.float32), z((mlp, d), np.float32),
                                             z((seq, d), np.float32), ts, 1e-6))
    assert [x.entry for x in launches] == ["ptowsp_block_attn_tile"]


def test_late_operands():
    q, k, v = (np.zeros((4, 16, 2048, 64), np.float32) for _ in range(3))
    launches, _ = hip_stub.run(W.rr4(W.tiled_attention(W.attention_arrays(q, k, v, 64), 64)))
    assert [(x.entry, x.blocks) for x in launches] == [("ptowsp_block_attention_tile", 2048)]


def test_phased_softmax_chain():
    launches, _ = hip_stub.run(W.rr4(W.softmax3(W.softmax3_arrays(np.zeros((2, 72, 512), np.float32)))))
    assert len(launches) == 1 and launches[0].entry.startswith("ptowsp_rows_")


@pytest.mark.parametrize("C", [19, 1001, 8128])
def test_masked_rows(C):
    a = {"x": np.zeros((2, 3, 4, C), np.float32), "y": np.zeros((2, 3, 4, C), np.float32)}
    launches, _ = hip_stub.run(W.rr4(W.softmax(a)))
    assert [x.entry for x in launches] == ["ptowsp_row_softmax_tile"]


@pytest.mark.parametrize("G,D,page,kind", [(1, 128, 16, "bf16"), (7, 64, 8, "f16"), (16, 256, 32, "bf16"), (5, 64, 16, "f32")])
def test_decode_forms(G, D, page, kind):
    a = W.paged_decode_arrays([100, 30], 1, G, D, page, f16=kind == "f16", f32=kind == "f32")
    launches, _ = hip_stub.run(W.rr4(W.paged_decode(a, dtype=DT[kind][0])))
    assert [x.entry for x in launches] == ["ptowsp_decode_decode_page"]
