"""Row blocks whose right operands do not fit in LDS whole (rv_matmul_stream), and tasks of 16 or 32
rows that share a workgroup, the last one of it not whole.

Against float64: fp32 sums of K terms in any order are within K * 2^-24 of the sum of magnitudes,
over random signs about sqrt(K) * 2^-24 of the norm: below the row-block tests' 1e-5 at K <= 512."""

import numpy as np
import pytest

import workloads as W
from test_gpu_row_blocks import _proj, _rel, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,K,N,n,layout", [
    (64, 128, 320, 3, "plain"),        # 16 rows of 320 columns at a time
    (16, 256, 160, 9, "plain"),        # four tasks a workgroup, the last with one
    (32, 160, 304, 5, "plain"),        # a slice that 256 threads do not divide
    (16, 320, 144, 4, "transposed"),   # along the other stride
    (32, 128, 320, 3, "transposed"),
    (16, 128, 320, 6, "offset"),       # unaligned: element by element
    (128, 416, 96, 2, "plain"),        # two workgroups a task
    (16, 64, 64, 1, "plain"),          # whole in LDS; one task in a workgroup of four
    (32, 64, 96, 7, "transposed"),
])
def test_streamed_right_operand(gpu, R, K, N, n, layout):
    import torch

    rng = np.random.default_rng(R + K + N)
    a = {"x": rng.standard_normal((n, R, K)), "w": rng.standard_normal((K, N)) / np.sqrt(K), "g": rng.uniform(0.5, 1.5, (1, K)),
         "r": rng.standard_normal((n, R, 1)), "h": np.zeros((n, R, K)), "y": rng.standard_normal((n, R, N))}
    a = {k: v.astype(np.float32) for k, v in a.items()}
    t = {k: torch.from_numpy(v).to(gpu) for k, v in a.items()}
    if layout == "transposed":
        t["w"] = t["w"].t().contiguous().t()
    elif layout == "offset":
        buf = torch.zeros(t["w"].numel() + 1, device=gpu)
        buf[1:].copy_(t["w"].reshape(-1))
        t["w"] = buf[1:].reshape(K, N)
    # What surrounds y stays as it is.
    buf = torch.full((n + 2, R, N), 5.0, device=gpu)
    buf[1:n + 1].copy_(t["y"])
    t["y"] = buf[1:n + 1]
    prog = _proj(t, R, K, N).compile(target="hip_gfx950")
    prog.execute()
    prog.synchronize()
    assert prog.stats.launches == 1
    h = a["x"].astype(np.float64) * a["g"]
    want = a["y"] + (np.maximum(h @ a["w"].astype(np.float64), 0) * a["r"] - a["r"])
    np.testing.assert_allclose(t["h"].cpu().numpy(), h, rtol=1e-6)
    assert _rel(t["y"].cpu().numpy(), want) <= 1e-5
    assert (buf[0] == 5).all() and (buf[n + 1] == 5).all()


@pytest.mark.parametrize("seq,d,mlp,ts", [(192, 128, 512, 64), (160, 128, 512, 32), (80, 128, 512, 16), (96, 128, 256, 32)])
def test_llama_block_streams_its_weights(gpu, seq, d, mlp, ts):
    rng = np.random.default_rng(seq + ts)
    x = rng.standard_normal((seq, d), dtype=np.float32)
    w1 = (rng.standard_normal((d, mlp)) / np.sqrt(d)).astype(np.float32)
    w2 = (rng.standard_normal((mlp, d)) / np.sqrt(mlp)).astype(np.float32)
    out = np.zeros_like(x)
    prog = _run(W.llama_block(x, w1, w2, out, ts, 1e-6))
    assert prog.stats.launches == 1
    assert _rel(out, W.llama_block_ref(x, w1, w2, ts, 1e-6)) <= 1e-5
