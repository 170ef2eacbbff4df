"""Paged decode with few units over all the waves: each unit is split into many partials, which
one wave folds after its stream (DecodeCombine::run_many, DecodeSplit::waves_for).

Against float64 attention.  p @ v carries at least 2^-18 relative (p enters in 16-bit parts), and the
fold of n partials adds a rounding per partial, so the decode tests' bound of 1e-5 relative Frobenius
holds whatever the split."""

import numpy as np
import pytest

import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths,hkv,G,D,page,kind", [
    ([2100], 1, 1, 128, 16, "bf16"),          # one row: the lanes past it fold it again
    ([3000, 17], 1, 3, 64, 32, "f16"),        # four rows per pass, three used; a unit of one partial beside it
    ([4000], 2, 4, 128, 16, "bf16"),          # two passes of two rows
    ([1500, 0, 900], 1, 7, 64, 8, "bf16"),    # two passes of four, the last one short; an empty unit
    ([2500], 1, 16, 256, 16, "f16"),          # one row per pass
    ([1800], 2, 20, 128, 32, "bf16"),         # more than 16 rows
    ([1700], 1, 5, 64, 16, "f32"),
    ([1025], 1, 16, 128, 16, "f32"),          # a square score tile, unmasked
    ([90000], 1, 2, 64, 64, "bf16"),          # more than 64 partials: two rounds of weights
    ([16 * 8 + 3] * 3, 1, 4, 128, 16, "bf16"),  # about as many partials as the limit between the two folds
])
def test_many_partials(gpu, lengths, hkv, G, D, page, kind):
    import torch

    a = W.paged_decode_arrays(lengths, hkv, G, D, page, seed=len(lengths) + G, f16=kind == "f16", f32=kind == "f32")
    dt = {"bf16": W.BF16, "f16": W.F16, "f32": W.F32}[kind]

    def dev(x):
        if x.dtype == np.uint16:
            return torch.from_numpy(x.view(np.int16)).to(gpu).view(torch.bfloat16)
        return torch.from_numpy(x).to(gpu)

    t = {k: dev(v) for k, v in a.items() if k != "lengths"}
    masked = not (G == page)  # a square score tile reads the mask by rows
    wl = W.rr4(W.paged_decode(t, masked=masked, dtype=dt))
    prog = wl.compile(target="hip_gfx950")
    assert prog._native.kernel_family("decode_page") == "decode"
    for _ in range(3):  # the counters return to zero; the accumulators start afresh
        t["m"].fill_(float("-inf"))
        t["l"].zero_()
        t["o"].zero_()
        prog.execute()
        prog.synchronize()
    ref = W.paged_decode_ref(a) if masked else _ref_all_tokens(a)
    got = t["out"].cpu().numpy()
    live = np.asarray(lengths) > 0
    assert np.isfinite(got[live]).all()
    assert np.linalg.norm(got[live] - ref[live]) <= 1e-5 * np.linalg.norm(ref[live])
    o, l = t["o"].cpu().numpy()[live], t["l"].cpu().numpy()[live]
    np.testing.assert_array_equal(got[live], o / l)


def _error(gpu, lengths, G, D):
    import torch

    a = W.paged_decode_arrays(lengths, 8, G, D, 16, seed=7)
    t = {k: torch.from_numpy(v.view(np.int16)).to(gpu).view(torch.bfloat16) if v.dtype == np.uint16 else torch.from_numpy(v).to(gpu)
         for k, v in a.items() if k != "lengths"}
    prog = W.rr4(W.paged_decode(t)).compile(target="hip_gfx950")
    prog.execute()
    prog.synchronize()
    ref = W.paged_decode_ref(a)
    return np.linalg.norm(t["out"].cpu().numpy() - ref) / np.linalg.norm(ref)


@pytest.mark.parametrize("G,D", [(1, 128), (4, 128), (7, 64), (12, 256), (20, 128), (48, 64)])
def test_few_units_are_as_exact_as_many(gpu, G, D):
    """bf16 p @ v takes the whole of p: what is left are the roundings of the fp32 sums, about
    sqrt(100) * 2^-24 = 6e-7 for a wave's pages and the fold.  Two bf16 parts of p would leave
    2^-18 / sqrt(3) = 2.2e-6, and the more of it the fewer waves share a unit."""
    assert _error(gpu, [6000, 3111], G, D) <= 1e-6
    if G <= 16:  # beyond, launches over all waves keep two parts
        assert _error(gpu, [700] * 40, G, D) <= 1e-6


def test_many_partials_special_values(gpu):
    """A value that is not finite in one page of one head, the lowest mask over whole runs of pages:
    only that head's value column is not finite (infinity or NaN: p enters in 16-bit parts, and a part may
    be zero), and masked pages weigh nothing."""
    import torch

    a = W.paged_decode_arrays([2100, 1900], 2, 4, 128, seed=5)
    a["mask"][0, 20:60] = np.finfo(np.float32).max
    a["v_cache"][a["page_table"][1, 100], 1, 3, 9] = W.bf16_round(np.float32([np.inf]))[0]
    t = {k: torch.from_numpy(v.view(np.int16)).to(gpu).view(torch.bfloat16) if v.dtype == np.uint16 else torch.from_numpy(v).to(gpu)
         for k, v in a.items() if k != "lengths"}
    prog = W.rr4(W.paged_decode(t)).compile(target="hip_gfx950")
    prog.execute()
    prog.synchronize()
    got = t["out"].cpu().numpy()
    q, k, v = (W.bf16_to_f32(a[n]).astype(np.float64) for n in ("q", "k_cache", "v_cache"))
    for b, pages in enumerate(a["npages"]):
        at = a["page_table"][b, :pages]
        s = np.einsum("hgd,phtd->hgpt", q[b], k[at]) / np.sqrt(128) - a["mask"][b, :pages, 0].astype(np.float64)
        w = np.exp(s - s.max((2, 3), keepdims=True))
        w /= w.sum((2, 3), keepdims=True)
        want = np.einsum("hgpt,phtd->hgd", w, np.where(np.isfinite(v[at]), v[at], 0.0))
        bad = np.zeros(want.shape, bool)
        bad[1, :, 9] = b == 1
        assert not np.isfinite(got[b][bad]).any() and np.isfinite(got[b][~bad]).all()
        assert np.linalg.norm((got[b] - want)[~bad]) <= 1e-5 * np.linalg.norm(want[~bad])


def _ref_all_tokens(a):
    """Without a mask the last page's padding tokens take part."""
    b = dict(a)
    page = a["k_cache"].shape[2]
    b["lengths"] = ((a["lengths"] + page - 1) // page) * page
    return W.paged_decode_ref(b)
