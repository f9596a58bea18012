"""GPU parity of multi-head latent attention (latent.hip behind
aigpu_latent_attention) against the oracle's restatement of
latentAttentionMixer's attention (LocalModel.hpp:3118-3158).

Bar: fp32 outputs within 1e-5 of max(1, max |out|) (the fold, the scores and
the context are summed in the device's own order)."""
import numpy as np
import pytest

from gpu_util import dev_bf16, dev_f32, dev_u32, host, say
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def run(gpu, count, start, heads, dn, dv, C, seed, bf16_w=False, selection=None):
    import torch
    r = np.random.default_rng(seed)
    q = r.standard_normal((count, heads, dn)).astype(np.float32)
    latent = r.standard_normal((start + count, C)).astype(np.float32)
    wkv = (r.standard_normal((heads * (dn + dv), C)) / np.sqrt(C)).astype(np.float32)
    if bf16_w:
        bits = O.pack_bf16(wkv).reshape(wkv.shape)
        wkv = O.unpack_bf16(bits).reshape(wkv.shape)
        dw = dev_bf16(bits)
    else:
        dw = dev_f32(wkv)
    scale = float(1.0 / np.sqrt(dn + 64))
    out = torch.zeros((count, heads, dv), dtype=torch.float32, device="cuda")
    sel = {}
    if selection is not None:
        st, ct, ks = O.selection_csr(selection, count)
        sel = dict(sel_start=dev_u32(st), sel_count=dev_u32(ct), sel_keys=dev_u32(ks))
    say("latent attention", dict(count=count, start=start, heads=heads, dn=dn, dv=dv, C=C, bf16=bf16_w,
                                 sparse=selection is not None))
    gpu.latent_attention(dev_f32(q), dev_f32(latent), dw, out, start, scale, **sel)
    want = O.latent_attention(q, latent, wkv, start, heads, dn, dv, scale, selection=selection)
    got = host(out)
    err = np.abs(got - want).max()
    assert err <= 1e-5 * max(1.0, np.abs(want).max()), f"max err {err}"


def test_decode_splits_keys(gpu):
    """one token against 300 cached latents: the keys split over workgroups"""
    run(gpu, 1, 300, 20, 64, 48, 512, 1)


def test_prefill_single_split(gpu):
    run(gpu, 300, 5, 16, 128, 128, 256, 2)


def test_small_prefill_bf16_weights(gpu):
    run(gpu, 7, 90, 4, 32, 16, 64, 3, bf16_w=True)


def test_sparse_selection(gpu):
    count, start = 6, 150
    r = np.random.default_rng(4)
    selection = []
    for t in range(count):
        if t % 3 == 1:
            selection.append(None)   # dense
        else:
            n = 40 + 17 * t
            selection.append(np.sort(r.choice(start + t + 1, size=n, replace=False)).tolist())
    run(gpu, count, start, 20, 64, 32, 128, 5, selection=selection)


def test_empty_selection_gives_zero_context(gpu):
    """tokens whose selection is empty (indexTail off, before the first full
    pool) attend to nothing: their output is 0, on one split and when the
    keys of a decode token are split over workgroups"""
    count, start = 5, 40
    selection = [[], [1, 3], [], None, list(range(0, 40, 3))]
    run(gpu, count, start, 20, 64, 32, 128, 6, selection=selection)
    run(gpu, 1, 300, 20, 64, 48, 512, 7, selection=[[]])


def test_rejects_bad_rank(gpu):
    import torch
    q = torch.zeros((1, 2, 8), device="cuda")
    lat = torch.zeros((1, 20), device="cuda")
    w = torch.zeros((2 * 16, 20), device="cuda")
    out = torch.zeros((1, 2, 8), device="cuda")
    with pytest.raises(RuntimeError, match="kvLoraRank"):
        gpu.latent_attention(q, lat, w, out, 0, 1.0)


@pytest.mark.parametrize("count,start,heads,dn,dv,C,bf16", [
    (1, 0, 1, 1, 1, 16, False), (1, 15, 16, 9, 65, 272, True), (1, 16, 17, 64, 128, 512, True),
    (1, 31, 33, 128, 130, 496, False), (1, 32, 128, 192, 256, 512, True), (1, 4200, 40, 32, 24, 512, False),
    (9, 63, 18, 200, 72, 400, True), (2, 64, 16, 256, 256, 512, False)])
def test_tiles(gpu, count, start, heads, dn, dv, C, bf16):
    """16 and 32 heads a workgroup with heads left over, splits of one to several
    blocks of 32 keys whose last holds 1, 16, 17 or all of its keys, ranks past
    one 256-column piece and short of two, v rows past one workgroup's 64"""
    run(gpu, count, start, heads, dn, dv, C, 11, bf16_w=bf16)


def test_kv_b_off_16_byte_boundaries(gpu):
    """kv_b_proj 8 bytes past a 16-byte boundary: its rows are read 16 bytes at a time all the same"""
    import torch
    r = np.random.default_rng(12)
    heads, dn, dv, C, start = 18, 40, 33, 64, 70
    q, latent = (r.standard_normal(s).astype(np.float32) for s in ((1, heads, dn), (start + 1, C)))
    bits = O.pack_bf16((r.standard_normal((heads * (dn + dv), C)) / 8).astype(np.float32)).reshape(-1, C)
    wkv = O.unpack_bf16(bits).reshape(bits.shape)
    store = torch.zeros(bits.size + 4, dtype=torch.bfloat16, device="cuda")
    dw = store[4:].view(bits.shape)
    dw.copy_(dev_bf16(bits))
    assert dw.data_ptr() % 16 == 8
    out = torch.zeros((1, heads, dv), dtype=torch.float32, device="cuda")
    say("latent attention, kv_b off 16 bytes", {})
    gpu.latent_attention(dev_f32(q), dev_f32(latent), dw, out, start, 0.125)
    want = O.latent_attention(q, latent, wkv, start, heads, dn, dv, 0.125)
    assert np.abs(host(out) - want).max() <= 1e-5 * max(1.0, np.abs(want).max())


@pytest.mark.parametrize("start", [39, 63, 300])
def test_scores_below_the_fp32_range_weigh_nothing(gpu, start):
    """finite latents whose scores sum to -infinity: their probability is 0
    wherever they stand (here the oldest 20 or 32 keys, a whole split or block),
    and a token that sees no other is NaN, as exp(-inf - -inf) is"""
    import torch
    heads, dn, dv, C, far = 2, 8, 8, 64, 20 if start == 39 else 32
    r = np.random.default_rng(13)
    q = np.abs(r.standard_normal((1, heads, dn))).astype(np.float32)
    wkv = np.abs(r.standard_normal((heads * (dn + dv), C))).astype(np.float32)
    latent = (r.standard_normal((start + 1, C)) / 8).astype(np.float32)
    want = O.latent_attention(q, latent[far:], wkv, start - far, heads, dn, dv, 0.125)
    latent[:far] = -3e38
    out = torch.zeros((1, heads, dv), dtype=torch.float32, device="cuda")
    say("latent attention, scores of -inf", dict(start=start))
    gpu.latent_attention(dev_f32(q), dev_f32(latent), dev_f32(wkv), out, start, 0.125)
    assert np.abs(host(out) - want).max() <= 1e-5 * max(1.0, np.abs(want).max())
    gpu.latent_attention(dev_f32(q), dev_f32(latent), dev_f32(wkv), out, far - 1, 0.125)
    assert np.isnan(host(out)).all()
