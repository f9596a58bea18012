"""GPU parity of the sparse-attention indexer (aigpu_select_keys) against the
oracle's restatement of selectKeys (LocalModel.hpp:2971-3068: or_index_update,
or_select_keys) over the oracle's matmul_nt for its four projections.

Bars: the new index keys and pooled keys within 1e-5 of max(1, |x|), the
gates within 1e-4 (a projection's 1e-5 of sum |a w|); the scores of every
sparse token within 1e-4 of the magnitude they pass through,
A = sum_h |w_h| headScale (|q_h| . |pool|) dimScale, plus 1e-6 (their q and w
come from projections held to 1e-5 of sum |a w|); the selection key for
key, except for pools whose oracle score is within that bound of the keep-th
best one, which a different summation order may swap. Equal scores take the
lower pools on both sides."""
import numpy as np
import pytest

from gpu_util import dev_f32, host, say
from oracle import oracle as O
from test_gpu_matmul import to_device
from test_gpu_mixer import weight

pytestmark = pytest.mark.gpu


def run(gpu, count, start, kind="f32", hidden=128, q_rank=64, heads=4, dim=64, pool=4, top_k=16, tail=True,
        seed=5, zero_q=False, bias=True):
    import torch
    cap = start + count + pool
    r = np.random.default_rng(seed)
    shapes = {"k": (dim, hidden), "gate": (dim, hidden), "q": (heads * dim, q_rank), "w": (heads, hidden)}
    dev, ref = {}, {}
    for i, (name, (n, k)) in enumerate(shapes.items()):
        stored, scales, _ = weight(n, k, kind, seed + 7 * i, "ix" + name)
        if zero_q and name == "q":
            stored = np.zeros_like(stored)
        dev[name] = {"w": to_device(stored), "kind": kind, "out": n, "in": k,
                     "scales": None if scales is None else dev_f32(scales)}
        ref[name] = (stored, scales)

    def proj(a, name):
        stored, scales = ref[name]
        return O.matmul_nt(a, stored, kind, scales)

    k_norm = r.uniform(0.5, 1.5, dim).astype(np.float32)
    k_bias = (r.standard_normal(dim) * 0.1).astype(np.float32) if bias else None
    ape = r.standard_normal((pool, dim)).astype(np.float32)
    # history [0, start) through the oracle
    keys = np.zeros((cap, dim), np.float32)
    gates = np.zeros((cap, dim), np.float32)
    pools = np.zeros((cap // pool + 1, dim), np.float32)
    if start:
        hh = O.fill_normal((start, hidden), seed, "hist")
        gates[:start] = proj(hh, "gate")
        O.index_update(proj(hh, "k"), k_norm, k_bias, ape, keys, gates, pools, 0, pool)
    h = O.fill_normal((count, hidden), seed, "h")
    qr = O.fill_normal((count, q_rank), seed, "qr")
    d_keys, d_gates, d_pools = dev_f32(keys), dev_f32(gates), dev_f32(pools)
    want_keys, want_gates, want_pools = keys.copy(), gates.copy(), pools.copy()
    want_gates[start:start + count] = proj(h, "gate")
    O.index_update(proj(h, "k"), k_norm, k_bias, ape, want_keys, want_gates, want_pools, start, pool)
    q_o, w_o = proj(qr, "q"), proj(h, "w")
    sel, sc = O.select_keys(q_o, w_o, want_pools, start, heads, dim, pool, top_k, tail)

    stride = top_k // pool * pool + pool
    i32 = dict(dtype=torch.int32, device="cuda")
    ss, sn, sk = torch.zeros(count, **i32), torch.zeros(count, **i32), torch.zeros(count * stride, **i32)
    max_pools = (start + count) // pool
    scores = torch.zeros((count, max(1, max_pools)), dtype=torch.float32, device="cuda")
    say("select keys", dict(count=count, start=start, kind=kind, heads=heads, dim=dim, pool=pool, top_k=top_k,
                            tail=tail, zero_q=zero_q))
    gpu.select_keys(dev_f32(h), dev_f32(qr), dev, dev_f32(k_norm), None if k_bias is None else dev_f32(k_bias),
                    dev_f32(ape), d_keys, d_gates, d_pools, ss, sn, sk, start, heads, dim, top_k, pool, tail=tail,
                    scores=scores)
    gk, gg, gp = host(d_keys), host(d_gates), host(d_pools)
    np.testing.assert_allclose(gg, want_gates, rtol=0, atol=1e-4)
    np.testing.assert_allclose(gk, want_keys, rtol=0, atol=1e-5 * max(1.0, np.abs(want_keys).max()))
    np.testing.assert_allclose(gp, want_pools, rtol=0, atol=1e-5 * max(1.0, np.abs(want_pools).max()))
    st = host(ss).view(np.uint32)
    ct = host(sn).view(np.uint32)
    ks = host(sk).view(np.uint32)
    gsc = host(scores)
    budget = top_k // pool
    for t in range(count):
        pos = start + t
        complete = (pos + 1) // pool
        assert st[t] == t * stride
        if sel[t] is None:
            assert ct[t] == 0xFFFFFFFF, f"token {t} should see every key"
            continue
        got = ks[st[t]:st[t] + ct[t]]
        s = sc[t, :complete]
        mag = (np.abs(w_o[t])[:, None] / np.sqrt(heads) *
               (np.abs(q_o[t].reshape(heads, dim)) @ np.abs(want_pools[:complete]).T) / np.sqrt(dim)).sum(0)
        tol = 1e-4 * mag + 1e-6
        assert (np.abs(gsc[t, :complete] - s) <= tol).all(), f"token {t} scores"
        if list(got) == list(sel[t]):
            continue
        keep = min(budget, complete)
        boundary = np.sort(s)[::-1][keep - 1]
        diff = set(int(x) // pool for x in set(got.tolist()) ^ set(sel[t].tolist()))
        assert all(abs(s[p] - boundary) <= 2 * tol.max() for p in diff), f"token {t}: {sorted(diff)}"
        assert len(got) == len(sel[t]) and list(got) == sorted(got)


@pytest.mark.parametrize("kind", ["f32", "bf16", "q8"])
def test_prefill_from_empty(gpu, kind):
    run(gpu, 120, 0, kind)


@pytest.mark.parametrize("tail", [True, False])
def test_continuation_mid_pool(gpu, tail):
    run(gpu, 45, 37, tail=tail)


def test_decode_step_against_a_long_history(gpu):
    run(gpu, 1, 700, top_k=64, heads=8, dim=128, q_rank=96)


def test_pool_of_one_and_many_heads(gpu):
    run(gpu, 60, 20, pool=1, top_k=8, heads=16, dim=32)


def test_equal_scores_take_the_lower_pools(gpu):
    run(gpu, 30, 40, zero_q=True)


def test_rejects_bad_shapes(gpu):
    import torch
    z = torch.zeros((4, 64), dtype=torch.float32, device="cuda")
    w = {n: {"w": torch.zeros(64 * 64 * 4, dtype=torch.uint8, device="cuda"), "kind": "f32", "out": 64}
         for n in ("k", "gate", "q", "w")}
    i = torch.zeros(64, dtype=torch.int32, device="cuda")
    with pytest.raises(RuntimeError, match="weight shapes"):
        gpu.select_keys(z, z, w, z[0], None, z, z, z, z, i, i, i, 0, 2, 32, 8, 4)


def test_more_than_8192_pools_per_token(gpu):
    """past 256 x 32 pools a token's scores are streamed rather than held in registers"""
    run(gpu, 3, 8300, pool=1, top_k=64, heads=2, dim=32)


@pytest.mark.parametrize("count,heads,dim", [(70, 48, 128), (40, 20, 100), (9, 7, 64), (17, 16, 36), (3, 64, 128),
                                             (33, 16, 256)])
def test_score_tiles(gpu, count, heads, dim):
    """heads and dim short of the matrix-core kernel's tiles of 16 and 32, one to
    four tokens a wave, token groups cut short, both ways of sharing a block of
    64 pools, and a dim past it (index_score_kernel); the last block of pools
    is cut short too"""
    run(gpu, count, 300, heads=heads, dim=dim, pool=2, top_k=16)


@pytest.mark.parametrize("count", [2, 40])
def test_scores_of_values_that_are_not_finite(gpu, count):
    """an infinite or NaN channel in a pool, and an infinite query: every score
    equals the fp32 sums' (relu of a NaN product is 0, infinities carry)"""
    import torch
    heads, dim, hidden, q_rank, pool, start = 4, 64, 64, 32, 1, 200
    r = np.random.default_rng(9)
    w = {n: r.standard_normal(s).astype(np.float32) for n, s in
         (("k", (dim, hidden)), ("gate", (dim, hidden)), ("q", (heads * dim, q_rank)), ("w", (heads, hidden)))}
    dev = {n: {"w": to_device(x), "kind": "f32", "out": x.shape[0], "in": x.shape[1], "scales": None}
           for n, x in w.items()}
    h, qr = (r.standard_normal((count, n)).astype(np.float32) for n in (hidden, q_rank))
    qr[count - 1, 3] = np.inf   # the last token's queries: infinities of both signs
    cap = start + count + 1
    pools = r.standard_normal((cap + 1, dim)).astype(np.float32)
    pools[5, 7], pools[70, 0], pools[131, 63] = np.inf, np.nan, -np.inf
    d_pools = dev_f32(pools)
    keys, gates = (torch.zeros((cap, dim), dtype=torch.float32, device="cuda") for _ in range(2))
    i32 = dict(dtype=torch.int32, device="cuda")
    scores = torch.zeros((count, start + count), dtype=torch.float32, device="cuda")
    say("select keys, not finite", dict(count=count))
    gpu.select_keys(dev_f32(h), dev_f32(qr), dev, dev_f32(np.ones(dim)), None, dev_f32(np.zeros((1, dim))), keys, gates,
                    d_pools, torch.zeros(count, **i32), torch.zeros(count, **i32), torch.zeros(count * 9, **i32), start,
                    heads, dim, 8, pool, scores=scores)
    got, p = host(scores), host(d_pools)
    with np.errstate(all="ignore"):
        q = np.stack([sum(qr[:, [j]] * w["q"][:, j][None] for j in range(q_rank))])[0].reshape(count, heads, dim)
        wt = h @ w["w"].T / np.sqrt(heads)
        for t in range(count):
            n = start + t + 1
            logit = np.zeros((heads, n), np.float32)
            for d in range(dim):   # plain sums: an infinity or a NaN anywhere shows as it does in any order
                logit += q[t][:, [d]] * p[None, :n, d]
            logit /= np.sqrt(dim)
            want = sum(wt[t, i] * np.where(logit[i] > 0, logit[i], 0) for i in range(heads))
            bad = ~np.isfinite(want)
            # the last token's q is infinities of both signs: its products are NaN and its scores 0
            assert bad.any() == (t < count - 1) and (np.isnan(got[t, :n]) == np.isnan(want)).all(), f"token {t}"
            inf = np.isinf(want)
            np.testing.assert_array_equal(got[t, :n][inf], want[inf])
            # finite scores: fp32 sums of dim products per head; those of a row that is not finite are sums of
            # relu(NaN) = relu(-inf) = 0 and so 0 themselves
            tol = 1e-4 * (np.abs(wt[t])[:, None] * (np.abs(q[t]) @ np.abs(p[:n]).T)).sum(0) + 1e-6
            tol = np.where(np.isfinite(tol), tol, 0.0)
            assert (np.abs(got[t, :n] - want)[~bad] <= tol[~bad]).all()


@pytest.mark.parametrize("count", [1, 16])
def test_rejects_an_empty_hidden_row(gpu, count):
    """hidden = 0, whose projections have no terms, is refused whichever way the
    rows of h would go (16 are enough for the matrix cores)"""
    import ctypes as C

    import aigpu
    import torch
    x = torch.zeros(64 * 64, dtype=torch.float32, device="cuda")
    i = torch.zeros(1024, dtype=torch.int32, device="cuda")
    f, n = C.c_void_p(x.data_ptr()), C.c_void_p(i.data_ptr())

    def w(k_in, out):
        return aigpu.AiGpuDenseWeight(codes=f, scales=None, type=aigpu.WEIGHT_TYPES["f32"], inDim=k_in, outDim=out, bias=None)

    args = aigpu.AiGpuSelectKeys(h=f, qResid=f, idxK=w(0, 32), idxGate=w(0, 32), idxQB=w(8, 64), idxWeights=w(0, 2),
                                 kNorm=f, kNormBias=None, ape=f, indexKeys=f, indexGates=f, poolKeys=f, selStart=n,
                                 selCount=n, selKeys=n, scores=None, indexTail=1, count=count, startPos=0, hidden=0,
                                 qRank=8, heads=2, dim=32, topK=8, pool=4, capacity=32,
                                 stream=C.c_void_p(torch.cuda.current_stream().cuda_stream))
    say("select keys, hidden 0", dict(count=count))
    assert gpu.lib().aigpu_select_keys(C.byref(args)) == 0
    assert b"k must be positive" in gpu.lib().aigpu_last_error()


@pytest.mark.parametrize("count", [2, 40])
@pytest.mark.parametrize("spread,shift,w_shift", [(0, 0, 0), (8, 0, 0), (26, 0, 0), (13, 70, 0), (13, 100, 20), (0, -60, 0)])
def test_scores_of_rows_of_wide_range(gpu, count, spread, shift, w_shift):
    """large channels of q meet small channels of the pools: every score within
    the bound of an fp32 chain of its dim + heads terms (2^-24 of the
    magnitudes each), whatever 2^+-spread the channels and 2^shift the rows
    span, and without an overflow that the score itself does not have"""
    import torch
    heads, dim, hidden, q_rank, start = 4, 128, 64, 8, 300
    r = np.random.default_rng(15)
    narrow = lambda *shape: (r.integers(64, 128, shape) * r.choice([-1, 1], shape) / 128).astype(np.float32)
    span = np.exp2(r.integers(-spread, spread + 1, dim)).astype(np.float32)
    # eight-bit mantissas and rows of a with a single 1: the projections are exact
    wq = narrow(heads * dim, q_rank) * np.tile(span, heads)[:, None] * np.float32(2.0) ** shift
    ww = narrow(heads, hidden) * np.float32(2.0) ** w_shift
    w = {"k": narrow(dim, hidden), "gate": narrow(dim, hidden), "q": wq, "w": ww}
    dev = {n: {"w": to_device(x), "kind": "f32", "out": x.shape[0], "in": x.shape[1], "scales": None}
           for n, x in w.items()}
    h, qr = np.zeros((count, hidden), np.float32), np.zeros((count, q_rank), np.float32)
    h[:, 5] = 1.0
    qr[np.arange(count), np.arange(count) % q_rank] = 1.0
    cap = start + count + 1
    pools = (r.standard_normal((cap + 1, dim)) / span * 2.0 ** -abs(shift) * (1 if shift >= 0 else 2.0 ** 120)).astype(np.float32)
    keys, gates = (torch.zeros((cap, dim), dtype=torch.float32, device="cuda") for _ in range(2))
    i32 = dict(dtype=torch.int32, device="cuda")
    scores = torch.zeros((count, start + count), dtype=torch.float32, device="cuda")
    say("select keys, wide rows", dict(count=count, spread=spread, shift=shift, w_shift=w_shift))
    d_pools = dev_f32(pools)
    gpu.select_keys(dev_f32(h), dev_f32(qr), dev, dev_f32(np.ones(dim)), None, dev_f32(np.zeros((1, dim))), keys, gates,
                    d_pools, torch.zeros(count, **i32), torch.zeros(count, **i32), torch.zeros(count * 9, **i32), start,
                    heads, dim, 8, 1, scores=scores)
    got, p = host(scores).astype(np.float64), host(d_pools).astype(np.float64)
    head = ww[:, 5].astype(np.float64) / np.sqrt(heads)
    for t in range(count):
        q = wq[:, t % q_rank].astype(np.float64).reshape(heads, dim)
        dots = q @ p[:start].T / np.sqrt(dim)
        size = np.abs(head) @ (np.abs(q) @ np.abs(p[:start]).T) / np.sqrt(dim)
        err = np.abs(got[t, :start] - head @ np.maximum(dots, 0.0))
        assert (err <= (dim + heads + 4) * 2.0 ** -24 * size).all(), f"token {t}: {np.nanmax(err / size):.3g} of the magnitudes"


@pytest.mark.parametrize("kind", ["f32", "bf16", "q8", "q4"])
def test_projections_of_h_in_one_launch_of_k_slices(gpu, kind):
    """k, the gates and w from 40 rows of h as three weights of one GEMM with K
    slices: segments of 100, 100 and 20 columns in tiles of 128, each with its
    bias, and a key cache that starts mid-way (run checks keys, gates and scores)"""
    import torch
    hidden, count, start, heads, dim = 2304, 40, 30, 20, 100
    r = np.random.default_rng(17)
    h = r.standard_normal((count, hidden)).astype(np.float32)
    qr = r.standard_normal((count, 32)).astype(np.float32)
    dev, dense, bias = {}, {}, {}
    for name, (n, k) in {"k": (dim, hidden), "gate": (dim, hidden), "q": (heads * dim, 32), "w": (heads, hidden)}.items():
        stored, scales, dense[name] = weight(n, k, "f32" if name == "q" else kind, 18, "seg" + name)
        bias[name] = r.standard_normal(n).astype(np.float32)
        dev[name] = {"w": to_device(stored), "kind": "f32" if name == "q" else kind, "out": n, "in": k,
                     "scales": None if scales is None else dev_f32(scales), "bias": dev_f32(bias[name])}
    cap = start + count + 1
    keys, gates, pools = (torch.full((cap + 1, dim), 7.0, dtype=torch.float32, device="cuda") for _ in range(3))
    i32 = dict(dtype=torch.int32, device="cuda")
    scores = torch.zeros((count, start + count), dtype=torch.float32, device="cuda")
    say("select keys, three weights in slices", dict(kind=kind))
    gpu.profile_reset()
    gpu.profile(True)
    gpu.select_keys(dev_f32(h), dev_f32(qr), dev, dev_f32(np.ones(dim)), None, dev_f32(np.zeros((1, dim))), keys, gates,
                    pools, torch.zeros(count, **i32), torch.zeros(count, **i32), torch.zeros(count * 5, **i32), start,
                    heads, dim, 4, 1, scores=scores)
    torch.cuda.synchronize()
    gpu.profile(False)
    assert gpu.profile_read("gemm_reduce_kernel")[1] == 1 and gpu.profile_read("gemm_dma_kernel")[1] == 2
    h64, want = h.astype(np.float64), {}
    for name in ("k", "gate", "w"):
        want[name] = h64 @ dense[name].T.astype(np.float64) + bias[name]
    tol = {n: 1e-5 * (np.abs(h64) @ np.abs(dense[n]).T.astype(np.float64)) + 1e-6 * (1 + np.abs(bias[n])) for n in want}
    got = host(gates)
    assert (np.abs(got[start:start + count] - want["gate"]) <= tol["gate"]).all()
    assert (got[:start] == 7.0).all() and (got[start + count:] == 7.0).all()
    k = want["k"]
    mean, spread = k.mean(1, keepdims=True), np.sqrt(k.var(1, keepdims=True) + 1e-6)
    got = host(keys)
    assert (np.abs(got[start:start + count] - (k - mean) / spread) <= 4 * tol["k"].max() / spread + 1e-5).all()
    q = (qr.astype(np.float64) @ dense["q"].T.astype(np.float64) + bias["q"]).reshape(count, heads, dim)
    p64 = host(pools).astype(np.float64)
    for t in range(count):
        dots = q[t] @ p64[:start + t + 1].T / np.sqrt(dim)
        size = (np.abs(want["w"][t]) + tol["w"][t])[:, None] / np.sqrt(heads) * (np.abs(q[t]) @ np.abs(p64[:start + t + 1]).T) / np.sqrt(dim)
        ref = (want["w"][t][:, None] / np.sqrt(heads) * np.maximum(dots, 0)).sum(0)
        assert (np.abs(host(scores)[t, :start + t + 1] - ref) <= 1e-4 * size.sum(0) + 1e-6).all(), f"token {t}"
