"""The calls whose speed this repository answers for, one dict per case.

Each kind below is one public entry point (or, for the Gated DeltaNet layer,
the three that a layer calls in a row) as a program that serves a language
model calls it: device tensors in, device tensors out, plans and weights kept
between calls. `listed` names twelve of them, `draw` gives more of the same
ranges, and `exact` restates each in float64.

    attention  fp32 attention over a position-major cache (kernels::attention)
    decode     one new token for each of a batch of sequences, ragged lengths
    prefill    norm -> RoPE -> append -> causal attention of a prompt or of a
               chunk of one behind a cached history
    mixer      the whole attention mixer of a prefill, projections included
    matmul     one projection, in the four weight encodings
    gdn        a Gated DeltaNet layer's token mixing: convolution, recurrence,
               gated norm
    kda        Kimi Delta Attention's recurrence from its raw gates
    latent     multi-head latent attention, dense or over selected keys
    select     the sparse-attention indexer's choice of keys
    decoder    one token through the resident decoder (a whole model)
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "math-utils_amd"))
import aigpu  # noqa: E402

BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
TYPES = {"bf16": BF16, "f32": F32}
EPS = 1e-6
THETA = 1e6


# ------------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call: GPT-2 small's attention over a short prompt, fp32
        dict(name="attention-f32-128", kind="attention", count=128, start=0, heads=12, kv_heads=12, dim=64),
        # one user, one token: Qwen3-0.6B's decode attention at 4096 cached positions
        dict(name="decode-1x4096", kind="decode", batch=1, low=4096, high=4096, heads=16, kv_heads=8, dim=128,
             dtype="bf16", window=0),
        # a serving batch: 32 sequences of 1k to 32k cached positions, Qwen3-30B-A3B's heads
        dict(name="decode-32-ragged", kind="decode", batch=32, low=1024, high=32768, heads=32, kv_heads=4, dim=128,
             dtype="bf16", window=0),
        # a long prompt in one call: Qwen3-8B's heads, 8192 tokens
        dict(name="prefill-8192", kind="prefill", count=8192, start=0, heads=32, kv_heads=8, dim=128, dtype="bf16",
             window=0, gate=False),
        # the next turn of a conversation: an odd number of new tokens behind a history
        dict(name="prefill-333-after-1500", kind="prefill", count=333, start=1500, heads=32, kv_heads=8, dim=128,
             dtype="bf16", window=0, gate=False),
        # a whole attention layer of Qwen3-8B over an ordinary prompt of odd length
        dict(name="mixer-1999", kind="mixer", count=1999, start=0, hidden=4096, heads=32, kv_heads=8, dim=128,
             weights="bf16"),
        # an MLP projection of a model stored in 8 bits, a short prompt
        dict(name="matmul-q8-500", kind="matmul", m=500, k=4096, n=12288, weights="q8"),
        # Qwen3-Next's linear attention over a long prompt
        dict(name="gdn-16384", kind="gdn", count=16384, key_heads=16, value_heads=32, dim=128),
        # Kimi-Linear's heads over an ordinary prompt
        dict(name="kda-4096", kind="kda", count=4096, heads=32, dim=128, safe=True),
        # one token of DeepSeek-V3's latent attention at 4096 cached positions
        dict(name="latent-1-after-4096", kind="latent", count=1, start=4096, heads=128, nope=128, vdim=128, rank=512,
             weights="bf16", keep=0),
        # DeepSeek-V3.2's indexer over a chunk of a prompt, deep enough that keys are dropped
        dict(name="select-1024-after-7000", kind="select", count=1024, start=7000, hidden=7168, q_rank=1536, heads=64,
             dim=128, pool=4, top_k=2048, weights="bf16"),
        # one token through all of Qwen3-0.6B
        dict(name="decoder-qwen3-0.6b", kind="decoder", layers=28, hidden=1024, heads=16, kv_heads=8, dim=128,
             mlp=3072, vocab=151936, length=2048, weights="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attention", "decode", "decode", "prefill", "prefill", "mixer", "matmul", "matmul", "gdn",
                       "kda", "latent", "select", "decoder"])
    if kind == "attention":
        heads, kv = rng.choice([(12, 12), (32, 8), (16, 8)])
        return dict(kind=kind, count=_log(rng, 1, 512), start=rng.choice([0, _log(rng, 1, 2000)]), heads=heads,
                    kv_heads=kv, dim=rng.choice([64, 128]))
    if kind == "decode":
        heads, kv = rng.choice([(16, 8), (32, 8), (32, 4)])
        high = _log(rng, 64, 32768)
        batch = _log(rng, 1, 64)
        while batch > 1 and batch * high * kv > 32 * 32768 * 4:
            batch = (batch + 1) // 2
        return dict(kind=kind, batch=batch, low=max(1, high // rng.choice([1, 2, 32])), high=high, heads=heads,
                    kv_heads=kv, dim=rng.choice([128, 128, 64]), dtype=rng.choice(["bf16", "bf16", "f32"]),
                    window=rng.choice([0, 0, 0, 1024]))
    if kind == "prefill":
        heads, kv = rng.choice([(16, 8), (32, 8), (32, 4)])
        return dict(kind=kind, count=_log(rng, 2, 4096), start=rng.choice([0, _log(rng, 1, 4000)]), heads=heads,
                    kv_heads=kv, dim=rng.choice([128, 128, 64]), dtype=rng.choice(["bf16", "bf16", "f32"]),
                    window=rng.choice([0, 0, 0, 1024]), gate=rng.choice([False, False, True]))
    if kind == "mixer":
        hidden, heads, kv = rng.choice([(4096, 32, 8), (1024, 16, 8), (2048, 32, 4)])
        return dict(kind=kind, count=_log(rng, 16, 2500), start=rng.choice([0, _log(rng, 1, 2000)]), hidden=hidden,
                    heads=heads, kv_heads=kv, dim=128, weights=rng.choice(["bf16", "bf16", "q8", "q4", "f32"]))
    if kind == "matmul":
        k, n = rng.choice([(4096, 12288), (4096, 4096), (1024, 3072), (3072, 1024), (4096, 1000), (2048, 8200)])
        return dict(kind=kind, m=_log(rng, 1, 2048), k=k, n=n, weights=rng.choice(["bf16", "q8", "q4", "f32"]))
    if kind == "gdn":
        return dict(kind=kind, count=_log(rng, 1, 8192), key_heads=16, value_heads=rng.choice([16, 32]), dim=128)
    if kind == "kda":
        return dict(kind=kind, count=_log(rng, 1, 4096), heads=rng.choice([8, 16, 32]), dim=rng.choice([128, 128, 64]),
                    safe=rng.choice([True, True, False]))
    if kind == "latent":
        start = _log(rng, 16, 8192)
        return dict(kind=kind, count=rng.choice([1, 1, _log(rng, 2, 128)]), start=start, heads=rng.choice([128, 64, 16]),
                    nope=rng.choice([128, 192]), vdim=rng.choice([128, 256]), rank=512,
                    weights=rng.choice(["bf16", "f32"]), keep=rng.choice([0, 0, 2048]))
    if kind == "select":
        return dict(kind=kind, count=rng.choice([1, _log(rng, 2, 1024)]), start=_log(rng, 2100, 16384), hidden=7168,
                    q_rank=1536, heads=rng.choice([64, 32]), dim=128, pool=rng.choice([4, 1]),
                    top_k=rng.choice([2048, 512]), weights=rng.choice(["bf16", "q8"]))
    return dict(kind=kind, layers=rng.choice([2, 6, 12]), hidden=1024, heads=16, kv_heads=8, dim=128, mlp=3072,
                vocab=rng.choice([151936, 32000]), length=_log(rng, 16, 4096),
                weights=rng.choice(["bf16", "q8", "q4"]))


# ------------------------------------------------------------------- inputs
class _Draws:
    """seeded tensors on the GPU"""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, dtype=F32, scale=1.0):
        x = torch.randn(shape, generator=self.gen, device="cuda")
        if scale != 1.0:
            x *= scale
        return x if dtype == F32 else x.to(dtype)

    def gamma(self, n):
        return torch.rand((n,), generator=self.gen, device="cuda") + 0.5

    def cache(self, *shape):
        """a bf16 cache of normal values, drawn in bf16 (it may be gigabytes)"""
        return torch.randn(shape, generator=self.gen, device="cuda", dtype=BF16)

    def weight(self, n, k, kind):
        """a projection's stored weight, rows of about unit norm, as the entry points take it"""
        if kind in ("f32", "bf16"):
            return {"w": self.normal(n, k, dtype=TYPES[kind], scale=k ** -0.5), "kind": kind, "out": n, "in": k}
        scales = (torch.rand((n, k // 32), generator=self.gen, device="cuda") + 0.5) * k ** -0.5
        if kind == "q8":
            codes = torch.randint(-127, 128, (n, k), generator=self.gen, device="cuda", dtype=torch.int8)
            return {"w": codes, "kind": kind, "out": n, "in": k, "scales": scales / 74.0}
        codes = torch.randint(0, 256, (n, k // 2), generator=self.gen, device="cuda", dtype=torch.uint8)
        return {"w": codes, "kind": kind, "out": n, "in": k, "scales": scales / 4.6}


def _freqs(dim):
    j = np.arange(dim // 2, dtype=np.float32)
    f = np.float32(1.0) / np.power(np.float32(THETA), np.float32(2) * j / np.float32(dim))
    return torch.from_numpy(f.astype(np.float32)).cuda()


def _lengths(c, seed):
    r = np.random.default_rng(seed)
    return r.integers(c["low"], c["high"] + 1, c["batch"]).astype(np.int32)


class _Decoder:
    """the resident decoder and the device weights it borrows"""

    def __init__(self, c, seed):
        self.d = d = _Draws(seed)
        self.keep, self.c = [], c
        H, D, KW = c["hidden"], c["dim"], c["kv_heads"] * c["dim"]
        kind = c["weights"]
        self.layers, self.caches = [], []
        for _ in range(c["layers"]):
            shapes = {"q": (c["heads"] * D, H), "k": (KW, H), "v": (KW, H), "o": (H, c["heads"] * D),
                      "gate": (c["mlp"], H), "up": (c["mlp"], H), "down": (H, c["mlp"])}
            layer = {n: d.weight(*s, kind) for n, s in shapes.items()}
            layer.update(input_norm=d.gamma(H), post_norm=d.gamma(H), q_norm=d.gamma(D), k_norm=d.gamma(D))
            self.layers.append(layer)
            self.caches.append((d.normal(c["length"], KW), d.normal(c["length"], KW)))
        self.head = d.weight(c["vocab"], H, kind)
        self.final_norm = d.gamma(H)
        self.embedding = d.normal(H).cpu().numpy()
        self.position = c["length"]
        self.decoder = None

    def start(self):
        c = self.c

        def w(x):
            return {"ptr": x["w"].data_ptr(), "kind": x["kind"], "in": x["in"], "out": x["out"],
                    "scales_ptr": x["scales"].data_ptr() if "scales" in x else None}

        def host(x):
            return x.cpu().numpy()

        layers = [dict({n: w(l[n]) for n in ("q", "k", "v", "o", "gate", "up", "down")},
                       input_norm=host(l["input_norm"]), post_norm=host(l["post_norm"]), q_norm=host(l["q_norm"]),
                       k_norm=host(l["k_norm"]), window=0) for l in self.layers]
        cfg = dict(hidden=c["hidden"], heads=c["heads"], kv_heads=c["kv_heads"], head_dim=c["dim"],
                   intermediate=c["mlp"], vocab=c["vocab"], capacity=c["length"] + 12000, rotary_dims=c["dim"], eps=EPS,
                   theta=THETA)
        self.decoder = aigpu.DenseDecoder(cfg, layers, w(self.head), host(self.final_norm),
                                          [host(k) for k, _ in self.caches], [host(v) for _, v in self.caches],
                                          c["length"], freqs=host(_freqs(c["dim"])))
        self.caches = None
        return self

    def __del__(self):
        if getattr(self, "decoder", None) is not None:
            self.decoder.close()


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "decoder":
        return dict(c=c, m=_Decoder(c, seed).start())
    d = _Draws(seed)
    s = dict(c=c)
    if kind == "attention":
        T = c["start"] + c["count"]
        s["q"] = d.normal(c["count"], c["heads"], c["dim"])
        s["keys"], s["values"] = d.normal(T, c["kv_heads"], c["dim"]), d.normal(T, c["kv_heads"], c["dim"])
        s["out"] = torch.zeros_like(s["q"])
    elif kind == "decode":
        B, H, KV, D = c["batch"], c["heads"], c["kv_heads"], c["dim"]
        L = _lengths(c, seed)
        s["lengths"], s["max"] = L, int(L.max())
        cap = c["high"] + 1
        t = TYPES[c["dtype"]]
        s["q"], s["k"], s["v"] = d.normal(B, H, D, dtype=t), d.normal(B, KV, D, dtype=t), d.normal(B, KV, D, dtype=t)
        s["kc"], s["vc"] = d.cache(B, KV, cap, D), d.cache(B, KV, cap, D)
        s["gq"], s["gk"], s["freqs"] = d.gamma(D), d.gamma(D), _freqs(D)
        s["positions"] = torch.from_numpy(L).cuda()
        s["out"] = torch.zeros((B, H, D), device="cuda")
    elif kind == "prefill":
        n, H, KV, D = c["count"], c["heads"], c["kv_heads"], c["dim"]
        t = TYPES[c["dtype"]]
        s["q"] = d.normal(n, H, D * (2 if c["gate"] else 1), dtype=t)
        s["k"], s["v"] = d.normal(n, KV, D, dtype=t), d.normal(n, KV, D, dtype=t)
        s["kc"], s["vc"] = d.cache(KV, c["start"] + n, D), d.cache(KV, c["start"] + n, D)
        s["gq"], s["gk"], s["freqs"] = d.gamma(D), d.gamma(D), _freqs(D)
        s["out"] = torch.zeros((n, H, D), device="cuda")
    elif kind == "mixer":
        n, hid, H, KV, D = c["count"], c["hidden"], c["heads"], c["kv_heads"], c["dim"]
        s["x"] = d.normal(n, hid)
        s["w"] = {"q": d.weight(H * D, hid, c["weights"]), "k": d.weight(KV * D, hid, c["weights"]),
                  "v": d.weight(KV * D, hid, c["weights"]), "o": d.weight(hid, H * D, c["weights"])}
        s["kc"], s["vc"] = d.cache(KV, c["start"] + n, D), d.cache(KV, c["start"] + n, D)
        s["gq"], s["gk"], s["freqs"] = d.gamma(D), d.gamma(D), _freqs(D)
        s["out"] = torch.zeros((n, hid), device="cuda")
    elif kind == "matmul":
        s["a"], s["w"] = d.normal(c["m"], c["k"]), d.weight(c["n"], c["k"], c["weights"])
        s["out"] = torch.zeros((c["m"], c["n"]), device="cuda")
    elif kind == "gdn":
        n, HK, HV, D = c["count"], c["key_heads"], c["value_heads"], c["dim"]
        G, CW = HV // HK, 2 * HK * D + HV * D
        s["x"], s["ba"] = d.normal(n, HK, 2 * D + 2 * G * D, dtype=BF16), d.normal(n, HK, 2 * G, dtype=BF16)
        s["kernel"], s["window"] = d.normal(CW, 4, scale=0.5), d.normal(3, CW, dtype=BF16).float()
        s["a_log"], s["dt"], s["gamma"] = d.normal(HV, scale=0.5), d.normal(HV), d.gamma(D)
        s["state"] = d.normal(HV, D, D, scale=0.1)
        s["q"], s["k"] = (torch.zeros((n, HK, D), dtype=BF16, device="cuda") for _ in range(2))
        s["v"], s["z"], s["y"] = (torch.zeros((n, HV, D), dtype=BF16, device="cuda") for _ in range(3))
        s["a"], s["b"] = (torch.zeros((n, HV), device="cuda") for _ in range(2))
        s["core"] = torch.zeros((n, HV, D), device="cuda")
    elif kind == "kda":
        n, H, D = c["count"], c["heads"], c["dim"]
        s["q"], s["k"], s["v"] = (d.normal(n, H, D, dtype=BF16) for _ in range(3))
        s["f"], s["b"] = d.normal(n, H, D), d.normal(n, H)
        s["a_log"], s["dt"] = d.normal(H, scale=0.5), d.normal(H, D)
        s["state"] = d.normal(H, D, D, scale=0.1)
        s["out"] = torch.zeros((n, H, D), device="cuda")
    elif kind == "latent":
        n, H, C = c["count"], c["heads"], c["rank"]
        T = c["start"] + n
        s["q"] = d.normal(n, H, c["nope"])
        s["latent"] = d.normal(T, C)
        s["kv_b"] = d.normal(H * (c["nope"] + c["vdim"]), C, dtype=TYPES[c["weights"]], scale=C ** -0.5)
        s["scale"] = (c["nope"] + 64) ** -0.5
        s["out"] = torch.zeros((n, H, c["vdim"]), device="cuda")
        s["sel"] = None
        if c["keep"]:
            # the indexer's form: each token's chosen keys in order; a token with no more keys than that sees them all
            r = np.random.default_rng(seed)
            starts, counts, keys = [], [], []
            for t in range(n):
                seen = c["start"] + t + 1
                starts.append(sum(map(len, keys)))
                dense = seen <= c["keep"]
                counts.append(-1 if dense else c["keep"])
                keys.append(np.zeros(0, np.int32) if dense else
                            np.sort(r.choice(seen, c["keep"], replace=False)).astype(np.int32))
            keys = np.concatenate(keys + [np.zeros(1, np.int32)])
            s["sel"] = [torch.from_numpy(np.asarray(x, np.int32)).cuda() for x in (starts, counts, keys)]
    elif kind == "select":
        n, D, P = c["count"], c["dim"], c["pool"]
        cap = c["start"] + n + P
        s["h"], s["qr"] = d.normal(n, c["hidden"]), d.normal(n, c["q_rank"])
        s["w"] = {"k": d.weight(D, c["hidden"], c["weights"]), "gate": d.weight(D, c["hidden"], c["weights"]),
                  "q": d.weight(c["heads"] * D, c["q_rank"], c["weights"]),
                  "w": d.weight(c["heads"], c["hidden"], c["weights"])}
        s["norm"], s["bias"], s["ape"] = d.gamma(D), d.normal(D, scale=0.1), d.normal(P, D)
        s["keys"], s["gates"], s["pools"] = d.normal(cap, D), d.normal(cap, D), d.normal(cap // P + 1, D)
        i32 = dict(dtype=torch.int32, device="cuda")
        s["starts"], s["counts"] = torch.zeros(n, **i32), torch.zeros(n, **i32)
        s["chosen"] = torch.zeros((n, c["top_k"] // P * P + P), **i32)
    return s


# ------------------------------------------------------------------- one pass
def run(s):
    c, kind = s["c"], s["c"]["kind"]
    if kind == "attention":
        H, KV, D = c["heads"], c["kv_heads"], c["dim"]
        aigpu.attention_device(s["q"], s["keys"], s["values"], s["out"], c["count"], c["start"], H, KV, D, D, KV * D, D)
        return s["out"]
    if kind == "decode":
        aigpu.decode(s["q"], s["k"], s["v"], s["out"], s["kc"], s["vc"], s["positions"], s["max"], c["heads"],
                     c["kv_heads"], c["dim"], q_norm=s["gq"], k_norm=s["gk"], freqs=s["freqs"], rotary_dims=c["dim"],
                     window=c["window"])
        return s["out"], s["kc"], s["vc"]
    if kind == "prefill":
        aigpu.prefill(s["q"], s["k"], s["v"], s["out"], s["kc"], s["vc"], c["start"], c["heads"], c["kv_heads"],
                      c["dim"], q_stride=s["q"].shape[2], q_norm=s["gq"], k_norm=s["gk"], freqs=s["freqs"],
                      rotary_dims=c["dim"], window=c["window"], output_gate=c["gate"])
        return s["out"], s["kc"], s["vc"]
    if kind == "mixer":
        aigpu.prefill_mixer(s["x"], s["w"], s["out"], s["kc"], s["vc"], c["start"], c["heads"], c["kv_heads"],
                            c["dim"], q_norm=s["gq"], k_norm=s["gk"], freqs=s["freqs"], rotary_dims=c["dim"])
        return s["out"], s["kc"], s["vc"]
    if kind == "matmul":
        return aigpu.matmul(s["a"], s["w"]["w"], s["out"], c["weights"], scales=s["w"].get("scales"))
    if kind == "gdn":
        aigpu.gdn_conv(s["x"], s["kernel"], s["window"], s["q"], s["k"], s["v"], c["key_heads"], c["value_heads"],
                       c["dim"], c["dim"], ba=s["ba"], z=s["z"], a=s["a"], b=s["b"])
        aigpu.gated_delta_rule(s["q"], s["k"], s["v"], s["state"], s["core"], a=s["a"], b=s["b"], a_log=s["a_log"],
                               dt_bias=s["dt"])
        aigpu.gdn_gated_norm(s["core"], s["z"], s["gamma"], s["y"])
        return s["y"], s["core"], s["state"], s["window"], s["q"], s["k"], s["v"]
    if kind == "kda":
        aigpu.kda_rule(s["q"], s["k"], s["v"], None, None, s["state"], s["out"], f=s["f"], b=s["b"], a_log=s["a_log"],
                       dt_bias=s["dt"], safe_gate=c["safe"], lower_bound=-5.0)
        return s["out"], s["state"]
    if kind == "latent":
        sel = s["sel"] or (None, None, None)
        return aigpu.latent_attention(s["q"], s["latent"], s["kv_b"], s["out"], c["start"], s["scale"], *sel)
    if kind == "select":
        aigpu.select_keys(s["h"], s["qr"], s["w"], s["norm"], s["bias"], s["ape"], s["keys"], s["gates"], s["pools"],
                          s["starts"], s["counts"], s["chosen"], c["start"], c["heads"], c["dim"], c["top_k"],
                          c["pool"])
        return s["keys"], s["gates"], s["pools"], s["starts"], s["counts"], s["chosen"]
    m = s["m"]
    logits = m.decoder.decode(m.embedding, m.position)
    m.position += 1
    return logits


# ------------------------------------------------------------------- what a pass needs
_WEIGHT_BYTES = {"f32": 4.0, "bf16": 2.0, "q8": 1.0 + 4 / 32, "q4": 0.5 + 4 / 32}


def _pairs(count, start, window=0):
    """query-key pairs of causal attention"""
    if not window:
        return count * start + count * (count + 1) / 2
    return float(sum(min(start + t + 1, window) for t in range(count)))


def work(case):
    c, kind = case, case["kind"]
    if kind == "attention":
        n, T = c["count"], c["start"] + c["count"]
        return {"bytes": 4.0 * c["dim"] * (2 * n * c["heads"] + 2 * T * c["kv_heads"]),
                "flops": 4.0 * c["dim"] * c["heads"] * _pairs(n, c["start"])}
    if kind == "decode":
        mean = (c["low"] + c["high"]) / 2 + 1
        if c["window"]:
            mean = min(mean, c["window"])
        es = 2 if c["dtype"] == "bf16" else 4
        B, H, KV, D = c["batch"], c["heads"], c["kv_heads"], c["dim"]
        return {"bytes": B * (4.0 * KV * D * mean + es * D * (H + 2 * KV) + 4 * H * D),
                "flops": 4.0 * B * H * D * mean}
    if kind == "prefill":
        n, H, KV, D, T = c["count"], c["heads"], c["kv_heads"], c["dim"], c["start"] + c["count"]
        es = 2 if c["dtype"] == "bf16" else 4
        return {"bytes": float(n * D * (es * (H * (2 if c["gate"] else 1) + 2 * KV) + 4 * H) + 4 * T * KV * D),
                "flops": 4.0 * D * H * _pairs(n, c["start"], c["window"])}
    if kind == "mixer":
        n, hid, H, KV, D = c["count"], c["hidden"], c["heads"], c["kv_heads"], c["dim"]
        params = float(hid * D * (2 * H + 2 * KV))
        return {"bytes": 8.0 * n * hid + 4.0 * (c["start"] + n) * KV * D + params * _WEIGHT_BYTES[c["weights"]],
                "flops": 2.0 * n * params + 4.0 * D * H * _pairs(n, c["start"])}
    if kind == "matmul":
        return {"bytes": 4.0 * c["m"] * (c["k"] + c["n"]) + c["k"] * c["n"] * _WEIGHT_BYTES[c["weights"]],
                "flops": 2.0 * c["m"] * c["k"] * c["n"]}
    if kind == "gdn":
        n, HK, HV, D = c["count"], c["key_heads"], c["value_heads"], c["dim"]
        # the three calls, each tensor that crosses an entry point read or written once; the state both ways
        conv = n * (2 * (2 * HK * D + 2 * HV * D) * 2 + 2 * HV * 6)
        rule = n * (2 * D * (2 * HK + HV) + 8 * HV + 4 * HV * D) + 8 * HV * D * D
        return {"bytes": float(conv + rule + n * HV * D * 8), "flops": n * HV * (7.0 * D * D)}
    if kind == "kda":
        n, H, D = c["count"], c["heads"], c["dim"]
        return {"bytes": float(n * H * (3 * D * 2 + 4 * D + 4 + 4 * D) + 8 * H * D * D), "flops": n * H * (7.0 * D * D)}
    if kind == "latent":
        n, H, C = c["count"], c["heads"], c["rank"]
        keys = _pairs(n, c["start"], c["keep"])
        es = 2 if c["weights"] == "bf16" else 4
        return {"bytes": float(4 * C * min(keys, c["start"] + n) + H * (c["nope"] + c["vdim"]) * C * es
                               + 4 * n * H * (c["nope"] + c["vdim"])),
                "flops": 4.0 * H * C * keys + 2.0 * n * H * C * (c["nope"] + c["vdim"])}
    if kind == "select":
        n, D, P = c["count"], c["dim"], c["pool"]
        params = c["hidden"] * (2 * D + c["heads"]) + c["heads"] * D * c["q_rank"]
        pools = (c["start"] + n) // P
        seen = sum((c["start"] + t + 1) // P for t in range(n))
        return {"bytes": float(4 * n * (c["hidden"] + c["q_rank"]) + params * _WEIGHT_BYTES[c["weights"]]
                               + 4 * D * (pools + 2 * n) + 4 * n * (c["top_k"] + 2)),
                "flops": 2.0 * n * params + 2.0 * c["heads"] * D * seen}
    H, D, KW = c["hidden"], c["dim"], c["kv_heads"] * c["dim"]
    params = c["layers"] * (2 * H * c["heads"] * D + 2 * H * KW + 3 * H * c["mlp"]) + c["vocab"] * H
    return {"bytes": float(params * _WEIGHT_BYTES[c["weights"]] + c["layers"] * 8 * c["length"] * KW + 4 * c["vocab"]),
            "flops": 2.0 * params + 4.0 * c["layers"] * c["heads"] * D * c["length"]}


def tolerance(case):
    """About four times what the calls show against float64, or, where an output is rounded to bf16 or fp16 operands
    are involved, what values rounding the other way amount to"""
    kind = case["kind"]
    if kind in ("attention", "latent"):
        return {"rel": 3e-6, "max": 5e-5}   # 32-bit sums (2e-7 measured) in another order
    if kind == "matmul":
        return {"rel": 1.2e-5, "max": 1e-4}   # activations as two bf16 terms (3e-6 measured)
    if kind == "decode":
        return {"rel": 5e-5, "max": 1e-2}   # two-term operands (3e-6); the new bf16 cache rows
    if kind in ("prefill", "mixer"):
        return {"rel": 1.5e-3, "max": 2e-2}   # fp16 operands (4e-4)
    if kind == "gdn":
        return {"rel": 1e-3, "max": 2e-2}   # bf16 between the calls and at the end; two-term operands (2e-5) inside
    if kind == "kda":
        return {"rel": 6e-6, "max": 1e-4}   # 32-bit products (1.4e-6)
    if kind == "select":
        return {"rel": 6e-6, "max": 2e-4, "differ": 0.005}   # (1e-6); pools near the last kept score may change places
    return {"rel": 5e-6, "max": 1e-4}   # 32-bit sums through 28 layers (8e-7)


# ------------------------------------------------------------------- float64 restatements
def _dequant(w):
    x, kind = w["w"], w["kind"]
    if kind in ("f32", "bf16"):
        return x.double()
    n, k = w["out"], w["in"]
    if kind == "q8":
        codes = x.double()
    else:
        b = x.view(n, k // 32, 16)
        codes = torch.cat([(b & 15), (b >> 4)], dim=2).view(n, k).double() - 8
    return (codes.view(n, k // 32, 32) * w["scales"].double()[:, :, None]).view(n, k)


def _norm(x, gamma, eps=EPS):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * gamma.double()


def _rope(x, positions, freqs):
    """x [n][heads][dim], the angle a float32 product as the models form it"""
    angle = (positions.float()[:, None] * freqs.float()).double()[:, None, :]
    h = freqs.numel()
    a, b = x[..., :h], x[..., h:2 * h]
    cs, sn = angle.cos(), angle.sin()
    return torch.cat([a * cs - b * sn, b * cs + a * sn, x[..., 2 * h:]], -1)


def _attend(q, k, v, start, window=0):
    """q [n][heads][dim] at positions start.. against k, v [kv_heads][T][dim], all float64"""
    n, H, D = q.shape
    G = H // k.shape[0]
    out = torch.empty_like(q)
    key = torch.arange(k.shape[1], device="cuda")
    for r0 in range(0, n, 4096):
        at = start + torch.arange(r0, min(n, r0 + 4096), device="cuda")[:, None]
        hidden = key[None] > at
        if window:
            hidden |= key[None] + window <= at
        for h in range(H):
            sc = (q[r0:r0 + 4096, h] @ k[h // G].T) * D ** -0.5
            out[r0:r0 + 4096, h] = torch.softmax(sc.masked_fill_(hidden, -math.inf), -1) @ v[h // G]
    return out


def _recur(q, k, v, decay, beta, state):
    """the delta rule token by token: q, k, v [n][heads][dim], decay [n][heads][1 or dim]"""
    out = torch.empty_like(v)
    S = state.clone()
    for t in range(q.shape[0]):
        S *= decay[t][:, :, None]
        u = torch.bmm(k[t][:, None], S)[:, 0]
        S.baddbmm_(k[t][:, :, None], (beta[t][:, None] * (v[t] - u))[:, None])
        out[t] = torch.bmm(q[t][:, None], S)[:, 0]
    return out, S


def _unit(x):
    return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "decoder":
        return _exact_decoder(_Decoder(c, seed))
    s = prepare(case, seed)
    if kind == "attention":
        return _attend(s["q"].double(), s["keys"].double().transpose(0, 1), s["values"].double().transpose(0, 1),
                       c["start"])
    if kind == "decode":
        kc, vc = s["kc"].double(), s["vc"].double()
        out = torch.empty((c["batch"], c["heads"], c["dim"]), dtype=F64, device="cuda")
        for b, L in enumerate(s["lengths"].tolist()):
            at = torch.tensor([L], device="cuda")
            q = _rope(_norm(s["q"][b:b + 1].double(), s["gq"]), at, s["freqs"])
            kc[b, :, L] = _rope(_norm(s["k"][b:b + 1].double(), s["gk"]), at, s["freqs"])[0]
            vc[b, :, L] = s["v"][b].double()
            out[b] = _attend(q, kc[b, :, :L + 1], vc[b, :, :L + 1], L, c["window"])[0]
        return out, kc, vc
    if kind == "prefill":
        D = c["dim"]
        at = c["start"] + torch.arange(c["count"], device="cuda")
        kc, vc = s["kc"].double(), s["vc"].double()
        q = _rope(_norm(s["q"][..., :D].double(), s["gq"]), at, s["freqs"])
        kc[:, c["start"]:] = _rope(_norm(s["k"].double(), s["gk"]), at, s["freqs"]).transpose(0, 1)
        vc[:, c["start"]:] = s["v"].double().transpose(0, 1)
        out = _attend(q, kc, vc, c["start"], c["window"])
        return (out * torch.sigmoid(s["q"][..., D:].double()) if c["gate"] else out), kc, vc
    if kind == "mixer":
        n, H, KV, D = c["count"], c["heads"], c["kv_heads"], c["dim"]
        w = {k: _dequant(x) for k, x in s["w"].items()}
        x = s["x"].double()
        at = c["start"] + torch.arange(n, device="cuda")
        kc, vc = s["kc"].double(), s["vc"].double()
        q = _rope(_norm((x @ w["q"].T).view(n, H, D), s["gq"]), at, s["freqs"])
        kc[:, c["start"]:] = _rope(_norm((x @ w["k"].T).view(n, KV, D), s["gk"]), at, s["freqs"]).transpose(0, 1)
        vc[:, c["start"]:] = (x @ w["v"].T).view(n, KV, D).transpose(0, 1)
        return _attend(q, kc, vc, c["start"]).view(n, H * D) @ w["o"].T, kc, vc
    if kind == "matmul":
        return s["a"].double() @ _dequant(s["w"]).T
    if kind == "gdn":
        return _exact_gdn(c, s)
    if kind == "kda":
        H, D = c["heads"], c["dim"]
        x = s["f"].double() + s["dt"].double()
        rate = s["a_log"].double().exp()[:, None]
        g = -5.0 * torch.sigmoid(rate * x) if c["safe"] else -rate * torch.nn.functional.softplus(x)
        return _recur(_unit(s["q"].double()) * D ** -0.5, _unit(s["k"].double()), s["v"].double(), g.exp(),
                      torch.sigmoid(s["b"].double()), s["state"].double())
    if kind == "latent":
        H, Dn, Dv, C = c["heads"], c["nope"], c["vdim"], c["rank"]
        kv = s["kv_b"].double().view(H, Dn + Dv, C)
        lat, q = s["latent"].double(), s["q"].double()
        out = torch.empty((c["count"], H, Dv), dtype=F64, device="cuda")
        for t in range(c["count"]):
            rows = lat[:c["start"] + t + 1]
            if s["sel"] and int(s["sel"][1][t]) >= 0:
                a = int(s["sel"][0][t])
                rows = lat[s["sel"][2][a:a + int(s["sel"][1][t])].long()]
            folded = torch.bmm(q[t][:, None], kv[:, :Dn])[:, 0]
            ctx = torch.softmax(folded @ rows.T * s["scale"], -1) @ rows
            out[t] = torch.bmm(kv[:, Dn:], ctx[:, :, None])[:, :, 0]
        return out
    n, D, P, start = c["count"], c["dim"], c["pool"], c["start"]
    w = {k: _dequant(x) for k, x in s["w"].items()}
    h = s["h"].double()
    keys, gates, pools = s["keys"].double(), s["gates"].double(), s["pools"].double()
    k = h @ w["k"].T
    k = k - k.mean(-1, keepdim=True)
    keys[start:start + n] = k / torch.sqrt((k * k).mean(-1, keepdim=True) + 1e-6) * s["norm"].double() + s["bias"].double()
    gates[start:start + n] = h @ w["gate"].T
    for p in range(start // P, (start + n) // P):
        m = torch.softmax(gates[p * P:p * P + P] + s["ape"].double(), 0)
        pools[p] = (m * keys[p * P:p * P + P]).sum(0)
    return keys, gates, pools, None, None, None


def _exact_gdn(c, s):
    """q, k, v and z leave the convolution in bf16 (the caller's choice), and the recurrence starts from those"""
    n, HK, HV, D = c["count"], c["key_heads"], c["value_heads"], c["dim"]
    G = HV // HK
    x = s["x"]
    qkv = torch.cat([x[..., :D].reshape(n, -1), x[..., D:2 * D].reshape(n, -1),
                     x[..., 2 * D:2 * D + G * D].reshape(n, -1)], 1).double()
    z = x[..., 2 * D + G * D:].reshape(n, HV, D).double()
    rows = torch.cat([s["window"].double(), qkv])
    y = torch.zeros_like(qkv)
    for j in range(4):
        y += rows[j:j + n] * s["kernel"][:, j].double()
    y = torch.nn.functional.silu(y)
    q, k, v = (t.view(n, -1, D) for t in (y[:, :HK * D], y[:, HK * D:2 * HK * D], y[:, 2 * HK * D:]))
    qb, kb, vb = (t.to(BF16).double() for t in (q, k, v))
    ba = s["ba"].double()
    b, a = ba[..., :G].reshape(n, HV), ba[..., G:].reshape(n, HV)
    g = -s["a_log"].double().exp() * torch.nn.functional.softplus(a + s["dt"].double())
    core, state = _recur((_unit(qb) * D ** -0.5).repeat_interleave(G, 1), _unit(kb).repeat_interleave(G, 1), vb,
                         g.exp()[:, :, None], torch.sigmoid(b), s["state"].double())
    out = _norm(core, s["gamma"]) * torch.nn.functional.silu(z)
    return out, core, state, rows[n:], q, k, v


def _exact_decoder(m):
    c = m.c
    H, KV, D = c["heads"], c["kv_heads"], c["dim"]
    at, freqs = torch.tensor([c["length"]], device="cuda"), _freqs(D)
    x = torch.from_numpy(m.embedding).cuda().double()

    def apply(w, a):
        return _dequant(w) @ a

    for l, (keys, values) in zip(m.layers, m.caches):
        a = _norm(x, l["input_norm"])
        q = _rope(_norm(apply(l["q"], a).view(1, H, D), l["q_norm"]), at, freqs)
        k = _rope(_norm(apply(l["k"], a).view(1, KV, D), l["k_norm"]), at, freqs)
        keys = torch.cat([keys.double().view(-1, KV, D), k]).transpose(0, 1)
        values = torch.cat([values.double().view(-1, KV, D), apply(l["v"], a).view(1, KV, D)]).transpose(0, 1)
        x = x + apply(l["o"], _attend(q, keys, values, c["length"]).view(-1))
        a = _norm(x, l["post_norm"])
        x = x + apply(l["down"], torch.nn.functional.silu(apply(l["gate"], a)) * apply(l["up"], a))
    return apply(m.head, _norm(x, m.final_norm)).cpu().numpy()
