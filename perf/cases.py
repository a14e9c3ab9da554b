"""Workloads of the attention library, as its users' programs issue them.

Every case goes through a public entry point (``flash_attention_v100`` or
``EnhancedMultiHeadAttention``) on GPU tensors the program already holds:

* ``infer``: one forward call under ``torch.no_grad()``;
* ``decode``: a forward of one (or a few) new queries per sequence over a
  key/value cache, read through a view of the cache's filled part;
* ``train``: forward, then the gradients of q, k, v (and of a learned bias)
  for a given output gradient;
* ``module``: one inference forward of the multi-head attention layer with a
  key padding mask.

The sizes are those of the repository's benchmark configurations, of its
tests, or generic.  ``draw`` gives further cases of the same ranges.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "flash-attn-v100_amd"))

import flash_attention_v100 as fa  # noqa: E402
from flash_attention_v100.modules import EnhancedMultiHeadAttention  # noqa: E402

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def _case(name, kind, B, Sq, Sk, H, Hkv, D, dtype, causal=False, p=0.0, bias="none", qk_std=1.0):
    return {"name": name, "kind": kind, "B": B, "Sq": Sq, "Sk": Sk, "H": H, "Hkv": Hkv, "D": D, "dtype": dtype,
            "causal": causal, "p": p, "bias": bias, "qk_std": qk_std}


def listed():
    return [
        # the smallest call in real use: one short sequence through a small encoder
        _case("tiny_infer", "infer", 1, 128, 128, 8, 8, 64, "fp16"),
        # benchmark configuration 1: inference of a base-size encoder layer
        _case("encoder_infer", "infer", 2, 1024, 1024, 12, 12, 64, "fp16"),
        # benchmark configuration 2: a training step of a base-size causal decoder layer
        _case("small_train", "train", 2, 1024, 1024, 12, 12, 64, "fp16", causal=True),
        # benchmark configuration 3, the headline: a training step at 4 x 4096 tokens, 32 heads of 128
        _case("llama_train", "train", 4, 4096, 4096, 32, 32, 128, "bf16", causal=True),
        # benchmark configuration 4: prefill of one long prompt, outlier-heavy scores
        _case("long_prefill", "infer", 1, 16384, 16384, 16, 16, 128, "bf16", causal=True, qk_std=2.0),
        # serving: one new token for each of 16 sequences over a long cache, grouped-query heads
        _case("decode_gqa", "decode", 16, 1, 8192, 32, 8, 128, "bf16"),
        # a training step of a text decoder's cross-attention over longer encoder states, ragged sizes
        _case("cross_train", "train", 8, 448, 1500, 12, 12, 64, "fp16"),
        # benchmark configuration 5 (fp16): training with attention dropout, a length that is no tile multiple
        _case("dropout_train", "train", 8, 1000, 1000, 16, 16, 64, "fp16", causal=True, p=0.1),
        # benchmark configuration 5 (fp32): the same in full precision
        _case("fp32_train", "train", 8, 1000, 1000, 16, 16, 64, "fp32", causal=True, p=0.1),
        # a training step with a learned relative-position bias shared by the batch, and its gradient
        _case("bias_train", "train", 2, 2048, 2048, 16, 16, 64, "bf16", causal=True, bias="heads"),
        # a training step of a vision encoder: head dim 80, 32 x 32 patches and a class token
        _case("vision_train", "train", 4, 1025, 1025, 16, 16, 80, "bf16"),
        # inference of the attention layer on padded batches (width 768, 12 heads)
        _case("module_padded", "module", 8, 512, 512, 12, 12, 64, "fp16", bias="padding"),
    ]


def _pairs(case):
    """Visible (query, key) pairs of one head."""
    Sq, Sk = case["Sq"], case["Sk"]
    if not case["causal"]:
        return Sq * Sk
    n = min(Sq, Sk)
    return n * (n + 1) // 2 + max(0, Sq - Sk) * Sk


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _groups(rng, H):
    return rng.choice([H, H, H // 2 if H % 2 == 0 else H, H // 4 if H % 4 == 0 else H])


# algorithmic FLOPs a drawn case may have, by what its path can do with them
# (the headline step has 1.9e12): small head dims, full precision, dropout, a
# bias, padded head dims and 256 run at lower rates
_MOST = {"plain": 1.2e12, "dropout": 2e11, "fp32": 5e10, "bias": 2e11, "odd_dim": 3e11}


def _draw_one(rng):
    what = rng.choice(["infer", "infer", "decode", "decode", "train", "train", "cross", "dropout", "fp32", "bias",
                       "odd_dim", "module"])
    dt = rng.choice(["fp16", "bf16"])
    D = rng.choice([64, 64, 128, 128, 32])
    H = rng.choice([8, 12, 16, 20, 32])
    causal = rng.random() < 0.6
    if what == "infer":
        S = _log(rng, 100, 16384)
        return "plain", _case("", "infer", _log(rng, 1, 8), S, S, H, _groups(rng, H), D, dt, causal,
                              qk_std=rng.choice([1.0, 1.0, 2.0]))
    if what == "decode":
        Hkv = rng.choice([H, H // 4, H // 4 if H % 8 else H // 8])
        return "plain", _case("", "decode", _log(rng, 1, 48), rng.choice([1, 1, 1, rng.randint(2, 8)]),
                              _log(rng, 512, 32768), H, Hkv, rng.choice([64, 128, 128]), dt)
    if what == "train":
        S = _log(rng, 200, 8192)
        return "plain", _case("", "train", _log(rng, 1, 8), S, S, H, _groups(rng, H), D, dt, causal)
    if what == "cross":
        return "plain", _case("", "train", _log(rng, 1, 16), _log(rng, 64, 4096), _log(rng, 64, 2048), H, H,
                              rng.choice([64, 64, 128]), dt)
    if what == "dropout":
        S = _log(rng, 200, 2048)
        return what, _case("", "train", _log(rng, 1, 8), S, S, H, H, D, dt, causal, p=rng.choice([0.1, 0.2]))
    if what == "fp32":
        S = _log(rng, 100, 2048)
        return what, _case("", rng.choice(["train", "infer"]), _log(rng, 1, 8), S, S, H, H, D, "fp32", causal,
                           p=rng.choice([0.0, 0.1]))
    if what == "bias":
        S = _log(rng, 200, 2304)
        return what, _case("", "train", _log(rng, 1, 4), S, S, H, H, rng.choice([64, 128]), dt, causal,
                           bias=rng.choice(["heads", "full"]))
    if what == "odd_dim":
        S = _log(rng, 200, 2304)
        return what, _case("", rng.choice(["train", "train", "infer"]), _log(rng, 1, 8), S, S, H, H,
                           rng.choice([72, 80, 96, 112, 160, 192, 256]), dt, causal)
    S = _log(rng, 64, 2048)
    return "bias", _case("", "module", _log(rng, 1, 16), S, S, 12, 12, 64, dt, False, bias="padding")


def draw(rng):
    while True:
        family, c = _draw_one(rng)
        cache = 4 * c["B"] * c["Sk"] * c["Hkv"] * c["D"]
        if work(c)["flops"] <= _MOST[family] * min(1.0, c["D"] / 128) and cache <= 2 ** 31:
            del c["name"]
            return c


# ---------------------------------------------------------------------------
# inputs

def _tensors(case, seed):
    """q, k, v (and dO, the bias or the padding mask where the case has them),
    from the seed alone."""
    g = torch.Generator("cuda").manual_seed(int(seed))
    dt = _DTYPES[case["dtype"]]
    B, Sq, Sk, H, Hkv, D = (case[n] for n in ("B", "Sq", "Sk", "H", "Hkv", "D"))

    def randn(*shape, std=1.0):
        x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
        return (x * std if std != 1.0 else x).to(dt)

    t = {}
    if case["kind"] == "module":
        E = H * D
        t["x"] = randn(B, Sq, E)
        bound = math.sqrt(6.0 / (2 * E))  # Xavier uniform
        for n in ("q_proj", "k_proj", "v_proj", "out_proj"):
            t[n + ".weight"] = ((torch.rand((E, E), generator=g, device="cuda") * 2 - 1) * bound).to(dt)
            t[n + ".bias"] = randn(E, std=0.02)
        lengths = torch.randint(Sk // 2, Sk + 1, (B,), generator=g, device="cuda")
        t["pad"] = torch.arange(Sk, device="cuda")[None, :] >= lengths[:, None]
        return t
    t["q"] = randn(B, Sq, H, D, std=case["qk_std"])
    # a decoder's cache holds room for further tokens: its filled part is a view
    room = 256 - Sk % 256 if case["kind"] == "decode" else 0
    t["k"] = randn(B, Sk + room, Hkv, D, std=case["qk_std"])[:, :Sk]
    t["v"] = randn(B, Sk + room, Hkv, D)[:, :Sk]
    if case["kind"] == "train":
        t["do"] = randn(B, Sq, H, D)
    if case["bias"] == "heads":
        t["bias"] = randn(1, H, Sq, Sk)
    elif case["bias"] == "full":
        t["bias"] = randn(B, H, Sq, Sk)
    return t


def prepare(case, seed):
    t = _tensors(case, seed)
    state = {"case": case, "dropout_seed": 1000 + int(seed), **t}
    if case["kind"] == "module":
        m = EnhancedMultiHeadAttention(case["H"] * case["D"], case["H"])
        m.to(device="cuda", dtype=_DTYPES[case["dtype"]]).eval()
        with torch.no_grad():
            for n, w in m.named_parameters():
                w.copy_(t[n])
        state["module"] = m
    elif case["kind"] == "train":
        for n in ("q", "k", "v", "bias"):
            if n in t:
                t[n].requires_grad_(True)
    return state


def run(state):
    c = state["case"]
    if c["kind"] == "module":
        with torch.no_grad():
            return state["module"](state["x"], key_padding_mask=state["pad"])[0]
    q, k, v = state["q"], state["k"], state["v"]
    if c["kind"] in ("infer", "decode"):
        with torch.no_grad():
            if c["p"] > 0:
                return fa.flash_attention_v100(q, k, v, causal=c["causal"], dropout_p=c["p"],
                                               dropout_seed=state["dropout_seed"], dropout_offset=0)
            return fa.flash_attention_v100(q, k, v, causal=c["causal"])
    bias = state.get("bias")
    if c["p"] > 0:
        o = fa.flash_attention_v100(q, k, v, causal=c["causal"], dropout_p=c["p"], bias=bias,
                                    dropout_seed=state["dropout_seed"], dropout_offset=0)
    else:
        o = fa.flash_attention_v100(q, k, v, causal=c["causal"], bias=bias)
    leaves = (q, k, v) if bias is None else (q, k, v, bias)
    grads = torch.autograd.grad(o, leaves, state["do"])
    return (o.detach(),) + tuple(grads)


def work(case):
    es = 4 if case["dtype"] == "fp32" else 2
    B, Sq, Sk, H, Hkv, D = (case[n] for n in ("B", "Sq", "Sk", "H", "Hkv", "D"))
    nq, nk = B * Sq * H * D, B * Sk * Hkv * D
    flops = 4.0 * B * H * _pairs(case) * D
    if case["kind"] == "module":
        E = H * D
        # x and out, the four projections' weights and biases, the mask
        return {"bytes": es * (2 * B * Sq * E + 4 * (E * E + E)) + B * Sk, "flops": flops + 8.0 * B * Sq * E * E}
    nbytes = es * (2 * nq + 2 * nk)
    if case["kind"] == "train":
        # dO in, dQ, dK, dV out; the bias read and its gradient written
        nbytes += es * (2 * nq + 2 * nk)
        flops *= 3.5
        nb = {"none": 0, "heads": H * Sq * Sk, "full": B * H * Sq * Sk}[case["bias"]]
        nbytes += 2 * es * nb
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # the 2-norm errors against 64 bits measured over the listed and many drawn
    # cases are at most 3.3e-4 (fp16), 2.6e-3 (bf16) and 5e-7 (fp32); the
    # layer, whose projections round too, 5e-4 and 3.9e-3.  About four times that.
    if case["kind"] == "module":
        return {"rel": {"fp16": 2e-3, "bf16": 1.6e-2}[case["dtype"]]}
    return {"rel": {"fp16": 1.4e-3, "bf16": 1e-2, "fp32": 2e-6}[case["dtype"]]}


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch

def _philox_keep(seed, first, rows, cols, p):
    """Keep mask of the dropout stream for the counters first + row * cols + col:
    word 0 of Philox4x32-10 (Salmon et al., SC'11) on (lo, hi, 0, 0) with the
    seed as key, folded to 31 bits and scaled to [0, 1) in float32; kept where
    it exceeds p."""
    m32 = 0xFFFFFFFF
    ctr = first + torch.arange(rows * cols, device="cuda", dtype=torch.int64)
    c = [ctr & m32, ctr >> 32, torch.zeros_like(ctr), torch.zeros_like(ctr)]
    k0, k1 = seed & m32, (seed >> 32) & m32

    def mul(a, m):  # (high, low) words of the 64-bit product
        lo16, hi16 = (a & 0xFFFF) * m, (a >> 16) * m
        mid = hi16 + (lo16 >> 16)
        return mid >> 16, ((mid & 0xFFFF) << 16) | (lo16 & 0xFFFF)

    for _ in range(10):
        ha, la = mul(c[0], 0xD2511F53)
        hb, lb = mul(c[2], 0xCD9E8D57)
        c = [hb ^ c[1] ^ k0, lb, ha ^ c[3] ^ k1, la]
        k0, k1 = (k0 + 0x9E3779B9) & m32, (k1 + 0xBB67AE85) & m32
    x = torch.where(c[0] >= 2 ** 31, m32 - c[0], c[0])
    u = x.to(torch.float32) * torch.tensor(4.6566127342e-10, dtype=torch.float32, device="cuda")
    return (u > torch.tensor(p, dtype=torch.float32, device="cuda")).view(rows, cols)


def _exact_attention(case, t, seed):
    """O and the gradients in float64, one (batch, head) at a time."""
    B, Sq, Sk, H, Hkv, D, p = (case[n] for n in ("B", "Sq", "Sk", "H", "Hkv", "D", "p"))
    scale = D ** -0.5
    f64 = dict(device="cuda", dtype=torch.float64)
    train, bias = case["kind"] == "train", t.get("bias")
    o = torch.empty((B, Sq, H, D), **f64)
    if train:
        dq = torch.empty((B, Sq, H, D), **f64)
        dk, dv = torch.zeros((B, Sk, Hkv, D), **f64), torch.zeros((B, Sk, Hkv, D), **f64)
        db = torch.zeros(bias.shape, **f64) if bias is not None else None
    hidden = torch.ones((Sq, Sk), device="cuda", dtype=torch.bool).triu(1) if case["causal"] else None
    for b in range(B):
        for h in range(H):
            hk = h // (H // Hkv)
            q, k, v = t["q"][b, :, h].double(), t["k"][b, :, hk].double(), t["v"][b, :, hk].double()
            s = (q @ k.t().contiguous()) * scale
            if bias is not None:
                s += bias[b if bias.shape[0] > 1 else 0, h].double()
            if "pad" in t:
                s.masked_fill_(t["pad"][b][None, :], float("-inf"))
            if hidden is not None:
                s.masked_fill_(hidden, float("-inf"))
            pr = torch.softmax(s, dim=-1)
            drop = None
            if p > 0:
                keep = _philox_keep(1000 + int(seed), (b * H + h) * Sq * Sk, Sq, Sk, p)
                drop = keep.double() / (1.0 - p)
            pd = pr if drop is None else pr * drop
            o[b, :, h] = pd @ v
            if train:
                do = t["do"][b, :, h].double()
                dp = do @ v.t().contiguous()
                if drop is not None:
                    dp *= drop
                ds = pr * (dp - (do * o[b, :, h]).sum(-1, keepdim=True))
                dq[b, :, h] = (ds @ k) * scale
                dk[b, :, hk] += (ds.t().contiguous() @ q) * scale
                dv[b, :, hk] += pd.t().contiguous() @ do
                if db is not None:
                    db[b if bias.shape[0] > 1 else 0, h] += ds
    if not train:
        return o
    return (o, dq, dk, dv) if db is None else (o, dq, dk, dv, db)


def exact(case, seed):
    t = _tensors(case, seed)
    if case["kind"] != "module":
        return _exact_attention(case, t, seed)
    B, S, H, D = case["B"], case["Sq"], case["H"], case["D"]
    x = t["x"].double()

    def linear(y, n):
        return y @ t[n + ".weight"].double().t().contiguous() + t[n + ".bias"].double()

    q, k, v = (linear(x, n).view(B, S, H, D) for n in ("q_proj", "k_proj", "v_proj"))
    o = _exact_attention(case, {"q": q, "k": k, "v": v, "pad": t["pad"]}, seed)
    return linear(o.reshape(B, S, H * D), "out_proj")
