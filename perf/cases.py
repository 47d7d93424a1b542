"""The workloads this framework is timed on: what a program calls through its public entry points.

``functional.scaled_dot_product_attention`` (prefill and training; flash kernels, and the composed
path when dropout is asked for), ``functional.flash_decode`` (one generation step against a KV
cache) and ``nn.MultiheadAttention``, over the sizes of this repository's own configurations and
tests: sequences of 32 to 8192, caches of 64 to 16384 keys, head dims 32 to 256, float32 and bf16,
causal, unmasked and key-padded, equal and grouped heads.

A case is a dict: ``kind`` (decode, attention, dropout, mha), ``dtype``, B, H, Hkv, L, S, E (head
dim), ``mask`` (causal, none, padding) and ``train`` (forward + backward, or forward only).
"""
import math

import numpy as np
import torch

from densecore_amd import functional, nn
from densecore_amd import random as dc_random

DEV = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
DROPOUT_P = 0.1


def _case(name, kind, dtype, B, H, Hkv, L, S, E, mask, train):
    c = {"kind": kind, "dtype": dtype, "B": B, "H": H, "Hkv": Hkv, "L": L, "S": S, "E": E,
         "mask": mask, "train": train}
    return {"name": name, **c} if name else c


def listed():
    return [
        # One generated token of a small model, its context nearly full: latency, not bytes.
        _case("decode_small_f32", "decode", "f32", 1, 6, 6, 1, 255, 64, "none", False),
        # A serving step of a large float32 batch: the KV cache streams once (4.3 GB).
        _case("decode_batch_f32", "decode", "f32", 32, 32, 32, 1, 4096, 128, "none", False),
        # A serving step of a grouped-head bf16 model with long contexts.
        _case("decode_gqa_bf16", "decode", "bf16", 16, 32, 8, 1, 8192, 128, "none", False),
        # Scoring (forward only) of short texts with a small float32 model.
        _case("prefill_short_f32", "attention", "f32", 64, 6, 6, 256, 256, 64, "causal", False),
        # A training step's attention in a 12-head float32 language model.
        _case("train_causal_f32", "attention", "f32", 8, 12, 12, 1024, 1024, 64, "causal", True),
        # A training step's attention in a float32 encoder on batches padded to the longest text.
        _case("train_padded_f32", "attention", "f32", 16, 16, 16, 512, 512, 64, "padding", True),
        # A training step's attention at long context in bf16: the largest case.
        _case("train_long_bf16", "attention", "bf16", 2, 32, 32, 8192, 8192, 128, "causal", True),
        # Reading one user's prompt, of no round length, with a grouped-head bf16 model.
        _case("prefill_gqa_bf16", "attention", "bf16", 1, 32, 8, 3001, 3001, 128, "causal", False),
        # A training step's attention in a bf16 encoder on padded batches.
        _case("train_padded_bf16", "attention", "bf16", 16, 12, 12, 512, 512, 64, "padding", True),
        # A training step's attention with dropout on the weights (the composed path).
        _case("train_dropout_f32", "dropout", "f32", 8, 12, 12, 512, 512, 64, "causal", True),
        # A training step of the whole attention module, 768 wide, on padded batches.
        _case("train_module_f32", "mha", "f32", 8, 12, 12, 384, 384, 64, "padding", True),
        # A training step's attention at head dim 256 in bf16.
        _case("train_wide_bf16", "attention", "bf16", 2, 16, 16, 2048, 2048, 256, "causal", True),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode"] * 4 + ["attention"] * 7 + ["wide"] * 2 + ["dropout", "mha"])
    if kind == "decode":
        dtype = rng.choice(["f32", "bf16"])
        E = rng.choice([64, 64, 80, 128, 128, 128, 256])
        rep = rng.choice([1, 1, 2, 4, 8])
        Hkv = rng.choice([1, 2, 4, 6, 8, 12, 16, 32])
        while Hkv * rep > 64:
            Hkv //= 2
        B, S = _log_int(rng, 1, 64), _log_int(rng, 64, 16384)
        elem = 4 if dtype == "f32" else 2
        while B > 1 and 2 * B * Hkv * S * E * elem > 4.0e9:
            B //= 2
        return _case(None, "decode", dtype, B, Hkv * rep, Hkv, 1, S, E, "none", False)
    if kind == "mha":
        B, L = _log_int(rng, 1, 32), _log_int(rng, 16, 768)
        H, E = rng.choice([6, 8, 12, 16]), rng.choice([32, 64, 64, 80])
        while B > 1 and B * H * L * L > 2 ** 25:
            B //= 2
        return _case(None, "mha", "f32", B, H, H, L, L, E, rng.choice(["padding", "none"]), True)
    if kind == "dropout":
        B, L = _log_int(rng, 1, 32), _log_int(rng, 32, 1024)
        H, E = rng.choice([4, 6, 8, 12, 16]), rng.choice([32, 64, 64, 96, 128])
        while B > 1 and B * H * L * L > 2 ** 25:
            B //= 2
        return _case(None, "dropout", "f32", B, H, H, L, L, E, rng.choice(["causal", "none"]), True)
    dtype = rng.choice(["f32", "f32", "bf16"]) if kind == "attention" else rng.choice(["f32", "bf16"])
    train = rng.random() < 0.65
    mask = rng.choice(["causal", "causal", "causal", "none", "padding"])
    if kind == "wide":
        E = rng.choice([160, 192, 256])
    else:
        E = rng.choice([32, 64, 64, 64, 80, 96, 128, 128, 128])
    L = _log_int(rng, 32, 8192)
    # Cross attention now and then: another number of keys than of queries.
    S = _log_int(rng, 32, 4096) if mask != "causal" and rng.random() < 0.4 else L
    rep = rng.choice([1, 1, 1, 2, 4])
    Hkv = rng.choice([1, 2, 4, 6, 8, 12, 16])
    B = _log_int(rng, 1, 64)
    c = _case(None, "attention", dtype, B, Hkv * rep, Hkv, L, S, E, mask, train)
    # No dearer than the largest listed case (float32 products run at about a tenth of bf16's rate;
    # the wide heads at less).
    most = {"f32": 4.0e10, "bf16": 6.0e11}[dtype] / (4 if kind == "wide" else 1)
    while work(c)["flops"] > most:
        if c["B"] > 1:
            c["B"] = (c["B"] + 1) // 2
        elif c["Hkv"] > 1:
            c["Hkv"] = (c["Hkv"] + 1) // 2
            c["H"] = c["Hkv"] * rep
        else:
            same = c["L"] == c["S"]
            c["L"] = c["L"] * 3 // 4
            c["S"] = c["L"] if same else c["S"] * 3 // 4
    return c


# ---- inputs ----

def _lengths(case, seed):
    """The padded texts' lengths: evenly spread from a quarter of S to S, in a random order."""
    B, S = case["B"], case["S"]
    lens = np.array([max(1, S // 4 + (S - S // 4) * (b + 1) // B) for b in range(B)])
    return np.random.RandomState(seed % 2 ** 32).permutation(lens)


def _inputs(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    B, H, Hkv, L, S, E = (case[k] for k in ("B", "H", "Hkv", "L", "S", "E"))

    def normal(*shape, std=1.0):
        return (torch.randn(shape, generator=gen, device=DEV, dtype=torch.float32) * std).to(dtype)

    x = {}
    if case["kind"] == "mha":
        width = H * E
        x["x"], x["g"] = normal(B, L, width), normal(B, L, width)
        x["in_w"] = normal(3 * width, width, std=width ** -0.5)
        x["in_b"] = normal(3 * width, std=0.02)
        x["out_w"] = normal(width, width, std=width ** -0.5)
        x["out_b"] = normal(width, std=0.02)
    else:
        x["q"], x["k"], x["v"] = normal(B, H, L, E), normal(B, Hkv, S, E), normal(B, Hkv, S, E)
        if case["train"]:
            x["g"] = normal(B, H, L, E)
    if case["mask"] == "padding":
        lens = torch.from_numpy(_lengths(case, seed)).to(DEV)
        x["valid"] = torch.arange(S, device=DEV)[None, :] < lens[:, None]
    return x


def prepare(case, seed):
    x = _inputs(case, seed)
    state = {"case": case, "seed": seed % 2 ** 32}
    if case["kind"] == "mha":
        m = nn.MultiheadAttention(case["H"] * case["E"], case["H"], batch_first=True, device=DEV)
        with torch.no_grad():
            m.in_proj_weight.copy_(x["in_w"])
            m.in_proj_bias.copy_(x["in_b"])
            m.out_proj.weight.copy_(x["out_w"])
            m.out_proj.bias.copy_(x["out_b"])
        state["module"] = m
        state["x"], state["g"] = x["x"].requires_grad_(True), x["g"]
        state["pad"] = ~x["valid"] if "valid" in x else None
        return state
    if case["train"]:
        for n in ("q", "k", "v"):
            x[n].requires_grad_(True)
    state.update(x)
    # The API's boolean mask: True where attention is allowed, one row of keys per text.
    state["mask"] = x["valid"][:, None, None, :] if "valid" in x else None
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode":
        return functional.flash_decode(state["q"], state["k"], state["v"])
    if kind == "mha":
        m, x = state["module"], state["x"]
        out, _ = m(x, x, x, key_padding_mask=state["pad"], need_weights=False)
        params = (x, m.in_proj_weight, m.in_proj_bias, m.out_proj.weight, m.out_proj.bias)
        return [out.detach(), *torch.autograd.grad(out, params, state["g"])]
    q, k, v = state["q"], state["k"], state["v"]
    dropout_p = 0.0
    if kind == "dropout":
        dropout_p = DROPOUT_P
        dc_random.manual_seed(state["seed"])  # a step whose masks can be drawn again
    out = functional.scaled_dot_product_attention(
        q, k, v, attn_mask=state["mask"], dropout_p=dropout_p, is_causal=case["mask"] == "causal",
        enable_gqa=case["Hkv"] != case["H"])
    if not case["train"]:
        return out
    return [out.detach(), *torch.autograd.grad(out, (q, k, v), state["g"])]


# ---- what a pass cannot do without ----

def _pairs(case):
    """Visible (query, key) pairs over the batch, per head."""
    B, L, S = case["B"], case["L"], case["S"]
    if case["mask"] == "causal":
        n = min(L, S)
        return B * (n * (n + 1) // 2 + (L - n) * S)
    if case["mask"] == "padding":
        return L * int(_lengths(case, 0).sum())
    return B * L * S


def work(case):
    B, H, Hkv, L, S, E = (case[k] for k in ("B", "H", "Hkv", "L", "S", "E"))
    elem = 4 if case["dtype"] == "f32" else 2
    fwd = 4.0 * H * E * _pairs(case)
    if case["kind"] == "mha":
        w = H * E
        linear = 2.0 * B * L * w * w * 4  # three input projections and the output's
        return {"flops": 3 * linear + 3.5 * fwd, "bytes": 4.0 * (4 * B * L * w + 2 * (4 * w * w + 4 * w))}
    qn, kn = B * H * L * E, 2 * B * Hkv * S * E
    if not case["train"]:
        return {"flops": fwd, "bytes": float(elem) * (2 * qn + kn)}
    # q, k, v and the gradient in; the output and three gradients out.
    return {"flops": 3.5 * fwd, "bytes": float(elem) * (4 * qn + 2 * kn)}


# ---- what the results are held to ----

def tolerance(case):
    """About four times the distance from float64 (``exact``) measured over these cases and drawn
    ones, and room for the longest rows: float32 sums up to 1.4e-6, bf16 outputs 1.8e-3."""
    if case["dtype"] == "bf16":
        return {"rel": 8e-3}
    return {"rel": 1e-5}


def _keep_mask(case, seed):
    """The dropout mask of a freshly seeded generator: PyTorch's mt19937, two 32-bit outputs per
    draw with the first as the high half, a 53-bit uniform below 1 - p keeps."""
    n = case["B"] * case["H"] * case["L"] * case["S"]
    bits = np.random.MT19937()
    bits._legacy_seeding(seed % 2 ** 32)
    raw = bits.random_raw(2 * n).astype(np.uint64)
    r = ((raw[0::2] << np.uint64(32)) | raw[1::2]) & np.uint64(2 ** 53 - 1)
    keep = r.astype(np.float64) * 2.0 ** -53 < 1 - DROPOUT_P
    return torch.from_numpy(keep).to(DEV).reshape(case["B"], case["H"], case["L"], case["S"])


def _attention64(case, x, g, keep=None):
    """Attention in float64, one kv head at a time: out and, given ``g``, dq, dk, dv."""
    B, H, Hkv, L, S, E = (case[k] for k in ("B", "H", "Hkv", "L", "S", "E"))
    rep, scale = H // Hkv, 1.0 / math.sqrt(E)
    out = torch.empty(B, H, L, E, dtype=torch.float64, device=DEV)
    grads = [torch.empty(B, n, m, E, dtype=torch.float64, device=DEV)
             for n, m in ((H, L), (Hkv, S), (Hkv, S))] if g is not None else []
    hidden = None
    if case["mask"] == "causal":
        hidden = torch.ones(L, S, dtype=torch.bool, device=DEV).triu(1).repeat(rep, 1)
    for b in range(B):
        if case["mask"] == "padding":
            hidden = ~x["valid"][b][None, :]
        for j in range(Hkv):
            heads = slice(j * rep, (j + 1) * rep)
            q = x["q"][b, heads].double().reshape(rep * L, E)
            k, v = x["k"][b, j].double(), x["v"][b, j].double()
            p = (q * scale) @ k.t().contiguous()
            if hidden is not None:
                p.masked_fill_(hidden, float("-inf"))
            p = torch.softmax(p, -1)
            noise = 1.0
            if keep is not None:
                noise = keep[b, heads].reshape(rep * L, S).double() / (1 - DROPOUT_P)
            w = p * noise
            o = w @ v
            out[b, heads] = o.reshape(rep, L, E)
            if g is None:
                continue
            do = g[b, heads].double().reshape(rep * L, E)
            grads[2][b, j] = w.t().contiguous() @ do
            dw = do @ v.t().contiguous()
            # sum over keys of w * dw is the row sum of do * o
            ds = p * (dw * noise - (do * o).sum(-1, keepdim=True)) * scale
            grads[0][b, heads] = (ds @ k).reshape(rep, L, E)
            grads[1][b, j] = ds.t().contiguous() @ q
    return [out, *grads]


def exact(case, seed):
    x = _inputs(case, seed)
    with torch.no_grad():
        if case["kind"] != "mha":
            keep = _keep_mask(case, seed) if case["kind"] == "dropout" else None
            r = _attention64(case, x, x.get("g"), keep)
            return r if case["train"] else r[0]
        B, H, L, E = (case[k] for k in ("B", "H", "L", "E"))
        w = H * E

        def heads(t):
            return t.reshape(B, L, H, E).transpose(1, 2).contiguous()

        def merge(t):
            return t.transpose(1, 2).reshape(B * L, w)

        rows, g = x["x"].double().reshape(B * L, w), x["g"].double().reshape(B * L, w)
        in_w, out_w = x["in_w"].double(), x["out_w"].double()
        proj = rows @ in_w.t().contiguous() + x["in_b"].double()
        a = dict(x)
        a["q"], a["k"], a["v"] = (heads(p) for p in proj.chunk(3, -1))
        da = heads(g @ out_w)
        attn, dq, dk, dv = _attention64(case, a, da)
        attn = merge(attn)
        out = attn @ out_w.t().contiguous() + x["out_b"].double()
        dproj = torch.cat([merge(t) for t in (dq, dk, dv)], -1)
        return [out.reshape(B, L, w), (dproj @ in_w).reshape(B, L, w), dproj.t().contiguous() @ rows,
                dproj.sum(0), g.t().contiguous() @ attn, g.sum(0)]
