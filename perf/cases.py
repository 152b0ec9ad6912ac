"""The attention calls that programs make of this package, for timing it and checking its outputs.

Each case is one call (or one training step of one attention layer) through a public entry point:

  forward   flash_attention_forward, the drop-in call: contiguous [B, H, N, D] float16
  lse       flash_attention_forward_lse, the same with the row log-sum-exp
  ex        flash_attention_forward_ex, separate query and key lengths, either dtype
  sdpa      torch's scaled_dot_product_attention with the package's patch applied, called the way
            HuggingFace models call it: [B, N, H, D] buffers viewed as [B, H, N, D] in prefill, a
            contiguous key/value cache in decode, enable_gqa, masks as bool tensors
  train     flash_attention and the gradients of Q, K and V for a given dO

Masks: "keys" hides each sequence's tail from every query ([B, 1, 1, Nk], a padded batch in decode);
"causal" is the causal mask with left padding as one bool tensor ([B, 1, N, N], a padded prefill).
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "flash-attention-sm75-register-fused_amd", "src"))
import flash_attention_sm75 as fa  # noqa: E402
from flash_attention_sm75 import sdpa_patch  # noqa: E402

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _case(name, call, dtype, b, hq, hkv, nq, nk, d, causal="none", mask="none", peaked=False):
    c = {"call": call, "dtype": dtype, "b": b, "hq": hq, "hkv": hkv, "nq": nq, "nk": nk, "d": d,
         "causal": causal, "mask": mask, "peaked": peaked}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: one head of a short sequence, where the launch and the host count
        _case("one_head_512", "forward", "fp16", 1, 1, 1, 512, 512, 64),
        # an encoder layer on a batch of ordinary length, with the row log-sum-exp
        _case("encoder_1024", "lse", "fp16", 4, 12, 12, 1024, 1024, 64),
        # a small decoder's causal layer
        _case("causal_2048", "forward", "fp16", 4, 8, 8, 2048, 2048, 64, "top_left"),
        # a Llama-shaped prefill (the repository's headline configuration)
        _case("prefill_8192", "forward", "fp16", 1, 32, 8, 8192, 8192, 128, "top_left"),
        # a later chunk of a long prompt against the cache
        _case("chunk_2048_8192", "ex", "bf16", 1, 32, 8, 2048, 8192, 128, "bottom_right"),
        # a small GQA model's prefill at an odd length, through the patch
        _case("ragged_prefill_1777", "sdpa", "bf16", 3, 14, 2, 1777, 1777, 64, "top_left"),
        # a padded batch's prefill: the mask arrives as a bool tensor
        _case("padded_prefill_2048", "sdpa", "fp16", 4, 14, 2, 2048, 2048, 64, "none", "causal"),
        # one generated token of one sequence: once per layer and token, latency counts
        _case("decode_step_4097", "sdpa", "bf16", 1, 14, 2, 1, 4097, 64),
        # one token of a serving batch: streaming the cache
        _case("decode_batch_8192", "ex", "fp16", 32, 32, 8, 1, 8192, 128),
        # one token of a padded batch with long contexts
        _case("decode_padded_32768", "sdpa", "bf16", 16, 14, 2, 1, 32768, 64, "none", "keys"),
        # a training step's attention, a small GQA model
        _case("train_2048", "train", "bf16", 4, 14, 2, 2048, 2048, 64, "top_left"),
        # a training step's attention, Llama-shaped: the largest
        _case("train_8192", "train", "bf16", 1, 32, 8, 8192, 8192, 128, "top_left"),
    ]


# (query heads, KV heads, head_dim) of the repository's configurations, tests and benchmark
HEADS = [(1, 1, 64), (8, 8, 64), (8, 8, 128), (12, 12, 64), (14, 2, 64), (16, 4, 128), (32, 8, 64),
         (32, 8, 128), (64, 8, 128)]


def _length(rng, lo, hi):
    """Spread over the logarithm; one in three a multiple of 64."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(64, n // 64 * 64) if rng.random() < 1 / 3 else n


def draw(rng):
    kind = rng.choice(["forward", "forward", "sdpa", "padded", "chunk", "decode", "decode",
                       "decode_padded", "train", "train", "train"])
    hq, hkv, d = rng.choice(HEADS)
    b = rng.choice([1, 1, 2, 3, 4, 8])
    dtype = rng.choice(["fp16", "bf16"])
    if kind in ("decode", "decode_padded"):
        nk = _length(rng, 128, 65536)
        b = rng.choice([1, 1, 2, 7, 16, 32])
        while b > 1 and 4 * b * hkv * nk * d > 2.5e9:
            b //= 2
        if kind == "decode":
            return _case("", rng.choice(["ex", "sdpa"]), dtype, b, hq, hkv, 1, nk, d)
        return _case("", "sdpa", dtype, b, hq, hkv, 1, nk, d, "none", "keys")
    n = _length(rng, 128, 8192)
    nk = n
    most = 5e11 if kind != "train" else 1.5e11  # of 4 B Hq Nq Nk D
    if kind == "chunk":
        nk = n + _length(rng, 128, 8192)
        most = 3e11
    while 4 * b * hq * n * nk * d > most and b > 1:
        b //= 2
    while 4 * b * hq * n * nk * d > most:
        n, nk = n * 3 // 4, nk * 3 // 4
    causal = rng.choice(["none", "top_left"])
    if kind == "forward":
        return _case("", rng.choice(["forward", "lse"]), "fp16", b, hq, hkv, n, n, d, causal,
                     "none", rng.random() < 0.25)
    if kind == "sdpa":
        return _case("", "sdpa", dtype, b, hq, hkv, n, n, d, causal)
    if kind == "padded":
        return _case("", "sdpa", dtype, b, hq, hkv, n, n, d, "none", "causal")
    if kind == "chunk":
        return _case("", "ex", dtype, b, hq, hkv, n, nk, d, "bottom_right")
    return _case("", "train", dtype, b, hq, hkv, n, n, d, causal,
                 "causal" if causal == "none" and rng.random() < 0.4 else "none")


def _lengths(c):
    """The padded batch's sequence lengths: evenly spread from half the longest to all of it."""
    b, nk = c["b"], c["nk"]
    return [nk - (nk // 2) * i // max(1, b) for i in range(b)]


def prepare(c, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    dev, dt = "cuda", DTYPES[c["dtype"]]
    b, hq, hkv, nq, nk, d = (c[k] for k in ("b", "hq", "hkv", "nq", "nk", "d"))

    def randn(h, n, rows_first):
        if rows_first:  # [B, N, H, D] storage, as the projections write it
            return torch.randn(b, n, h, d, device=dev, dtype=dt, generator=g).transpose(1, 2)
        return torch.randn(b, h, n, d, device=dev, dtype=dt, generator=g)

    model = c["call"] in ("sdpa", "train")
    q = randn(hq, nq, model)
    k = randn(hkv, nk, model and nq > 1)
    v = randn(hkv, nk, model and nq > 1)
    if c["peaked"]:  # a few large keys: the running row maximum is raised often
        q, v = q * 0.5, v * 0.5
        big = torch.rand(b, hkv, nk, 1, device=dev, generator=g) < 0.05
        k = torch.where(big, 2.0 * k, 0.5 * k)
    s = {"case": c, "q": q, "k": k, "v": v, "mask": None}
    if c["mask"] != "none":
        order = torch.randperm(b, device=dev, generator=g)
        n_of = torch.tensor(_lengths(c), device=dev)[order]
        key = torch.arange(nk, device=dev)
        if c["mask"] == "keys":  # the cache is filled from the front
            s["mask"] = (key[None, :] < n_of[:, None])[:, None, None, :]
        else:  # left padding and the causal rule; a padding row sees itself
            row = torch.arange(nq, device=dev)
            m = (key[None, None, :] <= row[None, :, None]) & (key[None, None, :] >= (nk - n_of)[:, None, None])
            s["mask"] = (m | (key[None, :] == row[:, None])[None])[:, None].contiguous()
    if c["call"] == "train":
        s["do"] = randn(hq, nq, True)
        for x in (q, k, v):
            x.requires_grad_()
    if c["call"] == "sdpa":
        sdpa_patch.apply_patch()
    return s


def run(s):
    c, q, k, v = s["case"], s["q"], s["k"], s["v"]
    if c["call"] == "forward":
        return fa.flash_attention_forward(q, k, v, causal=c["causal"] != "none")
    if c["call"] == "lse":
        return fa.flash_attention_forward_lse(q, k, v, causal=c["causal"] != "none")
    causal = False if c["causal"] == "none" else c["causal"]
    if c["call"] == "ex":
        return fa.flash_attention_forward_ex(q, k, v, causal=causal)
    if c["call"] == "sdpa":
        return torch.nn.functional.scaled_dot_product_attention(
            q, k, v, attn_mask=s["mask"], is_causal=bool(causal), enable_gqa=True)
    o = fa.flash_attention(q, k, v, causal=causal, attn_mask=s["mask"])
    return (o,) + torch.autograd.grad(o, (q, k, v), s["do"])


def _visible(c):
    """(query, key) pairs that take part, over the batch, for one head."""
    nq, nk = c["nq"], c["nk"]
    if c["mask"] == "keys":
        return nq * sum(_lengths(c))
    if c["mask"] == "causal":
        return sum(n * (n + 1) // 2 + (nk - n) for n in _lengths(c))
    if c["causal"] == "none":
        return c["b"] * nq * nk
    diag = nk - nq if c["causal"] == "bottom_right" else 0
    return c["b"] * sum(min(nk, i + 1 + diag) for i in range(nq))


def work(c):
    b, hq, hkv, nq, nk, d = (c[k] for k in ("b", "hq", "hkv", "nq", "nk", "d"))
    q_bytes = 2 * b * hq * nq * d
    kv_bytes = 2 * 2 * hkv * d * (sum(_lengths(c)) if c["mask"] == "keys" else b * nk)
    mask_bytes = {"none": 0, "keys": b * nk, "causal": b * nq * nk}[c["mask"]]
    flops = 4 * hq * d * _visible(c)
    bytes_ = 2 * q_bytes + kv_bytes + mask_bytes
    if c["call"] == "lse":
        bytes_ += 4 * b * hq * nq
    if c["call"] == "train":  # dO read, dQ, dK and dV written; five more products of the same size as two
        bytes_ += 2 * q_bytes + kv_bytes
        flops = flops * 7 // 2
    return {"bytes": bytes_, "flops": flops}


def tolerance(c):
    # Measured against 64 bits: 2.3e-4 to 3.8e-4 in float16 (outputs and gradients), 2.1e-3 to 3.0e-3
    # in bfloat16; the probabilities and the results are rounded to the element type.
    return {"rel": {"fp16": 1.5e-3, "bf16": 1.2e-2}[c["dtype"]]}


def exact(c, seed):
    s = prepare(c, seed)
    b, hq, hkv, nq, nk, d = (c[k] for k in ("b", "hq", "hkv", "nq", "nk", "d"))
    scale = 1.0 / math.sqrt(d)
    q, k, v = (s[x].detach() for x in "qkv")
    train = c["call"] == "train"
    o = torch.empty(b, hq, nq, d, dtype=torch.float64, device=q.device)
    lse = torch.empty(b, hq, nq, dtype=torch.float64, device=q.device)
    if train:
        dq = torch.empty_like(o)
        dk = torch.zeros(b, hkv, nk, d, dtype=torch.float64, device=q.device)
        dv = torch.zeros_like(dk)
    hidden = None
    if c["causal"] != "none":
        diag = nk - nq if c["causal"] == "bottom_right" else 0
        hidden = torch.ones(nq, nk, dtype=torch.bool, device=q.device).triu_(1 + diag)
    for i in range(b):
        if s["mask"] is not None:
            hidden = ~s["mask"][i, 0].expand(nq, nk)
        for h in range(hq):
            g = h // (hq // hkv)
            qi, ki, vi = q[i, h].double(), k[i, g].double(), v[i, g].double()
            x = qi @ ki.t() * scale
            if hidden is not None:
                x.masked_fill_(hidden, -math.inf)
            lse[i, h] = torch.logsumexp(x, -1)
            p = x.sub_(lse[i, h][:, None]).exp_()
            o[i, h] = p @ vi
            if train:
                di = s["do"][i, h].double()
                dv[i, g] += p.t() @ di
                ds = di @ vi.t()
                ds.sub_((di * o[i, h]).sum(-1, keepdim=True)).mul_(p).mul_(scale)
                dq[i, h] = ds @ ki
                dk[i, g] += ds.t() @ qi
    if train:
        return o, dq, dk, dv
    return (o, lse) if c["call"] == "lse" else o
