"""A query whose scores are no finite numbers gives NaN in its own row and in no
other: the head_dim-64 kernels sum the probabilities of queries c and c + 16 of a
wave with one matrix instruction, where the other query's enter against zeros and
0 x NaN is NaN.  Every kernel and mask mode that sums so, with NaN and infinite
query rows, and with a NaN key that only the later queries of a causal call see
(several waves then hold both kinds of rows).

Bars for the rows that see none: test_gpu_rowsum.py's (O |x - o| <= 2e-3 + 1e-2
|o| in binary16, 4e-3 + 1.6e-2 |o| in bfloat16; LSE ln(1 + 2^-11), ln(1 + 2^-8)
and 1e-5 (1 + |lse|) for the fp32 sums)."""
import math

import pytest
import torch

import flash_attn_sm75_cuda as _C
from flash_attention_sm75 import flash_attention_forward_ex

pytestmark = pytest.mark.gpu

AUTO, NARROW, WIDE, DYNAMIC, SPLIT, PAIRS = range(6)
CASES = [
    # policy, B, Hq, Hkv, Nq, Nk, causal, mask, bf16
    (NARROW, 1, 2, 2, 300, 333, False, None, False),
    (NARROW, 1, 2, 1, 777, 777, True, None, True),
    (WIDE, 1, 2, 2, 600, 700, False, None, True),
    (WIDE, 1, 2, 2, 700, 700, True, None, False),
    (DYNAMIC, 3, 24, 8, 1000, 1000, True, None, False),
    (SPLIT, 1, 2, 2, 500, 1000, False, None, False),
    (SPLIT, 1, 2, 2, 640, 640, True, None, True),
    (PAIRS, 1, 2, 2, 640, 640, True, None, False),     # five blocks: a middle one alone
    (PAIRS, 1, 2, 1, 1000, 1000, True, None, True),
    (NARROW, 2, 2, 2, 300, 300, False, "bits", False),
    (WIDE, 2, 2, 2, 600, 600, True, "bits", True),
    (NARROW, 2, 2, 1, 300, 500, False, "keys", False),
    (NARROW, 2, 2, 1, 500, 500, True, "keys", True),
    (AUTO, 3, 24, 24, 1000, 333, False, None, False),  # several rounds: v_dot2 sums
]


@pytest.mark.parametrize("poison", ["q", "k"])
@pytest.mark.parametrize("policy,B,Hq,Hkv,Nq,Nk,causal,mask,bf16", CASES)
def test_other_rows_are_untouched(device, policy, B, Hq, Hkv, Nq, Nk, causal, mask, bf16, poison):
    print(f"[nonfinite] {(policy, B, Hq, Hkv, Nq, Nk, causal, mask, bf16, poison)}", flush=True)
    if poison == "k" and not causal:
        pytest.skip("every query sees the key")
    dt = torch.bfloat16 if bf16 else torch.float16
    g = torch.Generator("cuda").manual_seed(Nq + Nk)
    q = torch.randn(B, Hq, Nq, 64, device=device, generator=g).to(dt)
    k, v = (torch.randn(B, Hkv, Nk, 64, device=device, generator=g).to(dt) for _ in range(2))
    m = None
    if mask == "bits":
        m = torch.rand(B, 1, Nq, Nk, device=device, generator=g) < 0.7
        m[..., 0] = True
    elif mask == "keys":
        m = torch.ones(B, 1, 1, Nk, dtype=torch.bool, device=device)
        m[1, ..., Nk // 2:] = False
    if poison == "q":  # one of a pair (c, c + 16) of a wave, both, in several waves
        q[0, 0, 5, 3] = math.nan
        q[0, 0, 33, 7] = q[0, 0, 49, 7] = math.nan
        q[0, 0, 100, 0] = math.inf
        q[0, 0, Nq - 3, 9] = -math.inf
    else:
        k[0, 0, Nk // 2 + 9, 5] = math.nan
    _C.set_kernel_policy(policy)
    try:
        o, lse = flash_attention_forward_ex(q, k, v, causal=causal, return_lse=True, attn_mask=m)
    finally:
        _C.set_kernel_policy(AUTO)
    ao, ro, al = (4e-3, 1.6e-2, math.log1p(2 ** -8)) if bf16 else (2e-3, 1e-2, math.log1p(2 ** -11))
    for b, h in {(0, 0), (B - 1, Hq - 1)}:
        kv = h // (Hq // Hkv)
        s = q[b, h].double() @ k[b, kv].double().t() / 8.0
        hidden = torch.zeros(Nq, Nk, dtype=torch.bool, device=device)
        if causal:
            hidden |= torch.ones_like(hidden).triu_(1)
        if m is not None:
            hidden |= ~m[b, 0].expand(Nq, Nk)
        s.masked_fill_(hidden, -math.inf)
        bad = ~(s.masked_fill(hidden, 0.0).isfinite().all(-1))
        assert bad.any() == ((b, kv) == (0, 0) and (poison == "k" or h == 0))
        assert o[b, h][bad].isnan().all() and lse[b, h][bad].isnan().all()
        s = s[~bad]
        want_l = torch.logsumexp(s, -1)
        want = torch.softmax(s, -1) @ v[b, kv].double()
        got, got_l = o[b, h][~bad].double(), lse[b, h][~bad].double()
        print(f"  {int(got.isnan().any(-1).sum())} rows of others are NaN", flush=True)
        assert ((got_l - want_l).abs() <= al + 1e-5 * (1 + want_l.abs())).all()
        assert ((got - want).abs() <= ao + ro * want.abs()).all()
