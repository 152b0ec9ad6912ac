"""Head_dim-64 row sums on the matrix pipe (the 16x16x32 MFMAs with a constant
operand) and the launches that take them or the v_dot2 sums: each kernel's
outputs and row LSE against float64 on the device, on both sides of the
one-round rule, and rows whose weights sit in a single key so that a lane or
half-wave taking another query's sum would show.

Bars: the forward's O |x - o| <= 2e-3 + 1e-2 |o| (binary16), 1.6e-2 |o| + 4e-3
(bfloat16); the LSE sums the rounded probabilities, each within 2^-11 (2^-8)
of its value, so it is within ln(1 + 2^-11) = 4.9e-4 (ln(1 + 2^-8) = 3.9e-3)
of the exact one, and 1e-5 for the fp32 sums."""
import math

import pytest
import torch

from flash_attention_sm75 import flash_attention_forward_ex

pytestmark = pytest.mark.gpu

CASES = [
    # B, Hq, Hkv, Nq, Nk, causal, bf16
    (2, 8, 8, 1000, 333, False, False),    # 4 waves, one round: matrix-pipe sums
    (3, 24, 24, 1000, 333, False, True),   # several rounds: v_dot2 sums
    (2, 24, 8, 1000, 700, False, False),   # 256-row workgroups, short rows
    (1, 20, 4, 4097, 4100, False, True),   # several rounds of long rows
    (1, 8, 8, 1100, 2100, False, False),   # key split
    (3, 14, 2, 777, 777, True, True),      # causal, one round
    (8, 16, 4, 1000, 1000, True, False),   # causal, several rounds
    (1, 16, 16, 4100, 4100, True, False),  # paired key split
]


@pytest.mark.parametrize("spread", [1.0, 6.0])
@pytest.mark.parametrize("B,Hq,Hkv,Nq,Nk,causal,bf16", CASES)
def test_row_sums(device, B, Hq, Hkv, Nq, Nk, causal, bf16, spread):
    print(f"[rowsum] {(B, Hq, Hkv, Nq, Nk, causal, bf16, spread)}", flush=True)
    dt = torch.bfloat16 if bf16 else torch.float16
    g = torch.Generator("cuda").manual_seed(Nq + Nk)
    q = (spread * torch.randn(B, Hq, Nq, 64, device=device, generator=g)).to(dt)
    k, v = (torch.randn(B, Hkv, Nk, 64, device=device, generator=g).to(dt) for _ in range(2))
    o, lse = flash_attention_forward_ex(q, k, v, causal=causal, return_lse=True)
    ao, ro, al = (4e-3, 1.6e-2, math.log1p(2 ** -8)) if bf16 else (2e-3, 1e-2, math.log1p(2 ** -11))
    for b, h in {(0, 0), (B - 1, Hq - 1), (B // 2, Hq // 2)}:
        kv = h // (Hq // Hkv)
        s = q[b, h].double() @ k[b, kv].double().t() / 8.0
        if causal:
            s.masked_fill_(torch.ones(Nq, Nk, dtype=torch.bool, device=device).triu_(1), -math.inf)
        want_l = torch.logsumexp(s, -1)
        want = torch.softmax(s, -1) @ v[b, kv].double()
        assert ((lse[b, h].double() - want_l).abs() <= al + 1e-5 * (1 + want_l.abs())).all()
        err = (o[b, h].double() - want).abs() - ro * want.abs()
        # bfloat16 rows of peaked weights: each P and the row sum round to 8
        # bits, 2^-8 (sum P |V| + 2 |O|) to first order
        bound = ao if not bf16 else ao + 2 ** -8 * (torch.softmax(s, -1) @ v[b, kv].double().abs())
        assert (err <= bound).all(), float(err.max())
