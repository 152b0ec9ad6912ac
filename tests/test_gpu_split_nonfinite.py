"""A decode or small-launch query that holds a NaN gives NaN, and LSE NaN, however
its keys are split; a query that sees no key gives zeros and -inf, and the other
queries' bits do not change.  One case for each way that splits merge: in the
split-K kernel (one and several items per thread), by fa_decode_combine and by
its wide form."""
import math

import pytest
import torch

from flash_attention_sm75 import flash_attention_forward_ex

pytestmark = pytest.mark.gpu

CASES = [
    # B, Hq, Hkv, Nq, Nk, D
    (1, 14, 2, 1, 4097, 64),     # in the kernel, groups of splits
    (2, 8, 1, 1, 2000, 128),     # in the kernel, one item per thread
    (1, 9, 1, 1, 1100, 128),     # in the kernel, some threads with two
    (1, 4, 4, 777, 1100, 128),   # in the kernel, row blocks: four each
    (1, 2, 2, 200, 1900, 64),    # row blocks, combine
    (2, 8, 8, 1, 4096, 64),      # combine
    (1, 32, 8, 8, 2048, 128),    # combine
    (1, 1, 1, 1, 65536, 64),     # wide combine
    (1, 2, 1, 2, 33000, 128),    # wide combine
    (1, 4, 2, 1, 300, 64),       # one split
]


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,Nq,Nk,D", CASES)
def test_nan_queries_and_queries_without_keys(device, B, Hq, Hkv, Nq, Nk, D, bf16):
    print(f"[split nonfinite] {(B, Hq, Hkv, Nq, Nk, D, bf16)}", flush=True)
    dt = torch.bfloat16 if bf16 else torch.float16
    g = torch.Generator("cuda").manual_seed(Nq + Nk)
    q = torch.randn(B, Hq, Nq, D, device=device, generator=g).to(dt)
    k, v = (torch.randn(B, Hkv, Nk, D, device=device, generator=g).to(dt) for _ in range(2))
    m = torch.ones(B, Hq, Nq, Nk, dtype=torch.bool, device=device)
    m[B - 1, Hq - 1, Nq - 1] = False
    clean = q.clone()
    q[0, 0, 0, 5] = math.nan
    for mask in (None, m):
        want, want_l = flash_attention_forward_ex(clean, k, v, attn_mask=mask, return_lse=True)
        got, got_l = flash_attention_forward_ex(q, k, v, attn_mask=mask, return_lse=True)
        nan = torch.zeros(B, Hq, Nq, dtype=torch.bool, device=device)
        nan[0, 0, 0] = mask is None or (B, Hq, Nq) != (1, 1, 1)  # there the mask hides all
        assert got[nan].isnan().all() and got_l[nan].isnan().all()
        assert torch.equal(got[~nan], want[~nan]) and torch.equal(got_l[~nan], want_l[~nan])
        if mask is not None:
            assert (got[B - 1, Hq - 1, Nq - 1] == 0).all()
            assert got_l[B - 1, Hq - 1, Nq - 1] == -math.inf
