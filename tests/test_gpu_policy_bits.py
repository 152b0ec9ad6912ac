"""The kernels that can be forced for a head_dim-64 call (128-row and 256-row
workgroups, the dynamic schedule) give the same bits, also where a launch fits the
GPU in one round: the way the rows are summed follows from the shape alone."""
import pytest
import torch

import flash_attn_sm75_cuda as _C
from flash_attention_sm75 import flash_attention_forward_ex

pytestmark = pytest.mark.gpu

AUTO, NARROW, WIDE, DYNAMIC = 0, 1, 2, 3


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,Nq,Nk,causal", [
    (2, 8, 8, 1000, 333, False),    # 128 blocks
    (2, 32, 8, 1024, 700, False),   # 512 blocks: the last size of one round
    (1, 57, 19, 1100, 500, False),  # 513 blocks
    (1, 20, 4, 600, 600, True),
])
def test_forced_kernels_agree(device, B, Hq, Hkv, Nq, Nk, causal, bf16):
    print(f"[policy bits] {(B, Hq, Hkv, Nq, Nk, causal, bf16)}", flush=True)
    dt = torch.bfloat16 if bf16 else torch.float16
    g = torch.Generator("cuda").manual_seed(Nq)
    q = torch.randn(B, Hq, Nq, 64, device=device, generator=g).to(dt)
    k, v = (torch.randn(B, Hkv, Nk, 64, device=device, generator=g).to(dt) for _ in range(2))
    outs = []
    for policy in (NARROW, WIDE, DYNAMIC):
        _C.set_kernel_policy(policy)
        try:
            outs.append(flash_attention_forward_ex(q, k, v, causal=causal, return_lse=True))
        finally:
            _C.set_kernel_policy(AUTO)
    for o, lse in outs[1:]:
        assert torch.equal(o, outs[0][0]) and torch.equal(lse, outs[0][1])
