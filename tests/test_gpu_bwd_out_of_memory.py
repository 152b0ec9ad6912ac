"""A backward call whose split partials do not fit the GPU's memory runs with the
required workspace alone, unsplit.  The allocator's limit stands in for a full
GPU.  dQ does not depend on the split (equal bits); dK and dV are the unsplit
kernel's, |x - y| <= 2^-7 |y| + 1e-5 max|y| from the split's (test_gpu_bwd_split.py)."""
import pytest
import torch

from flash_attention_sm75 import flash_attention_backward, flash_attention_forward_ex

pytestmark = pytest.mark.gpu

MB = 1 << 20


@pytest.mark.parametrize("causal", [True, "bottom_right"])
def test_partials_that_do_not_fit(device, causal):
    # dQ, dK and dV: 8 + 2 + 2 MB; workspace 31.7 MB with the partials, 0.3 without.
    B, Hq, Hkv, N, D = 1, 32, 8, 1024, 128
    q, do = (torch.randn(B, Hq, N, D, device=device, dtype=torch.bfloat16) for _ in range(2))
    k, v = (torch.randn(B, Hkv, N, D, device=device, dtype=torch.bfloat16) for _ in range(2))
    o, lse = flash_attention_forward_ex(q, k, v, causal=causal, return_lse=True)
    want = flash_attention_backward(do, q, k, v, o, lse, causal=causal)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    hogs, held = [], torch.cuda.memory_reserved(device)
    while torch.cuda.memory_reserved(device) == held:  # no free block takes the partials
        hogs.append(torch.empty(16 * MB, dtype=torch.uint8, device=device))
    del hogs[-1]
    torch.cuda.empty_cache()
    ooms = torch.cuda.memory_stats(device)["num_ooms"]
    total = torch.cuda.get_device_properties(device).total_memory
    # Room for the three gradients in the allocator's 20 MB segments, one or two.
    room = torch.cuda.memory_reserved(device) + 30 * MB
    torch.cuda.set_per_process_memory_fraction(room / total, device)
    try:
        got = flash_attention_backward(do, q, k, v, o, lse, causal=causal)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, device)
    assert torch.cuda.memory_stats(device)["num_ooms"] > ooms  # the partials were refused
    assert torch.equal(got[0], want[0])
    for x, y in zip(got[1:], want[1:]):
        x, y = x.double(), y.double()
        assert ((x - y).abs() <= 2.0 ** -7 * y.abs() + 1e-5 * y.abs().max()).all()
