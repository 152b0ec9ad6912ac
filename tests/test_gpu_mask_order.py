"""Padded batches whose eight units (batch x KV heads) go out as one sequence
over the XCDs instead of one unit per XCD (plan_xcds), on both sides of the
one-workgroup-per-CU rule: outputs and gradients of every sequence and head
against float64 on the device, rows that see no key included.  The order of
the workgroups is all that changes, so a block left out or done for the wrong
unit shows as a wrong or unwritten slice.

Bars: O |x - o| <= 2e-3 + 1e-2 |o|; gradients 2e-3 max|R| + 1e-2 |R|
(test_gpu_backward.py's)."""
import pytest
import torch

from flash_attention_sm75 import flash_attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,N,D", [(4, 8, 2, 1100, 64),   # 288 blocks
                                          (4, 8, 2, 900, 128),   # 256 blocks: unit by unit
                                          (8, 7, 1, 700, 128),   # 336 blocks, a group of 7
                                          (8, 8, 1, 300, 64),    # 192 blocks
                                          (8, 10, 1, 500, 64)])  # 320 blocks, short rows: unit by unit
def test_padded_batch_order(device, B, Hq, Hkv, N, D):
    print(f"[mask order] {(B, Hq, Hkv, N, D)}", flush=True)
    g = torch.Generator("cuda").manual_seed(N)
    q, do = (torch.randn(B, Hq, N, D, device=device, generator=g).half() for _ in range(2))
    k, v = (torch.randn(B, Hkv, N, D, device=device, generator=g).half() for _ in range(2))
    i = torch.arange(N, device=device)
    pad = torch.arange(B, device=device)[:, None, None] * (N // (B + 1))
    mask = ((i[None, :] <= i[:, None])[None] & (i[None, None, :] >= pad))[:, None]
    leaves = [t.clone().requires_grad_() for t in (q, k, v)]
    o = flash_attention(*leaves, attn_mask=mask)
    grads = torch.autograd.grad(o, leaves, do)
    want = [torch.zeros(t.shape, dtype=torch.float64, device=device) for t in (q, q, k, v)]
    for b in range(B):
        for h in range(Hq):
            kv = h // (Hq // Hkv)
            qd, kd, vd, dd = (t.double() for t in (q[b, h], k[b, kv], v[b, kv], do[b, h]))
            s = (qd @ kd.t() * D ** -0.5).masked_fill_(~mask[b, 0], float("-inf"))
            p = torch.softmax(s, -1).nan_to_num_(0.0)  # rows of padding see no key
            want[0][b, h] = p @ vd
            ds = p * (dd @ vd.t() - (dd * want[0][b, h]).sum(-1, keepdim=True)) * D ** -0.5
            want[1][b, h] = ds @ kd
            want[2][b, kv] += ds.t() @ qd
            want[3][b, kv] += p.t() @ dd
    assert ((o.double() - want[0]).abs() <= 2e-3 + 1e-2 * want[0].abs()).all()
    for name, x, w in zip(("dQ", "dK", "dV"), grads, want[1:]):
        worst = ((x.double() - w).abs() / (2e-3 * w.abs().max() + 1e-2 * w.abs())).max().item()
        print(f"  {name}: worst/bar={worst:.3f}", flush=True)
        assert worst <= 1.0, name
