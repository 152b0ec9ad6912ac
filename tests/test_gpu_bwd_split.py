"""The dK/dV key blocks split over several workgroups (fp32 partials, then a
merge): shapes at the edges of the split against the float64 closed form, the
unsplit kernel and itself.  The plan's own rules are checked on the CPU
(test_bwd_split_plan.py).

Against the unsplit kernel (a workspace without room for the partials) the
two sum the same fp32 products in another grouping, so before the final
rounding they differ by a few fp32 ulps of the sums' terms; after it by at
most one ulp of the element type where a value sits at a rounding boundary:
|x - y| <= 2^-10 |y| (binary16, 2^-7 bfloat16) + 1e-5 max|y| for the terms
that cancel.  dQ does not depend on the split: equal bits."""
import ctypes

import numpy as np
import pytest
import torch

from capi_types import LIB, BwdParams
from flash_attention_sm75 import flash_attention_forward_ex
from oracle import attention_ref as ref

pytestmark = pytest.mark.gpu

CASES = [
    # B, Hq, Hkv, Nq, Nk, D, causal, bf16, mask
    (1, 2, 1, 1024, 100, 128, 0, False, None),     # one ragged key block, many pieces
    (1, 14, 2, 512, 512, 64, 1, True, None),       # causal: pieces of unequal blocks
    (1, 8, 2, 1000, 300, 64, 2, False, None),      # rows that see no key
    (2, 6, 2, 500, 200, 128, 1, True, None),       # top-left, Nq > Nk, ragged rows and keys
    (1, 3, 1, 700, 257, 64, 1, False, None),       # group of 3, one key in the last block
    (1, 8, 1, 300, 900, 128, 1, False, None),      # keys no query sees: empty last blocks
    (2, 4, 1, 640, 640, 64, 0, True, "padded"),    # mask ranges cut the steps of pieces
    (1, 8, 2, 520, 520, 128, 0, False, "heads"),
    (1, 8, 2, 600, 600, 64, 1, False, "heads"),    # both, and rows that see nothing
]


def make_mask(kind, B, Hq, N, seed):
    i = torch.arange(N)
    if kind == "padded":
        m = (i[None, :] <= i[:, None])[None, None].expand(B, 1, N, N).clone()
        for b in range(B):
            m[b, :, :, : (b * N) // (2 * B)] = False
        return m
    g = torch.Generator("cpu").manual_seed(seed)
    lo = torch.randint(0, N, (B, Hq, N, 1), generator=g)
    w = torch.randint(0, N // 2, (B, Hq, N, 1), generator=g)  # 0: the row sees nothing
    return (i >= lo) & (i < lo + w)


@pytest.mark.parametrize("B,Hq,Hkv,Nq,Nk,D,causal,bf16,mask", CASES)
def test_split_matches_unsplit_and_oracle(device, B, Hq, Hkv, Nq, Nk, D, causal, bf16, mask):
    print(f"[bwd split] {(B, Hq, Hkv, Nq, Nk, D, causal, bf16, mask)}", flush=True)
    lib = ctypes.CDLL(LIB)
    lib.fa_sm75_backward_workspace_size.restype = ctypes.c_int64
    lib.fa_sm75_last_error.restype = ctypes.c_char_p
    pk = lib.fa_sm75_pack_mask_ranges
    pk.argtypes = [ctypes.c_void_p] + [ctypes.c_int64] * 8 + [ctypes.c_void_p] * 3
    dt = torch.bfloat16 if bf16 else torch.float16
    g = torch.Generator("cpu").manual_seed(Nq + Nk + D)
    q, do = (torch.randn(B, Hq, Nq, D, generator=g).to(dt) for _ in range(2))
    k, v = (torch.randn(B, Hkv, Nk, D, generator=g).to(dt) for _ in range(2))
    m = make_mask(mask, B, Hq, Nq, Nk) if mask else None
    qd, kd, vd, dod = (t.to(device) for t in (q, k, v, do))
    md = m.to(device) if mask else None
    o, lse = flash_attention_forward_ex(qd, kd, vd, causal={0: False, 1: True, 2: "bottom_right"}[causal],
                                        attn_mask=md, return_lse=True)
    stream = torch.cuda.current_stream().cuda_stream
    if mask:
        mh, words = m.size(1), (Nk + 63) // 64
        bits = torch.empty(B, mh, Nq, words, dtype=torch.int64, device=device)
        rng = torch.empty(B, mh, Nq, 2, dtype=torch.int32, device=device)
        st = md.stride()
        assert pk(md.data_ptr(), B, mh, Nq, Nk, st[0], st[1] if mh > 1 else 0, st[2], st[3],
                  bits.data_ptr(), rng.data_ptr(), stream) == 0

    def run(split, ranges=True):
        dq, dk, dv = torch.empty_like(qd), torch.empty_like(kd), torch.empty_like(vd)
        p = BwdParams()
        p.q, p.k, p.v, p.o, p.dout, p.lse, p.dq, p.dk, p.dv = (
            t.data_ptr() for t in (qd, kd, vd, o, dod, lse, dq, dk, dv))
        p.batch, p.heads_q, p.heads_kv, p.seq_len, p.seq_len_kv, p.head_dim = B, Hq, Hkv, Nq, Nk, D
        lib.fa_sm75_set_contiguous_bwd_strides(ctypes.byref(p))
        p.scale, p.dtype, p.stream, p.causal = D ** -0.5, 1 if bf16 else 0, stream, causal
        if mask:
            p.mask_bits, p.mask_stride_b, p.mask_stride_q = bits.data_ptr(), mh * Nq * words, words
            p.mask_stride_h = Nq * words if mh > 1 else 0
            if ranges:
                p.mask_ranges, p.mask_ranges_stride_b = rng.data_ptr(), mh * Nq
                p.mask_ranges_stride_h, p.mask_ranges_stride_q = (Nq if mh > 1 else 0), 1
        need = B * Hq * ((Nq + 63) // 64) * 520
        n = lib.fa_sm75_backward_workspace_size(ctypes.byref(p))
        assert n > need  # the plan splits this shape
        if not split:
            n = need
        # The partials' room holds NaN: every one read has been written.
        ws = torch.full(((n + 3) // 4,), float("nan"), device=device)
        p.workspace, p.workspace_bytes = ws.data_ptr(), n
        assert lib.fa_sm75_backward(ctypes.byref(p)) == 0, lib.fa_sm75_last_error()
        torch.cuda.synchronize()
        return dq, dk, dv

    got, again, plain = run(True), run(True), run(False)
    for x, y in zip(got, again):
        assert torch.equal(x, y)
    if mask:
        for x, y in zip(got, run(True, ranges=False)):
            assert torch.equal(x, y)
    assert torch.equal(got[0], plain[0])
    ulp = 2.0 ** -7 if bf16 else 2.0 ** -10
    for x, y in zip(got[1:], plain[1:]):
        x, y = x.double(), y.double()
        assert ((x - y).abs() <= ulp * y.abs() + 1e-5 * y.abs().max()).all()
    npf = lambda t: t.float().cpu().numpy()
    wants = ref.attention_backward_f64(npf(q), npf(k), npf(v), npf(do), causal=causal,
                                       attn_mask=m.numpy() if mask else None, delta_from_o=npf(o))
    ba, br = (1e-2, 4e-2) if bf16 else (2e-3, 1e-2)  # test_gpu_backward.py's bar
    for name, x, w in zip(("dQ", "dK", "dV"), got, wants):
        sc = max(float(np.abs(w).max()), 1e-2)
        worst = float((np.abs(npf(x) - w) / (ba * sc + br * np.abs(w))).max())
        print(f"  {name}: worst/bar={worst:.3f}", flush=True)
        assert worst <= 1.0, (name, worst)
