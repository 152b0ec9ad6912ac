"""Split-K calls with less workspace than they ask for: a call takes as many
splits as there is room for (two or more), merges them with the combine kernel
where the marks of the in-kernel merge do not fit, and writes nothing past the
bytes it was given.  Every size against the float64 oracle.

Bars: O |x - o64| <= 2e-3 + 1e-2 |o64| (binary16; test_gpu_decode.py's), LSE
1e-3 + 1e-4 |lse|."""
import ctypes

import numpy as np
import pytest
import torch

from capi_types import LIB, Params
from oracle import attention_ref as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,Nq,Nk,D,causal", [
    (1, 14, 2, 1, 2048, 64, 0),     # 7 rows a unit
    (2, 8, 8, 1, 3000, 128, 0),
    (1, 8, 2, 3, 1500, 64, 2),
    (1, 2, 2, 100, 2600, 128, 0),   # row blocks
])
def test_smaller_workspaces(device, B, Hq, Hkv, Nq, Nk, D, causal):
    print(f"[decode workspace] {(B, Hq, Hkv, Nq, Nk, D, causal)}", flush=True)
    lib = ctypes.CDLL(LIB)
    lib.fa_sm75_workspace_size.restype = ctypes.c_int64
    lib.fa_sm75_last_error.restype = ctypes.c_char_p
    g = torch.Generator("cpu").manual_seed(Nk)
    q, k, v = (torch.randn(B, h, n, D, generator=g).half() for h, n in ((Hq, Nq), (Hkv, Nk), (Hkv, Nk)))
    qd, kd, vd = (t.to(device) for t in (q, k, v))
    npf = lambda t: t.float().cpu().numpy()
    want = ref.attention_f64(npf(q), npf(k), npf(v), causal=causal)
    want_l = ref.attention_lse(npf(q), npf(k), causal=causal)
    p = Params()
    o = torch.empty_like(qd)
    lse = torch.empty(B, Hq, Nq, dtype=torch.float32, device=device)
    p.q, p.k, p.v, p.o, p.lse = (t.data_ptr() for t in (qd, kd, vd, o, lse))
    p.batch, p.heads_q, p.heads_kv, p.seq_len, p.seq_len_kv, p.head_dim = B, Hq, Hkv, Nq, Nk, D
    lib.fa_sm75_set_contiguous_strides(ctypes.byref(p))
    p.scale, p.causal, p.stream = D ** -0.5, causal, torch.cuda.current_stream().cuda_stream
    need = lib.fa_sm75_workspace_size(ctypes.byref(p))
    rows = Hq // Hkv * Nq
    blocks = -(-rows // 32)
    units = B * Hkv * blocks
    filled = rows / (blocks * min(rows, 32))  # of a record: the last block may be ragged
    record = units * min(rows, 32) * (D + 2) * 4  # one split's partials
    splits = need // record
    assert splits >= 4
    pattern = 0x5A
    for size in (need, need - 1, splits * record, splits * record - 1, 3 * record, 2 * record,
                 2 * record - 1, 0):
        ws = torch.full((need + 64,), pattern, dtype=torch.uint8, device=device)
        o.fill_(float("nan"))
        lse.fill_(float("nan"))
        p.workspace, p.workspace_bytes = ws.data_ptr(), size
        assert lib.fa_sm75_forward(ctypes.byref(p)) == 0, lib.fa_sm75_last_error()
        torch.cuda.synchronize()
        assert (ws[size:] == pattern).all(), size
        used = int((ws != pattern).sum())
        print(f"  {size} of {need} bytes: {used} written", flush=True)
        # Values that happen to hold the pattern's bytes are few.
        assert used == 0 if size < 2 * record else used > 0.9 * filled * 2 * record, size
        if size >= splits * record:  # all the splits, whichever way they are merged
            assert used > 0.9 * filled * splits * record, size
        got = npf(o)
        assert (np.abs(got - want) <= 2e-3 + 1e-2 * np.abs(want)).all(), size
        np.testing.assert_allclose(lse.cpu().numpy(), want_l, atol=1e-3, rtol=1e-4)
