"""The split-K kernel's own merge of a unit's splits (the last workgroup to
finish sums them): shapes at the edges of the merge's work split, against the
float64 oracle and the one-split path, on workspaces that hold anything.

Bars: O |x - o64| <= 2e-3 + 1e-2 |o64| (binary16; test_gpu_decode.py's), LSE
1e-3 + 1e-4 |lse|."""
import ctypes

import numpy as np
import pytest
import torch

from capi_types import LIB, Params
from oracle import attention_ref as ref

pytestmark = pytest.mark.gpu

CASES = [
    # B, Hq, Hkv, Nq, Nk, D, causal, mask: rows per unit x splits
    (1, 1, 1, 1, 1000, 64, 0, False),    # 1 row: 16 merge items, 16 groups
    (1, 7, 1, 1, 4097, 64, 0, False),    # 7 rows: groups that do not fill the workgroup
    (2, 8, 1, 1, 2000, 128, 0, False),   # 8 rows x 128 dims: one item per thread
    (1, 9, 1, 1, 1100, 128, 0, False),   # 9 rows: threads with one item and with two
    (1, 32, 1, 1, 520, 128, 0, False),   # 32 rows: four items per thread
    (1, 1, 1, 1, 9000, 64, 0, False),    # more splits than loads in flight
    (2, 8, 2, 3, 700, 64, 2, False),     # bottom-right
    (1, 4, 4, 4, 1500, 128, 1, False),   # top-left, 4 keys seen: one split, then many keys unseen
    (3, 14, 2, 1, 3000, 64, 0, True),    # key bytes: splits that see no key
    (1, 2, 2, 300, 1100, 128, 2, False), # row blocks merged by the combine kernel
    (1, 1, 1, 200, 2048, 64, 0, False),
    (1, 4, 4, 777, 1100, 128, 0, False), # row blocks merged here, the last one ragged
    (1, 2, 2, 1000, 1500, 64, 2, False),
]


@pytest.fixture(scope="module")
def lib():
    lib = ctypes.CDLL(LIB)
    lib.fa_sm75_workspace_size.restype = ctypes.c_int64
    lib.fa_sm75_last_error.restype = ctypes.c_char_p
    return lib


def make(B, Hq, Hkv, Nq, Nk, D, causal, mask, device, seed):
    g = torch.Generator("cpu").manual_seed(seed)
    t = [torch.randn(B, h, n, D, generator=g).half().to(device)
         for h, n in ((Hq, Nq), (Hkv, Nk), (Hkv, Nk))]
    m = None
    if mask:  # one full sequence, one of a few keys, one with a hole over whole splits
        m = torch.zeros(B, Nk, dtype=torch.bool)
        m[0] = True
        m[1, :5] = True
        m[2, :40] = m[2, -3:] = True
        m = m.to(device)
    return t, m


def params(lib, t, m, o, lse, shape, ws, ws_bytes):
    B, Hq, Hkv, Nq, Nk, D, causal = shape
    p = Params()
    p.q, p.k, p.v, p.o, p.lse = (x.data_ptr() for x in (*t, o, lse))
    p.batch, p.heads_q, p.heads_kv, p.seq_len, p.seq_len_kv, p.head_dim = B, Hq, Hkv, Nq, Nk, D
    lib.fa_sm75_set_contiguous_strides(ctypes.byref(p))
    p.scale, p.causal, p.stream = D ** -0.5, causal, torch.cuda.current_stream().cuda_stream
    if m is not None:
        p.mask_keys, p.mask_keys_stride_b, p.mask_keys_stride_k = m.data_ptr(), Nk, 1
    if ws is not None:
        p.workspace, p.workspace_bytes = ws.data_ptr(), ws_bytes
    return p


def run(lib, t, m, shape, ws=None, ws_bytes=0):
    o = torch.full_like(t[0], float("nan"))
    lse = torch.full(t[0].shape[:3], float("nan"), dtype=torch.float32, device=o.device)
    p = params(lib, t, m, o, lse, shape, ws, ws_bytes)
    assert lib.fa_sm75_forward(ctypes.byref(p)) == 0, lib.fa_sm75_last_error()
    torch.cuda.synchronize()
    return o, lse


@pytest.mark.parametrize("B,Hq,Hkv,Nq,Nk,D,causal,mask", CASES)
def test_merge_matches_oracle(device, lib, B, Hq, Hkv, Nq, Nk, D, causal, mask):
    shape = (B, Hq, Hkv, Nq, Nk, D, causal)
    print(f"[merge] {shape} mask={mask}", flush=True)
    t, m = make(*shape, mask, device, seed=Nk + D)
    need = lib.fa_sm75_workspace_size(ctypes.byref(params(lib, t, m, t[0], t[0], shape, None, 0)))
    if shape != (1, 4, 4, 4, 1500, 128, 1):
        assert need > 0
    ws = torch.full((max(need, 16) // 4 + 1,), float("nan"), device=device)
    o, lse = run(lib, t, m, shape, ws, need)
    npf = lambda x: x.float().cpu().numpy()
    mk = None if m is None else m.cpu().numpy()[:, None, None, :]
    want = ref.attention_f64(npf(t[0]), npf(t[1]), npf(t[2]), causal=causal, attn_mask=mk)
    assert (np.abs(npf(o) - want) <= 2e-3 + 1e-2 * np.abs(want)).all()
    lw = ref.attention_lse(npf(t[0]), npf(t[1]), causal=causal, attn_mask=mk)
    fin = np.isfinite(lw)
    gl = lse.cpu().numpy()
    assert np.array_equal(np.isfinite(gl), fin)
    np.testing.assert_allclose(gl[fin], lw[fin], atol=1e-3, rtol=1e-4)
    # The same workspace again (its marks are the last call's), other inputs in
    # between, and one full of set bits: the same bits.
    t2, _ = make(*shape, mask, device, seed=1)
    run(lib, t2, m, shape, ws, need)
    again = run(lib, t, m, shape, ws, need)
    ws.view(torch.int32).fill_(-1)
    ones = run(lib, t, m, shape, ws, need)
    for x in (again, ones):
        assert torch.equal(x[0], o) and torch.equal(x[1], lse)
    # Without room for the partials: one split, the same values to rounding.
    o1, l1 = run(lib, t, m, shape)
    assert (np.abs(npf(o1) - want) <= 2e-3 + 1e-2 * np.abs(want)).all()


def test_merge_on_many_streams(device, lib):
    """Calls on four streams at once, each with its own workspace, many times
    over: every one the bits of the call alone."""
    shape = (1, 14, 2, 1, 4097, 64, 0)
    streams = [torch.cuda.Stream() for _ in range(4)]
    jobs = []
    for i in range(4):
        t, _ = make(*shape, False, device, seed=i)
        need = lib.fa_sm75_workspace_size(ctypes.byref(params(lib, t, None, t[0], t[0], shape, None, 0)))
        ws = torch.empty(need, dtype=torch.uint8, device=device)
        alone = run(lib, t, None, shape, ws, need)
        jobs.append((t, ws, need, alone))
    outs = []
    for rep in range(25):
        for s, (t, ws, need, _) in zip(streams, jobs):
            s.wait_stream(torch.cuda.current_stream())
            o = torch.empty_like(t[0])
            lse = torch.empty(t[0].shape[:3], dtype=torch.float32, device=device)
            with torch.cuda.stream(s):
                p = params(lib, t, None, o, lse, shape, ws, need)
                assert lib.fa_sm75_forward(ctypes.byref(p)) == 0
            outs.append((o, lse))
    torch.cuda.synchronize()
    for i, (o, lse) in enumerate(outs):
        assert torch.equal(o, jobs[i % 4][3][0]) and torch.equal(lse, jobs[i % 4][3][1]), i


def test_merge_under_capture(device, lib):
    """A captured call replayed on rewritten inputs, with eager calls on the
    same workspace and unrelated work in between: the eager call's bits."""
    shape = (2, 8, 2, 1, 3000, 128, 0)
    t, _ = make(*shape, False, device, seed=0)
    need = lib.fa_sm75_workspace_size(ctypes.byref(params(lib, t, None, t[0], t[0], shape, None, 0)))
    ws = torch.full((need // 4 + 1,), float("nan"), device=device)
    run(lib, t, None, shape, ws, need)
    o = torch.full_like(t[0], float("nan"))
    lse = torch.empty(t[0].shape[:3], dtype=torch.float32, device=device)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        p = params(lib, t, None, o, lse, shape, ws, need)
        assert lib.fa_sm75_forward(ctypes.byref(p)) == 0, lib.fa_sm75_last_error()
    for rep in range(4):
        for x, y in zip(t, make(*shape, False, device, seed=10 + rep)[0]):
            x.copy_(y)
        o.fill_(float("nan"))
        graph.replay()
        torch.randn(1 << 18, device=device).sum()
        if rep % 2:
            graph.replay()
        torch.cuda.synchronize()
        want = run(lib, t, None, shape, ws, need)
        assert torch.equal(o, want[0]) and torch.equal(lse, want[1]), rep
