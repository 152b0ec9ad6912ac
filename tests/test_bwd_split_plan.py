"""Which backward calls split their dK/dV key blocks, seen through the
workspace size (no device needed): the required part alone where the launch
fills the GPU or the steps are few, bounded partials elsewhere."""
import ctypes
import os
import random

import pytest

from capi_types import LIB, BwdParams


def partials(B, Hq, Hkv, Nq, Nk, D, causal, mask=False):
    """(bytes beyond the required part, bytes of one piece's partials)"""
    if not os.path.exists(LIB):
        pytest.fail(f"{LIB} not built: run __graft_entry__.build()")
    f = ctypes.CDLL(LIB).fa_sm75_backward_workspace_size
    f.restype = ctypes.c_int64
    p = BwdParams()
    p.batch, p.heads_q, p.heads_kv, p.seq_len, p.seq_len_kv, p.head_dim, p.causal = (
        B, Hq, Hkv, Nq, Nk, D, causal)
    p.mask_bits = 256 if mask else None  # only tested for null
    need = B * Hq * ((Nq + 63) // 64) * 520
    extra = f(ctypes.byref(p)) - need
    assert extra >= 0
    return (extra - (-need) % 256 if extra else 0), 2 * 128 * D * 4


@pytest.mark.parametrize("call,split", [
    ((4, 14, 2, 2048, 2048, 64, 1), True), ((1, 14, 2, 4096, 4096, 64, 1), True),
    ((1, 32, 8, 1024, 1024, 128, 1), True), ((1, 2, 1, 1024, 100, 128, 0), True),
    ((1, 32, 8, 8192, 8192, 128, 1), False), ((4, 8, 8, 2048, 2048, 64, 1), False),
    ((4, 12, 12, 1024, 1024, 64, 0), False), ((2, 8, 2, 100, 100, 128, 0), False),
    ((1, 64, 1, 64, 40000, 64, 0), False),          # more key blocks than the tables hold
    ((1, 12, 12, 1114, 1114, 64, 0), False),        # saves less than the merge launch costs
    ((1, 8, 8, 6016, 6016, 128, 0), True),          # two whole rounds of equal blocks ...
    ((1, 8, 8, 6016, 6016, 128, 0, True), False),   # ... which a mask makes uneven
    ((4, 16, 4, 448, 448, 128, 0, True), True),
])
def test_which_calls_split(call, split):
    assert (partials(*call)[0] > 0) == split


def test_partials_are_whole_pieces_and_bounded():
    rng = random.Random(7)
    seen = 0
    for _ in range(4000):
        hkv, group = rng.choice([1, 2, 3, 8, 32]), rng.choice([1, 2, 7, 8, 64])
        nq, nk = (int(2 ** rng.uniform(0, 16)) for _ in range(2))
        extra, piece = partials(rng.choice([1, 2, 5, 16]), hkv * group, hkv, nq, nk,
                                rng.choice([64, 128]), rng.choice([0, 1, 2]))
        assert extra % piece == 0 and extra // piece <= 4 * 256
        seen += extra > 0
    assert seen > 100
