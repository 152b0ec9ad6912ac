"""How many splits decode and small-launch calls run as, seen through the workspace
they ask for (no device needed): one split while the range is short, and no
length at which the next longer one falls to a fraction of the splits."""
import ctypes
import os

import pytest
import test_gpu_split_merge
import test_gpu_split_nonfinite

from capi_types import LIB, Params


def size(B, Hq, Hkv, Nq, Nk, D, causal=0):
    if not os.path.exists(LIB):
        pytest.fail(f"{LIB} not built: run __graft_entry__.build()")
    lib = ctypes.CDLL(LIB)
    lib.fa_sm75_workspace_size.restype = ctypes.c_int64
    p = Params()
    p.q = p.k = p.v = p.o = 0x10000
    p.batch, p.heads_q, p.heads_kv, p.seq_len, p.seq_len_kv, p.head_dim = B, Hq, Hkv, Nq, Nk, D
    lib.fa_sm75_set_contiguous_strides(ctypes.byref(p))
    p.scale, p.causal = 0.125, causal
    return lib.fa_sm75_workspace_size(ctypes.byref(p))


@pytest.mark.parametrize("call,tiles", [
    ((1, 32, 8, 1), {128: 15, 64: 20}), ((16, 32, 8, 1), {128: 15, 64: 28}),
    ((1, 8, 8, 448), {128: 28, 64: 64}),  # row blocks; at 64, two splits are not worth it
    ((1, 1, 1, 448), {128: 28, 64: 36}),
])
@pytest.mark.parametrize("D", [64, 128])
def test_short_ranges_are_one_split(call, tiles, D):
    assert size(*call, 32 * tiles[D], D) == 0
    assert size(*call, 32 * tiles[D] + 33, D) > 0


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,Hq,Hkv,Nq", [(1, 14, 2, 1), (1, 8, 8, 1), (4, 14, 2, 1), (1, 32, 8, 1),
                                         (3, 16, 4, 1), (1, 1, 1, 1), (1, 1, 1, 200)])
def test_no_cliff_in_the_range(B, Hq, Hkv, Nq, D):
    sizes = [size(B, Hq, Hkv, Nq, 32 * t, D) for t in range(1, 400)]
    first = next(i for i, s in enumerate(sizes) if s)
    assert all(sizes[first:])
    # Equal splits of whole tiles: one tile more can take a fifth of them.
    assert all(b >= 0.75 * a for a, b in zip(sizes[first:], sizes[first + 1:]))


def merged_by(B, Hq, Hkv, Nq, Nk, D, causal=0):
    """"kernel" (a mark per workgroup in the workspace), "combine", or None: one split."""
    s = size(B, Hq, Hkv, Nq, Nk, D, causal)
    rows = Hq // Hkv * Nq
    units = B * Hkv * ((rows + 31) // 32)
    record = units * min(rows, 32) * (D + 2) * 4
    assert s % record == 0 or s % (record + 8 * units) == 0
    return None if s == 0 else "combine" if s % record == 0 else "kernel"


def test_the_merge_tests_take_the_routes_they_name():
    K, C = "kernel", "combine"
    assert [merged_by(*c[:7]) for c in test_gpu_split_merge.CASES] == (
        [K] * 7 + [None, K, C, C, K, K])
    assert [merged_by(*c) for c in test_gpu_split_nonfinite.CASES] == [K] * 4 + [C] * 5 + [None]
