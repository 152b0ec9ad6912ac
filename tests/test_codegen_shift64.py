"""Generated-code check (CPU only): no masked kernel shifts a 64-bit value by a
lane's amount held in the last vector register of its allocation.

Such a shift reads its amount as a register pair; with the amount in the last
register the pair ends outside the wave's registers and the shift returned
another amount's result now and then (a masked dQ instance that held 1 << k in
this form used P of hidden keys).  The kernels shift the two 32-bit halves of a
mask word apart instead; these are the instances with the most registers."""
import os
import re
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(REPO, "flash-attention-sm75-register-fused_amd"))
import build_native  # noqa: E402

HIPCC = os.path.join(build_native.ROCM, "bin", "hipcc")
SOURCES = ["fa_bwd_d64_mask.hip", "fa_bwd_d128_mask.hip", "fa_fwd_d128_mask.hip",
           "fa_fwd_d128_mask_w8.hip"]
SHIFT = re.compile(r"\s(v_lshlrev_b64|v_lshrrev_b64|v_ashrrev_i64)\S*\s+v\[\d+:\d+\], v(\d+),")


def last_register_shifts(asm):
    found = []
    for part in re.split(r"\n(?=_ZN2fa\S+:)", asm)[1:]:
        used = re.search(r"; NumVgprs: (\d+)", part)
        if used is None:
            continue
        last = (int(used.group(1)) + 7) // 8 * 8 - 1  # registers are allocated by eights
        body = part[:part.index(".Lfunc_end")]
        found += [(part[:part.index(":")], m.group(0).strip()) for m in SHIFT.finditer(body)
                  if int(m.group(2)) == last]
    return found


def test_the_check_finds_such_a_shift():
    asm = ("x\n_ZN2fa1kE:\n\tv_lshlrev_b64 v[2:3], v255, 1\n\tv_lshlrev_b64 v[2:3], v254, 1\n"
           ".Lfunc_end0:\n; NumVgprs: 256\n")
    assert last_register_shifts(asm) == [("_ZN2fa1kE", "v_lshlrev_b64 v[2:3], v255,")]


def test_no_shift_by_the_last_register():
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")

    def compile_one(src):
        r = subprocess.run([HIPCC, *build_native.HIPCC_FLAGS, f"-I{build_native.INCLUDE}",
                            f"-I{build_native.CSRC}", "--cuda-device-only", "-S",
                            os.path.join(build_native.CSRC, src), "-o", "-"],
                           capture_output=True, text=True, timeout=900)
        assert r.returncode == 0, r.stderr[-2000:]
        assert "; NumVgprs:" in r.stdout
        return last_register_shifts(r.stdout)

    with ThreadPoolExecutor(4) as pool:
        for src, found in zip(SOURCES, pool.map(compile_one, SOURCES)):
            assert not found, (src, found)
