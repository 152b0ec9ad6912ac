"""Generated-code check (CPU only): no kernel of the library shifts a 64-bit value
by a lane's amount held in the last vector register of its allocation.

A masked dQ instance that held 1 << k in this form used P of hidden keys now and
then, and shifting the two 32-bit halves of the mask word apart ended it.  Why was
not shown: such a shift reads its amount as a register pair, and with the amount in
the last register the pair ends outside the wave's registers.  This keeps the form
out of every kernel, masked or not."""
import re

from built_code import kernels

SHIFT = re.compile(r"(v_lshlrev_b64|v_lshrrev_b64|v_ashrrev_i64)\S*\s+v\[\d+:\d+\], v(\d+),")


def last_register_shifts(vgprs, lines):
    # Registers are allocated by eights, those before accumulation ones by fours.
    last = {(vgprs + n - 1) // n * n - 1 for n in (4, 8)}
    return [s for s in lines if (m := SHIFT.match(s)) and int(m.group(2)) in last]


def test_the_check_finds_such_a_shift():
    lines = ["v_lshlrev_b64 v[2:3], v255, 1", "v_lshrrev_b64 v[2:3], v254, v[4:5]", "s_endpgm"]
    assert last_register_shifts(256, lines) == lines[:1]
    assert last_register_shifts(253, lines) == lines[:1]
    assert last_register_shifts(240, lines) == []


def test_no_shift_by_the_last_register():
    seen = 0
    for name, vgprs, lines in kernels():
        found = last_register_shifts(vgprs, lines)
        assert not found, (name, vgprs, found)
        assert lines[0] != "" and vgprs > 0
        seen += 1
    assert seen > 200
