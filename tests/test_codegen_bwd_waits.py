"""Generated-code check (CPU only) of the head_dim-64 dQ kernel's prologue: its
first barrier waits for all but the second tile's direct loads.  vmcnt counts in
issue order, so the loads it leaves in flight must be exactly those: were a load of
the first tile among them, or a plain load counted with them that the compiler may
move, other waves could read the first tile before it is there."""
import re

from built_code import kernels

SECOND_TILE = 4  # direct loads a wave issues for a K and a V tile


def test_dq_prologue_leaves_only_the_second_tile_in_flight():
    seen = 0
    for name, _, lines in kernels():
        if "fa_bwd_dq_kernelILi64E" not in name:
            continue
        memory = [i for i, s in enumerate(lines) if re.match(r"(buffer|global|flat|scratch)_", s)]
        direct = [i for i in memory if lines[i].endswith(" lds")]
        barrier = next(i for i in range(direct[0], len(lines)) if lines[i].startswith("s_barrier"))
        before = [i for i in memory if i < barrier]
        assert sum(i < barrier for i in direct) == 2 * SECOND_TILE, name
        assert all(i in direct for i in before[-SECOND_TILE:]), (name, [lines[i] for i in before[-9:]])
        waits = [re.search(r"vmcnt\((\d+)\)", s) for s in lines[before[-1]:barrier]]
        assert [int(m.group(1)) for m in waits if m] == [SECOND_TILE], name
        seen += 1
    assert seen == 8  # causal, mask, element type
