"""CPU model of the reducing hops' launch (hop_kernel, launch_hop_prec in k_hop.inc): a launch
that sums |out|^2 takes one right-hand side per wave whatever its shape asks for, and a wave
covers one aligned 64-site chunk, so lane 0 of each wave writes that chunk's partial and
every partial is written once."""
import itertools

import pytest

from test_launch_map import SHAPES, remap_block


def partials(vh, nrhs, block, rb, rpw, rpt, gm, xcd, spt):
    rpw = 1  # b.partials: one right-hand side per wave
    sg = block // rb
    ngroups = -(-nrhs // (rb * rpw * rpt))
    sb = sg
    nsb = -(-vh // sb)
    nbx = -(-nsb // spt)
    grid = nbx * ngroups
    written = {}
    for bid, wave, it in itertools.product(range(grid), range(block // 64), range(spt)):
        lb = remap_block(bid, grid, xcd)
        bx0, grp = (lb % nbx, lb // nbx) if gm else (lb // ngroups, lb % ngroups)
        bx = bx0 + it * nbx
        if bx >= nsb:
            continue
        rl, tg = wave * 64 // sg, wave * 64 % sg
        r0 = (grp * rb + rl) * rpt
        l0 = bx * sb + tg  # lane 0
        if l0 >= vh:
            continue
        assert l0 % 64 == 0
        for r in range(r0, min(r0 + rpt, nrhs)):
            assert (r, l0 // 64) not in written
            written[r, l0 // 64] = True
    return written


@pytest.mark.parametrize("vh", [8, 48, 1000, 2048])
@pytest.mark.parametrize("nrhs", [1, 2, 5, 12, 16])
@pytest.mark.parametrize("shape", SHAPES)
def test_each_chunk_partial_written_once(vh, nrhs, shape):
    block, rb, rpw, rpt, spt = shape
    for gm, xcd in itertools.product((0, 1), (0, 1)):
        w = partials(vh, nrhs, block, rb, rpw, rpt, gm, xcd, spt)
        assert sorted(w) == [(r, c) for r in range(nrhs) for c in range(-(-vh // 64))]
