"""Sweep tiles whose cells do not fill them: grids one to a few cells over a
multiple of the tile in every direction (the remainder is spread evenly over the
tiles there, and on every small grid), with each tile shape, bit for bit against
the oracle."""
import numpy as np
import pytest

import xfluids_amd as xf
from parity import announce, oracle_for

pytestmark = pytest.mark.gpu

# 63 / 31 cells along x, 15 / 31 / 7 along y and z fill a tile; 16, 8 or 32 columns
GRIDS = [
    ("isentropic-vortex", "isentropic-vortex", dict(nx=64, ny=65)),
    ("isentropic-vortex", "isentropic-vortex", dict(nx=33, ny=16)),
    ("shock-bubble", "shock-bubble", dict(nx=94, ny=34)),
    ("shock-bubble-3d", "shock-bubble", dict(nx=65, ny=16, nz=17)),
    ("mixing-layer", "mixing-layer", dict(nx=33, ny=17, nz=8)),
    # over 512 blocks: only the smallest remainders are spread
    ("shock-bubble", "shock-bubble", dict(nx=316, ny=466)),
    ("reactive-shock-tube", "reactive-shock-tube", dict(nx=127)),
]


@pytest.mark.parametrize("case,workload,size", GRIDS)
def test_remainder_tiles_match_oracle(case, workload, size):
    announce("tile spans %s %s" % (case, size))
    s = xf.Setup(xf.case_path(case), **size)
    U, T = s.initial(workload, seed=4)
    o = oracle_for(s, U, T)
    assert o.initialize() == 0
    assert o.steps(2)[0] == 0
    Uo, To = o.field("U"), o.field("T")
    for shape in (None, 0, 1, 2):
        ctx = s.context()
        if shape is not None:
            for d in range(3):
                ctx.set_tile_shape(d, min(shape, 1) if d == 0 else shape)
        ctx.upload(U, T)
        ctx.initialize()
        ctx.steps(2)
        Ug, Tg = ctx.download()
        ctx.close()
        assert np.array_equal(Uo.view(np.uint64), Ug.view(np.uint64)), shape
        assert np.array_equal(To.view(np.uint64), Tg.view(np.uint64)), shape
