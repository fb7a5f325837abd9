"""Tile shapes and spans of an ensemble's sweep launches come from all of its cases: the
order of the cases does not matter, a shape that the caller has chosen stays, and every
case keeps the bits it has alone (where its own small launch spreads its cells)."""
import itertools

import numpy as np
import pytest

import xfluids_amd as xf
from parity import announce

pytestmark = pytest.mark.gpu

# a case whose own launch takes the 8 x 32 tiles in y, and larger ones
SIZES = [(64, 7), (130, 129), (128, 65)]


def contexts(case, sizes):
    out = []
    for n, m in sizes:
        s = xf.Setup(xf.case_path(case), nx=n, ny=m)
        c = s.context()
        c.upload(*s.initial(case, seed=n))
        c.initialize()
        out.append(c)
    return out


@pytest.mark.parametrize("case", ["isentropic-vortex", "shock-bubble"])
def test_order_does_not_matter(case):
    announce("ensemble shapes " + case)
    alone = {}
    for c, size in zip(contexts(case, SIZES), SIZES):
        shape = c.tile_shape()
        assert (shape[1] == 2) == (size == SIZES[0])
        c.steps(3)
        alone[size] = c.download()[0]
        c.close()
    shapes = set()
    for sizes in itertools.permutations(SIZES):
        # four times, for launches of more than two blocks per CU
        each = contexts(case, sizes * 4)
        ens = xf.Ensemble(each)
        shapes.add(tuple(ens.tile_shape()))
        ens.steps(3)
        ens.synchronize()
        for c, size in zip(each, sizes * 4):
            assert np.array_equal(c.download()[0].view(np.uint64), alone[size].view(np.uint64))
        ens.close()
        for c in each:
            c.close()
    assert len(shapes) == 1 and shapes.pop()[1] == 0


@pytest.mark.parametrize("tuned", [False, True])
def test_chosen_shape_stays(tuned):
    announce("ensemble shapes chosen, tuned=%s" % tuned)
    each = contexts("isentropic-vortex", SIZES)
    if tuned:
        chosen, _ = each[0].autotune(2)
    else:
        chosen = each[0].tile_shape()
        chosen[:2] = 0, 1
        each[0].set_tile_shape(0, 0)
        each[0].set_tile_shape(1, 1)
    ens = xf.Ensemble(each)
    assert np.array_equal(ens.tile_shape()[:2], chosen[:2])
    ens.close()
    for c in each:
        c.close()
