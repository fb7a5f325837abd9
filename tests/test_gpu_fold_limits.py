"""The grids at which UpdateStates' launch and the fold of its maxima change form, each
side of the limit by the count of its blocks of 256 cells: one block, the 256 blocks that
the readers fold at a time, the 512 up to which they fold for themselves, the 1024 up to
which the states kernel finishes its Newton chains on groups of lanes; bit for bit
against the oracle, and in an ensemble."""
import numpy as np
import pytest

import xfluids_amd as xf
from parity import announce, oracle_for

pytestmark = pytest.mark.gpu

# 8 ghost cells a direction: (nx + 8)(ny + 8) cells
VORTEX, BUBBLE = "isentropic-vortex", "shock-bubble"
GRIDS = [
    (VORTEX, dict(nx=8, ny=8), 1), (VORTEX, dict(nx=248, ny=248), 256), (VORTEX, dict(nx=248, ny=249), 257),
    (VORTEX, dict(nx=504, ny=248), 512), (VORTEX, dict(nx=505, ny=248), 513),
    (BUBBLE, dict(nx=504, ny=248), 512), (BUBBLE, dict(nx=505, ny=248), 513),
    (BUBBLE, dict(nx=1016, ny=248), 1024), (BUBBLE, dict(nx=1017, ny=248), 1025),
    ("reactive-shock-tube", dict(nx=248), 1), ("reactive-shock-tube", dict(nx=249), 2),
]


def blocks(s):
    return (s.desc.ncell + 255) // 256


@pytest.mark.parametrize("case,size,nb", GRIDS)
def test_maxima_and_state_match_oracle(case, size, nb):
    announce("fold limits %s %s" % (case, size))
    s = xf.Setup(xf.case_path(case), **size)
    assert blocks(s) == nb
    U, T = s.initial(case, seed=5)
    o = oracle_for(s, U, T)
    assert o.initialize() == 0
    assert o.steps(2)[0] == 0
    ctx = s.context()
    ctx.upload(U, T)
    ctx.initialize()
    ctx.steps(2)
    Ug, Tg = ctx.download()
    E = s.desc.E
    glf, cfl = ctx.maxima()
    dt = ctx.get_dt()
    again = ctx.maxima()[1]
    ctx.close()
    assert np.array_equal(o.field("eigen_block").reshape(3, -1)[:, :E], glf[:, :E])
    assert np.array_equal(o.field("U").view(np.uint64), Ug.view(np.uint64))
    assert np.array_equal(o.field("T").view(np.uint64), Tg.view(np.uint64))
    assert dt == o.get_dt()
    assert np.array_equal(again, cfl)


@pytest.mark.parametrize("sizes,nb", [((56, 504, 505), (64, 512, 513)), ((56, 504), (64, 512)), ((505,), (513,))])
def test_ensemble_around_the_fold_limit(sizes, nb):
    announce("fold limits ensemble %s" % (sizes,))
    setups = [xf.Setup(xf.case_path(VORTEX), nx=n, ny=248) for n in sizes]
    assert tuple(blocks(s) for s in setups) == nb
    states = [s.initial(VORTEX, seed=6) for s in setups]

    def started():
        out = [s.context() for s in setups]
        for c, (U, T) in zip(out, states):
            c.upload(U, T)
            c.initialize()
        return out

    alone, together = started(), started()
    for c in alone:
        c.steps(3)
    ens = xf.Ensemble(together)
    assert ens.one_launch
    ens.steps(3)
    ens.synchronize()
    for a, b in zip(alone, together):
        assert np.array_equal(a.download()[0].view(np.uint64), b.download()[0].view(np.uint64))
        for x, y in zip(a.maxima(), b.maxima()):
            assert np.array_equal(x, y)
        assert a.get_dt() == b.get_dt()
    ens.close()
    for c in alone + together:
        c.close()
