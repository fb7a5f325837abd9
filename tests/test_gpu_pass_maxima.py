"""The GLF and CFL maxima of an UpdateStates pass, which the sweeps and GetDt fold
from its blocks' maxima themselves up to 512 blocks of 256 cells: grids of one block,
at 256 and 512 blocks and one more, bit for bit against the oracle; and an ensemble
with a case on either side."""
import numpy as np
import pytest

import xfluids_amd as xf
from parity import announce, oracle_for

pytestmark = pytest.mark.gpu

# (nx + 6)(ny + 6) cells; 1-D nx + 6
GRIDS = [
    ("isentropic-vortex", "isentropic-vortex", dict(nx=10, ny=10)),  # 1 block
    ("isentropic-vortex", "isentropic-vortex", dict(nx=250, ny=250)),  # 256
    ("isentropic-vortex", "isentropic-vortex", dict(nx=250, ny=251)),  # 257
    ("shock-bubble", "shock-bubble", dict(nx=506, ny=250)),  # 512
    ("shock-bubble", "shock-bubble", dict(nx=507, ny=250)),  # 513
    ("reactive-shock-tube", "reactive-shock-tube", dict(nx=250)),  # 1, the Reaction's pass last
    ("reactive-shock-tube", "reactive-shock-tube", dict(nx=251)),  # 2
]


@pytest.mark.parametrize("case,workload,size", GRIDS)
def test_maxima_match_oracle(case, workload, size):
    announce("pass maxima %s %s" % (case, size))
    s = xf.Setup(xf.case_path(case), **size)
    U, T = s.initial(workload, seed=5)
    o = oracle_for(s, U, T)
    assert o.initialize() == 0
    assert o.steps(2)[0] == 0
    ctx = s.context()
    ctx.upload(U, T)
    ctx.initialize()
    ctx.steps(2)
    Ug, _ = ctx.download()
    E = s.desc.E
    glf, cfl = ctx.maxima()
    assert np.array_equal(o.field("eigen_block").reshape(3, -1)[:, :E], glf[:, :E])
    assert np.array_equal(o.field("U").view(np.uint64), Ug.view(np.uint64))
    assert ctx.get_dt() == o.get_dt()
    assert np.array_equal(ctx.maxima()[1], cfl)
    ctx.close()


def test_ensemble_on_either_side():
    announce("pass maxima ensemble")
    setups = [xf.Setup(xf.case_path("isentropic-vortex"), nx=n, ny=250) for n in (58, 506, 507)]
    states = [s.initial("isentropic-vortex", seed=6) for s in setups]

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
    ens.close()
    for c in alone + together:
        c.close()


@pytest.mark.parametrize("stops", [0, 1, 2])
def test_ensemble_case_that_has_stopped(stops):
    """A case that has reached its target time neither holds back the chemistry of the
    cells that share a wave with its own, nor goes on itself."""
    announce("ensemble with a stopped case %d" % stops)
    setups = [xf.Setup(xf.case_path("reactive-channel"), nx=n, ny=11) for n in (13, 9, 15)]
    states = [s.initial("reactive-channel", seed=7 + k) for k, s in enumerate(setups)]

    def started():
        out = [s.context() for s in setups]
        for c, (U, T) in zip(out, states):
            c.upload(U, T)
            c.initialize()
        out[stops].set_target_time(1.5 * out[stops].get_dt())
        return out

    alone, together = started(), started()
    for c in alone:
        c.steps(4)
    ens = xf.Ensemble(together)
    assert ens.one_launch
    ens.steps(4)
    ens.synchronize()
    for a, b in zip(alone, together):
        for x, y in zip(a.download(), b.download()):
            assert np.array_equal(x.view(np.uint64), y.view(np.uint64))
    ens.close()
    for c in alone + together:
        c.close()
