"""Launches with cells below 200 K, where the enthalpies are extrapolated: the chemistry of
a compiled mechanism for both fit families, and UpdateStates of a stream that lies there
throughout or around the limit, bit for bit against the oracle."""
import numpy as np
import pytest

import xfluids_amd as xf
from parity import announce, oracle_for

pytestmark = pytest.mark.gpu


def chemistry(thermo, lo, hi, driver, special, dt=1e-11):
    s = xf.Setup(xf.case_path("reactive-channel"), nx=18, ny=13, thermo=thermo)
    U, _ = s.initial("reactive-channel", seed=14)
    T = np.random.default_rng(15).uniform(lo, hi, U.size // s.desc.E)
    o = oracle_for(s, U, T)
    ctx = s.context(chem_driver=driver)
    ctx.set_chem_specialization(special)
    assert (ctx.chem_specialization() >= 0) == special
    ctx.upload(U, T)
    o.update_states(0)
    ctx.update_states(0)
    # the temperatures of the span, not the inverted ones
    o.field("T")[:] = T
    ctx.upload(ctx.download(0)[0], T)
    o.chemistry(dt)
    ctx.chemistry(dt)
    Ug, Tg = ctx.download(0)
    ctx.close()
    assert np.array_equal(o.field("U").view(np.uint64), Ug.view(np.uint64))
    assert np.array_equal(o.field("T").view(np.uint64), Tg.view(np.uint64))


@pytest.mark.parametrize("thermo", [1, 0])
@pytest.mark.parametrize("lo,hi", [(120.0, 190.0), (1.0, 260.0)])
def test_cold_cells_of_a_compiled_mechanism(thermo, lo, hi):
    announce("cold rates thermo %d T %g..%g" % (thermo, lo, hi))
    chemistry(thermo, lo, hi, xf.XF_CHEM_PER_CELL, True)


# grids of a launch with the Newton tail and of one without
@pytest.mark.parametrize("case,size", [
    ("shock-bubble", dict(nx=50, ny=13)), ("shock-bubble", dict(nx=640, ny=420)),
    ("inert-sbi", dict(nx=14, ny=9, nz=8)), ("reactive-channel", dict(nx=50, ny=13))])
@pytest.mark.parametrize("lo,hi", [(120.0, 190.0), (190.0, 230.0)])
def test_cold_stream(case, size, lo, hi):
    """UpdateStates of a stream below 200 K from guesses a few per cent off."""
    announce("cold stream %s %s T %g..%g" % (case, size, lo, hi))
    s = xf.Setup(xf.case_path(case), **size)
    U, T = s.initial("reactive-channel" if case == "reactive-channel" else "shock-bubble", seed=16)
    rng = np.random.default_rng(17)
    Tn = rng.uniform(lo, hi, T.size)
    U2 = U.reshape(-1, s.desc.E)
    U2[:, 4] += U2[:, 0] * 1000.0 * (Tn - T)
    o = oracle_for(s, U, Tn)
    ctx = s.context()
    ctx.upload(U, Tn)
    assert xf.lib().xf_update_states(ctx._h, 0) == o.update_states(0)
    cold = (o.field("T") < 200.0).mean()
    print("below 200 K: %.2f" % cold)
    assert cold > 0.05
    _, Tg = ctx.download(0)
    P = ctx.prims()
    ctx.close()
    assert np.array_equal(o.field("T").view(np.uint64), Tg.view(np.uint64))
    for name in ("p", "H", "c", "gamma"):
        assert np.array_equal(o.field(name).view(np.uint64), P[name].view(np.uint64)), name
