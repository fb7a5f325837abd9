"""The forms that the kernels take where their unscaled quotients, square roots and
straight-line fits do not hold, bit for bit against the oracle: thermal tables with a
coefficient too small for them, transport fits whose exponentials leave their range
before or after the first check, and states of extreme density and pressure (scaled by a
power of two: the flow is the same, the range checks fail)."""
import numpy as np
import pytest

import xfluids_amd as xf
from oracle_lib import Oracle, config_from_setup
from parity import announce, grid_shape, interior

pytestmark = pytest.mark.gpu

CASES = {
    "mixing": ("mixing-layer", "mixing-layer", dict(nx=12, ny=10, nz=9)),  # 9 species, reacting, viscous, JS
    "mixing21": ("mixing-layer-21", "mixing-layer", dict(nx=9, ny=8, nz=8)),  # 10 species, GhostSpecies
    "sbi": ("inert-sbi", "shock-bubble", dict(nx=16, ny=8, nz=8)),  # 5 species, viscous, CU6, limiter
    "bubble": ("shock-bubble", "shock-bubble", dict(nx=48, ny=24)),  # 3 species, JANAF, Z
    "channel": ("reactive-channel", "reactive-channel", dict(nx=18, ny=13)),  # 9 species, reacting
}


def tiny_coefficient(s):
    """The thermal tables with 1e-95, below 2^-300, for the coefficients that are zero."""
    Hia, Hib, Wi = s.thermo_tables()
    assert (Hia == 0.0).any()
    Hia[Hia == 0.0] = 1.0e-95
    return Hia, Hib, Wi


def transport(s, what):
    """Transport fits with one species' viscosity or conductivity, or one pair's
    diffusion coefficient, beyond exp(+-200)."""
    fcv, fct, Dkj = s.transport_tables()
    NS = s.desc.NS
    if what == "viscosity":
        fcv[4 * 1] -= 215.0
    elif what == "conductivity":
        fct[4 * (NS - 1)] -= 230.0
    else:
        D = Dkj.reshape(NS, NS, 4)
        D[0, 1, 0] += 230.0
        D[1, 0, 0] = D[0, 1, 0]
    return fcv, fct, Dkj


def matches(case, scale=1.0, thermo=None, tr=None, steps=2, driver=xf.XF_CHEM_PER_CELL, special=True):
    cf, wl, size = CASES[case]
    s = xf.Setup(xf.case_path(cf), **size)
    d = s.desc
    U, T = s.initial(wl, seed=12)
    U = U * scale
    cfg = config_from_setup(s)
    ctx = s.context(chem_driver=driver)
    dp = lambda a: a.ctypes.data_as(xf.C.POINTER(xf.C.c_double))  # noqa: E731
    if thermo:
        tables = thermo(s)
        for name, a in zip(("Hia", "Hib"), tables):
            getattr(cfg, name)[: a.size] = list(a)
        assert xf.lib().xf_set_thermo(ctx._h, *[dp(a) for a in tables]) == 0
    if tr:
        tables = transport(s, tr)
        for name, a in zip(("fcv", "fct", "Dkj"), tables):
            getattr(cfg, name)[: a.size] = list(a)
        assert xf.lib().xf_set_transport(ctx._h, *[dp(a) for a in tables]) == 0
    if d.react and not special:
        ctx.set_chem_specialization(False)
    o = Oracle(cfg)
    o.set_state(U, T)
    ctx.upload(U, T)
    assert o.initialize() == 0
    ctx.initialize()
    st, dts = o.steps(steps)
    assert st == 0
    assert np.array_equal(ctx.steps(steps, record_dt=True), dts)
    Ug, Tg = ctx.download(0)
    ctx.close()
    assert np.isfinite(Ug).all()
    assert np.array_equal(o.field("U").view(np.uint64), Ug.view(np.uint64))
    assert np.array_equal(o.field("T").view(np.uint64), Tg.view(np.uint64))


@pytest.mark.parametrize("case", sorted(CASES))
def test_thermal_table_out_of_range(case):
    announce("general forms, thermal table, " + case)
    matches(case, thermo=tiny_coefficient)


@pytest.mark.parametrize("driver", [xf.XF_CHEM_PER_CELL, xf.XF_CHEM_QUEUE, xf.XF_CHEM_WAVE])
@pytest.mark.parametrize("special", [True, False])
def test_thermal_table_out_of_range_chemistry(driver, special):
    announce("general forms, thermal table, channel driver %d special %s" % (driver, special))
    matches("channel", thermo=tiny_coefficient, driver=driver, special=special)


@pytest.mark.parametrize("what", ["viscosity", "conductivity", "diffusion"])
@pytest.mark.parametrize("case", ["mixing", "mixing21", "sbi"])
def test_transport_fits_out_of_range(case, what):
    announce("general forms, %s fit, %s" % (what, case))
    matches(case, tr=what)


# 2^-130: outside the face's [2^-100, 2^100]; 2^-330: outside the transport's and the
# chemistry's [2^-300, 2^300] too.  (Thin viscous states do not survive a step, dense
# reacting ones take more passes than the bound.)
@pytest.mark.parametrize("case,exponent", [("bubble", -130), ("bubble", 130), ("bubble", -330), ("channel", -130),
                                           ("channel", -330), ("sbi", 130)])
def test_extreme_states(case, exponent):
    announce("general forms, state scaled by 2^%d, %s" % (exponent, case))
    matches(case, scale=2.0**exponent)


@pytest.mark.parametrize("exponent", [-130, -330])
@pytest.mark.parametrize("case", ["mixing", "mixing21", "sbi"])
def test_extreme_viscous_divergence(case, exponent):
    announce("general forms, divergence of a state scaled by 2^%d, %s" % (exponent, case))
    cf, wl, size = CASES[case]
    s = xf.Setup(xf.case_path(cf), **size)
    U, T = s.initial(wl, seed=12)
    U = U * 2.0**exponent
    o = Oracle(config_from_setup(s))
    o.set_state(U, T)
    ctx = s.context()
    ctx.upload(U, T)
    assert o.initialize() == 0
    ctx.initialize()
    o.compute_lu(0)
    ctx.compute_lu(0)
    LU = o.field("LU").reshape(grid_shape(s.desc, s.desc.E))
    G = ctx.lu().reshape(LU.shape)
    assert np.isfinite(interior(LU, s.desc)).all()
    assert np.array_equal(interior(LU, s.desc).view(np.uint64), interior(G, s.desc).view(np.uint64))
    if s.desc.react:
        o.chemistry(1e-9)
        ctx.chemistry(1e-9)
        Ug, Tg = ctx.download(0)
        assert np.array_equal(o.field("U").view(np.uint64), Ug.view(np.uint64))
        assert np.array_equal(o.field("T").view(np.uint64), Tg.view(np.uint64))
    ctx.close()
