"""The chemistry drivers' straight-line paths and what they leave to the general ones,
bit for bit: temperatures around the fit ranges and below 200 K against the oracle, and
the wave driver against one lane per cell for mechanisms whose reactions do and do not
fit the packed records, and for negative rates (which one lane per cell divides as
IEEE, like the wave driver)."""
import numpy as np
import pytest

import xfluids_amd as xf
from parity import announce, oracle_for

pytestmark = pytest.mark.gpu


def case(thermo, lo, hi):
    s = xf.Setup(xf.case_path("reactive-channel"), nx=18, ny=13, thermo=thermo)
    U, _ = s.initial("reactive-channel", seed=9)
    return s, U, np.random.default_rng(12).uniform(lo, hi, U.size // s.desc.E)


def context(s, U, T, driver):
    ctx = s.context(chem_driver=driver)
    ctx.upload(U, T)
    ctx.initialize()
    ctx.upload(U, T)
    return ctx


@pytest.mark.parametrize("thermo", [1, 0])
@pytest.mark.parametrize("lo,hi", [(150.0, 260.0), (900.0, 1100.0), (5500.0, 6500.0), (160.0, 3000.0)])
def test_ranges_match_oracle(thermo, lo, hi):
    announce("wave rates thermo %d T %g..%g" % (thermo, lo, hi))
    s, U, T = case(thermo, lo, hi)
    o = oracle_for(s, U, T)
    ctx = context(s, U, T, xf.XF_CHEM_WAVE)
    p = o.field("p")
    ctx.update_states(0)
    o.update_states(0)
    assert np.array_equal(p.view(np.uint64), ctx.prims()["p"].view(np.uint64))
    o.chemistry(1e-11)
    ctx.chemistry(1e-11)
    Ug, Tg = ctx.download(0)
    ctx.close()
    assert np.array_equal(o.field("U").view(np.uint64), Ug.view(np.uint64))
    assert np.array_equal(o.field("T").view(np.uint64), Tg.view(np.uint64))


# orders written over reaction r's, the same on both sides so that it is in balance:
# squares of two species, a cube, four species, none
@pytest.mark.parametrize("nu", [{0: 2, 3: 2}, {1: 3}, {0: 1, 1: 1, 2: 1, 4: 1}, {}])
@pytest.mark.parametrize("r,sign", [(0, 1.0), (-1, 1.0), (0, -1.0)])
def test_mechanisms_match_per_cell(nu, r, sign):
    announce("wave rates mechanism %s %d %g" % (nu, r, sign))
    s, U, T = case(1, 900.0, 1300.0)
    d = s.desc
    Nu_f, Nu_b, third, Rargus = s.mechanism()
    for side in (Nu_f, Nu_b):
        row = side.reshape(d.NR, d.NS)[r]
        row[:] = 0
        for n, v in nu.items():
            row[n] = v
    Rargus.reshape(d.NR, 6)[r, 2] = 0.0
    Rargus.reshape(d.NR, 6)[r, 0] *= sign
    i32 = lambda a: a.ctypes.data_as(xf.C.POINTER(xf.C.c_int))
    f64 = lambda a: a.ctypes.data_as(xf.C.POINTER(xf.C.c_double))
    out = []
    for driver in (xf.XF_CHEM_PER_CELL, xf.XF_CHEM_WAVE):
        ctx = context(s, U, T, driver)
        assert xf.lib().xf_set_mechanism(ctx._h, i32(Nu_f), i32(Nu_b), f64(third), f64(Rargus)) == 0
        ctx.update_states(0)
        sub = ctx.chemistry(1e-13, record=True)
        out.append((sub, *ctx.download(0)))
        ctx.close()
    assert np.array_equal(out[0][0], out[1][0])
    for a, b in zip(out[0][1:], out[1][1:]):
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64))
