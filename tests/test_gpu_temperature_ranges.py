"""Temperature fits where a wave's lanes sit in different fit ranges or outside
the interval of the straight-line fits (200 K to 1e5 K): UpdateStates' Newton
inversion, the species enthalpies behind the primitives, and the chemistry's
rates, bit for bit against the oracle for both fit families."""
import numpy as np
import pytest

import xfluids_amd as xf
from parity import announce, oracle_for

pytestmark = pytest.mark.gpu

# nominal spans whose inverted temperatures lie around 200 K, around the range
# limits 1000 K and 6000 K, over all of them, and above the straight-line interval
SPANS = [(150.0, 260.0), (1000.0, 1250.0), (3500.0, 5000.0), (160.0, 8000.0), (0.8e5, 1.2e5)]


@pytest.mark.parametrize("thermo", [1, 0])
@pytest.mark.parametrize("lo,hi", SPANS)
def test_states_and_chemistry_across_fit_ranges(thermo, lo, hi):
    announce("fit ranges thermo %d T %g..%g" % (thermo, lo, hi))
    s = xf.Setup(xf.case_path("reactive-channel"), nx=18, ny=13, thermo=thermo)
    d = s.desc
    U, T = s.initial("reactive-channel", seed=5)
    rng = np.random.default_rng(11)
    Tn = rng.uniform(lo, hi, T.size)
    # about the energy of Tn: the Newton inversion starts at Tn and ends nearby
    U2 = U.reshape(-1, d.E)
    U2[:, 4] += U2[:, 0] * 900.0 * (Tn - T)
    o = oracle_for(s, U, Tn)
    ctx = s.context()
    ctx.upload(U, Tn)
    o.boundary(0)
    ctx.boundary(0)
    assert xf.lib().xf_update_states(ctx._h, 0) == o.update_states(0)
    P = ctx.prims()
    for name in ("p", "H", "c", "gamma"):
        assert np.array_equal(o.field(name).view(np.uint64), P[name].view(np.uint64)), name
    _, Tg = ctx.download(0)
    assert np.array_equal(o.field("T").view(np.uint64), Tg.view(np.uint64))
    if hi > 1e4:
        ctx.close()
        return  # thousands of passes per cell up there: the inversion only
    o.chemistry(1e-11)
    ctx.chemistry(1e-11)
    Ug, Tg = ctx.download(0)
    ctx.close()
    assert np.array_equal(o.field("U").view(np.uint64), Ug.view(np.uint64))
    assert np.array_equal(o.field("T").view(np.uint64), Tg.view(np.uint64))
