"""Newton chains of which a few per wave outlast the others (newton_tail): one straggler,
as many as a wave's groups hold and more, long chains that reach the iteration limit,
and stragglers that leave the interval of the straight-line fits, for species counts of
either group size, bit for bit against the oracle."""
import numpy as np
import pytest

import xfluids_amd as xf
from parity import announce, oracle_for

pytestmark = pytest.mark.gpu

# 3, 5, 9 species
CASES = [
    ("shock-bubble", "shock-bubble", dict(nx=50, ny=13)),
    ("inert-sbi", "shock-bubble", dict(nx=14, ny=9, nz=8)),
    ("reactive-channel", "reactive-channel", dict(nx=50, ny=13)),
]


@pytest.mark.parametrize("case,workload,size", CASES)
@pytest.mark.parametrize("every", [64, 16, 8, 7])
@pytest.mark.parametrize("off", [0.6, 0.85, 1.2, 2.5])
def test_stragglers_match_oracle(case, workload, size, every, off):
    announce("newton tail %s every %d off %g" % (case, every, off))
    s = xf.Setup(xf.case_path(case), **size)
    U, T = s.initial(workload, seed=6)
    o = oracle_for(s, U, T)
    assert o.initialize() == 0
    U, T = o.field("U").copy(), o.field("T").copy()
    guess = T.copy()
    guess[3::every] *= off
    o = oracle_for(s, U, guess)
    ctx = s.context()
    ctx.upload(U, guess)
    assert xf.lib().xf_update_states(ctx._h, 0) == o.update_states(0)
    P = ctx.prims()
    for name in ("p", "c", "gamma"):
        assert np.array_equal(o.field(name).view(np.uint64), P[name].view(np.uint64)), name
    _, Tg = ctx.download(0)
    ctx.close()
    assert np.array_equal(o.field("T").view(np.uint64), Tg.view(np.uint64))
