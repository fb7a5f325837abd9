"""Upload and download of the host's cell-by-cell order: every value lands in its
plane and comes back, for odd and even component counts, cell counts around the
256 cells a block turns, and states of more than one 32 MiB piece."""
import numpy as np
import pytest

import xfluids_amd as xf
from parity import announce

pytestmark = pytest.mark.gpu

# (case, sizes): E = 5, 6, 7, 8, 9, 13, 14; one-dimensional grids of 255, 256 and
# 257 padded cells; the last two take two pieces
GRIDS = [
    ("isentropic-vortex", dict(nx=9, ny=5)),
    ("shock-bubble-h2n2", dict(nx=33, ny=7)),
    ("shock-bubble", dict(nx=31, ny=17)),
    ("inert-sbi-without-fuel", dict(nx=24, ny=11)),
    ("inert-sbi", dict(nx=12, ny=9, nz=10)),
    ("reactive-shock-tube", dict(nx=247)),
    ("reactive-shock-tube", dict(nx=248)),
    ("reactive-shock-tube", dict(nx=249)),
    ("mixing-layer-21", dict(nx=9, ny=8, nz=7)),
    ("mixing-layer", dict(nx=67, ny=65, nz=63)),
    ("shock-bubble", dict(nx=1030, ny=613)),
]


@pytest.mark.parametrize("case,size", GRIDS)
def test_exchange_round_trip(case, size):
    announce("state exchange %s %s" % (case, size))
    s = xf.Setup(xf.case_path(case), **size)
    d = s.desc
    rng = np.random.default_rng(3)
    ctx = s.context()
    for which in (0, 1, 2):
        U, T = rng.standard_normal(d.ncell * d.E), rng.standard_normal(d.ncell)
        ctx.upload(U, T, which=which)
        for back in ((0, 1, 2) if which == 0 else (which,)):  # U also sets U1 and U2
            Ug, Tg = ctx.download(back)
            assert np.array_equal(U.view(np.uint64), Ug.view(np.uint64)), (which, back)
            assert np.array_equal(T.view(np.uint64), Tg.view(np.uint64)), (which, back)
    # the U exchange leaves T alone when none is given
    ctx.upload(U, None, which=1)
    assert np.array_equal(ctx.download(1)[1].view(np.uint64), T.view(np.uint64))
    ctx.close()
