"""Reading a case's maxima while an ensemble steps it: the read leaves nothing behind, on
grids whose kernels fold the maxima themselves (up to 512 blocks of 256 cells) and on
larger ones, whose sweeps read the folded slots."""
import numpy as np
import pytest

import xfluids_amd as xf
from parity import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [96, 420])
def test_maxima_during_ensemble_steps(n):
    announce("maxima in flight, %d x 330" % n)
    s = xf.Setup(xf.case_path("shock-bubble"), nx=n, ny=330)
    d = s.desc
    assert ((d.Xmax * d.Ymax + 255) // 256 > 512) == (n == 420)
    U, T = s.initial("shock-bubble", seed=2)
    alone, each = s.context(), s.context()
    for c in (alone, each):
        c.upload(U, T)
        c.initialize()
    alone.steps(60)
    ens = xf.Ensemble([each])
    assert ens.one_launch
    for _ in range(12):
        ens.steps(5)
        each.maxima()
    ens.synchronize()
    assert np.array_equal(alone.download()[0].view(np.uint64), each.download()[0].view(np.uint64))
    for a, b in zip(alone.maxima(), each.maxima()):
        assert np.array_equal(a, b)
    assert alone.get_dt() == each.get_dt()
    ens.close()
    alone.close()
    each.close()
