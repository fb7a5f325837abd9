"""The shared chemistry queue of an ensemble with stopped cases, one of them with more
cells than the queue has lanes: the running cases keep the bits they have alone."""
import numpy as np
import pytest

import xfluids_amd as xf
from parity import announce

pytestmark = pytest.mark.gpu

LANES = 256 * 8 * 64  # lanes of the chemistry kernels that fit the chip at once (two waves per SIMD)


SMALL, LARGE = (24, 13), (400, 350)


@pytest.mark.parametrize("sizes,stops", [
    ((LARGE, SMALL), (0,)), ((SMALL, LARGE, SMALL), (1,)), ((SMALL, LARGE), (1,)),
    ((SMALL, LARGE, SMALL, SMALL), (0, 1, 3)), ((LARGE, SMALL), (0, 1))])
def test_running_cases_keep_their_bits(sizes, stops):
    announce("ensemble %s with the cases %s stopped" % (sizes, stops))
    setups = [xf.Setup(xf.case_path("reactive-channel"), nx=n, ny=m) for n, m in sizes]
    assert max(s.desc.ninner for s in setups) > LANES
    states = [s.initial("reactive-channel", seed=8 + k) for k, s in enumerate(setups)]

    def started():
        out = [s.context() for s in setups]
        for c, (U, T) in zip(out, states):
            c.upload(U, T)
            c.initialize()
        for k in stops:
            out[k].set_target_time(0.5 * out[k].get_dt())
        return out

    alone, together = started(), started()
    for c in alone:
        c.steps(3)
    ens = xf.Ensemble(together)
    assert ens.one_launch
    ens.steps(3)
    ens.synchronize()
    for a, b in zip(alone, together):
        for x, y in zip(a.download(), b.download()):
            assert np.array_equal(x.view(np.uint64), y.view(np.uint64))
    ens.close()
    for c in alone + together:
        c.close()
