"""A NaN that the check after a Reaction finds halts the step behind that launch, not
within it: every cell of the launch has its chemistry, and the lowest bad cell is
reported, whatever the order of the blocks."""
import numpy as np
import pytest

import xfluids_amd as xf
from parity import announce
from test_gpu_errors import same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("driver", [xf.XF_CHEM_PER_CELL, xf.XF_CHEM_QUEUE, xf.XF_CHEM_WAVE])
def test_every_cell_of_the_launch_reacts(driver):
    announce("nan after the reaction, driver %d" % driver)
    # more cells than the chip holds lanes of the chemistry (256 CUs, 8 waves each)
    nx = 256 * 8 * 64 + 20000
    s = xf.Setup(xf.case_path("reactive-shock-tube"), nx=nx)
    d = s.desc
    U, T = s.initial("reactive-shock-tube", seed=3)
    bad = d.Bwidth_X + 5 + 64 * np.arange(2000)  # one in each of the first blocks
    ctx, ref = s.context(chem_driver=driver), s.context(chem_driver=driver)
    for c in (ctx, ref):
        c.upload(U, T)
        c.initialize()
    U0, T0 = ctx.download(0)
    # a transverse momentum in one dimension: only the check after the Reaction sees it
    U0.reshape(-1, d.E)[bad, 2] = np.nan
    for c in (ctx, ref):
        c.upload(U0, T0)
    dt = ref.get_dt()
    ref.update_states(0)
    ref.chemistry(0.5 * dt)
    with pytest.raises(xf.XfError) as ei:
        ctx.steps(1)
    assert (ei.value.status, ei.value.cell, ei.value.step, ei.value.stage) == (3, (int(bad[0]), 0, 0), 1, 4)
    for a, b in zip(ctx.download(0), ref.download(0)):
        assert same_bits(a, b)
    ctx.close()
    ref.close()
