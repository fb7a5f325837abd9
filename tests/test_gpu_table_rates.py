"""Mechanisms that are not compiled in: the loop over the device tables with the species
values of the straight-line fits, over the fit ranges and below 200 K, for both fit
families and the drivers that run it, bit for bit against the oracle."""
import pytest

import xfluids_amd as xf
from parity import announce
from test_gpu_cold_cells import chemistry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("driver", [xf.XF_CHEM_PER_CELL, xf.XF_CHEM_QUEUE])
@pytest.mark.parametrize("thermo", [1, 0])
@pytest.mark.parametrize("lo,hi", [(900.0, 1100.0), (5500.0, 6500.0), (160.0, 3000.0), (120.0, 190.0), (1.0, 260.0)])
def test_table_loop_matches_oracle(thermo, lo, hi, driver):
    announce("table rates thermo %d T %g..%g driver %d" % (thermo, lo, hi, driver))
    chemistry(thermo, lo, hi, driver, False)


