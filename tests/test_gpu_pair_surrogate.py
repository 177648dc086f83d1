"""Which march a plan takes when a surrogate may serve some of its instances:
those march singly (only the few that the gate sends back march at all) and do
not count for the others' choice; results are the same bits."""

import numpy as np
import pytest

import test_gpu_pair_plans as base

pytestmark = pytest.mark.gpu


def _batch(nplain, nserved):
    from bldfm_amd import _lib
    from bldfm_amd.batch import FootprintSpec, _instance

    insts, ints = [], []
    for i in range(nplain + nserved):
        spec = FootprintSpec(nx=base.NX, ny=base.NY, domain=base.DOMAIN, modes=(base.NX, base.NY), meas_pt=(170.0, 230.0),
                             n=base.N, meas_height=10.0, wind=(3.0 + 0.05 * i, 1.0 - 0.04 * i), ustar=0.4, mol=-70.0)
        inst, lv, _ = _instance(spec, "double", False, surrogate=i >= nplain)
        insts.append(inst)
        ints.append(lv)
    return _lib.Plan(insts, np.concatenate(ints).astype(np.int32), _lib.device())


@pytest.mark.parametrize("nplain,nserved,paired", [
    (46, 0, True), (0, 46, False), (46, 82, True), (2, 126, False), (20, 26, False), (46, 1, True)])
def test_served_instances_march_singly(nplain, nserved, paired):
    plan = _batch(nplain, nserved)
    assert plan.marches() == ((nserved, nplain) if paired else (nplain + nserved, 0))


def test_served_and_plain_instances_equal_single_solves():
    """No network attached: every instance is solved, 46 in pairs and 3 singly."""
    import torch

    both = _batch(46, 3)
    assert both.marches() == (3, 46)
    conc, flx = base._solve(both, 49, None)
    alone = _batch(49, 0)
    assert alone.marches() == (49, 0)
    c, f = base._solve(alone, 49, None)
    assert torch.equal(conc, c) and torch.equal(flx, f)
