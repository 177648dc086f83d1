"""Plans that march two modes per lane, asked for by count: dispersion (whose
lanes read the source's modes q^0 of both) and footprints, at one output level
and at more than a lane keeps (the second march), against single-instance
plans, which march one mode per lane, bit for bit.

46 instances of 128 x 126 modes are 46 * 128 waves of single modes or 46 * 66 of
pairs; over 1024 SIMDs that is 6 rounds of 84 operations against 3 of 155.
"""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NX, NY, DOMAIN, N, COUNT = 128, 126, (600.0, 500.0), 9, 46


def _plan(winds, levels, footprint, meas_pt=(0.0, 0.0)):
    from bldfm_amd import _lib
    from bldfm_amd.solver import _geometry, _instance, _level_maps

    insts, ints = [], []
    for w in winds:
        met = _lib.make_met(N, 10.0, w, 0.4, None, -70.0, 1.0, "MOST", None, None, None)
        nz = _lib._I32()
        _lib.check(_lib.load().bldfm_profile_query(ctypes.byref(met), ctypes.byref(nz), None, None))
        g = _geometry((NY, NX), np.zeros(nz.value), DOMAIN, levels, (NX, NY), meas_pt, footprint, None, "double")
        slot, idx = _level_maps(g["levels"], nz.value)
        inst = _instance(g, len(g["levels"]), footprint, False, "double", 0.5)
        inst.prof_from_met = 1
        inst.met = met
        insts.append(inst)
        ints.append(np.concatenate([slot, idx]))
    return _lib.Plan(insts, np.concatenate(ints).astype(np.int32), _lib.device())


def _solve(plan, count, src):
    import torch

    dev = plan.device
    buf = lambda k, t: torch.empty(max(k, 1), dtype=t, device=dev)  # noqa: E731
    conc, flx = buf(plan.out_elems, torch.float64), buf(plan.out_elems, torch.float64)
    plan.execute(buf(plan.prof_doubles, torch.float64), None if src is None else src.repeat(count), conc, flx,
                 buf(plan.workspace_bytes, torch.uint8))
    torch.cuda.synchronize()
    return conc.view(count, -1), flx.view(count, -1)


@pytest.mark.parametrize("footprint", [False, True])
@pytest.mark.parametrize("levels", [[N], [0, 2, 3, 5, 8, 9]])
@pytest.mark.parametrize("meas_pt", [(0.0, 0.0), (170.0, 230.0)])
def test_paired_plans_equal_single_solves(footprint, levels, meas_pt):
    import torch

    src = None if footprint else torch.as_tensor(np.random.default_rng(3).random(NY * NX), device="cuda")
    winds = [(3.0 + 0.05 * i, 1.0 - 0.04 * i) for i in range(COUNT)]
    batch = _plan(winds, levels, footprint, meas_pt)
    assert batch.marches() == (0, COUNT)
    conc, flx = _solve(batch, COUNT, src)
    for i, w in enumerate(winds):
        one = _plan([w], levels, footprint, meas_pt)
        assert one.marches() == (1, 0)
        c, f = _solve(one, 1, src)
        assert torch.equal(conc[i], c[0]) and torch.equal(flx[i], f[0]), i


def test_marches_of_a_null_plan():
    from bldfm_amd import _lib

    assert _lib.load().bldfm_plan_marches(None, None, None) == -1
