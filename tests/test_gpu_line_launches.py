"""Chirp lines of several lengths in one launch and, where there are many, in a
launch each, dispersion (four passes) and footprints: single-instance plans,
whose passes have one length, bit for bit.
"""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (nx, ny, px, py): M = 64, 128, 256, 512, 1024 and 2048 along one axis or both
SMALL = [(32, 32, 1, 3), (48, 60, 17, 20), (64, 66, 15, 10), (128, 130, 33, 30), (200, 222, 202, 150), (400, 258, 47, 70)]
LONG = (1022, 1022, 190, 190)  # 1402 = 2*701: M = 2048, a workgroup a line


def _plan(geometry, footprint, winds):
    from bldfm_amd import _lib
    from bldfm_amd.solver import _geometry, _instance, _level_maps

    insts, ints = [], []
    for (nx, ny, px, py), w in zip(geometry, winds):
        met = _lib.make_met(8, 10.0, w, 0.4, None, -70.0, 1.0, "MOST", None, None, None)
        nz = _lib._I32()
        _lib.check(_lib.load().bldfm_profile_query(ctypes.byref(met), ctypes.byref(nz), None, None))
        domain = (nx * 100.0 / (px + 0.25), ny * 100.0 / (py + 0.25))
        g = _geometry((ny, nx), np.zeros(nz.value), domain, [8], (nx, ny), (0.0, 0.0), footprint, 100.0, "double")
        slot, idx = _level_maps(g["levels"], nz.value)
        inst = _instance(g, 1, footprint, False, "double", 0.5)
        inst.prof_from_met = 1
        inst.met = met
        insts.append(inst)
        ints.append(np.concatenate([slot, idx]))
    return _lib.Plan(insts, np.concatenate(ints).astype(np.int32), _lib.device())


def _solve(plan, src):
    import torch

    buf = lambda k, t: torch.empty(max(k, 1), dtype=t, device=plan.device)  # noqa: E731
    conc, flx = buf(plan.out_elems, torch.float64), buf(plan.out_elems, torch.float64)
    plan.execute(buf(plan.prof_doubles, torch.float64), src, conc, flx, buf(plan.workspace_bytes, torch.uint8))
    torch.cuda.synchronize()
    return conc, flx


@pytest.mark.parametrize("footprint", [False, True])
@pytest.mark.parametrize("nlong", [0, 1, 9])  # 9198 tiles a pass: more than one launch takes
def test_lines_of_several_lengths_equal_single_plans(footprint, nlong):
    import torch

    geometry = SMALL + [LONG] * nlong + SMALL[::-1]
    winds = [(3.0 + 0.1 * i, 1.0 - 0.05 * i) for i in range(len(geometry))]
    rng = np.random.default_rng(4)
    srcs = [None if footprint else torch.as_tensor(rng.random(g[0] * g[1]), device="cuda") for g in geometry]
    batch = _plan(geometry, footprint, winds)
    conc, flx = _solve(batch, None if footprint else torch.cat(srcs))
    for i, g in enumerate(geometry):
        c, f = _solve(_plan([g], footprint, [winds[i]]), srcs[i])
        o = batch.offsets[i][2]
        assert torch.equal(conc[o : o + c.numel()], c) and torch.equal(flx[o : o + f.numel()], f), i
