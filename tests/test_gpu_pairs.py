"""The march with two modes per lane (plans of many waves) against the march
with one (plans of one instance), bit for bit: footprints at one and at six
levels, dispersion, every launch block, even and odd retained mode counts.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [64, 128, 256])
@pytest.mark.parametrize("levels", [None, [0, 3, 8, 9, 11, 12]])
def test_batch_of_pairs_equals_single_solves(block, levels):
    import torch

    from bldfm_amd.batch import FootprintBatch, FootprintSpec

    rng = np.random.default_rng(17)
    specs = []
    for i in range(44):
        nx, ny = [(128, 130), (126, 128), (130, 134), (129, 127)][i % 4]  # odd grids at zero halo retain odd modes
        halo = 0.0 if i % 4 == 3 else None
        a = rng.uniform(0.0, 2 * np.pi)
        specs.append(FootprintSpec(nx=nx, ny=ny, domain=(4.0 * nx, 4.0 * ny), modes=(136, 136) if halo == 0.0 else (nx, ny),
                                   meas_pt=(2.0 * nx, 2.0 * ny), n=8, meas_height=10.0,
                                   wind=(4.0 * np.cos(a), 4.0 * np.sin(a)), ustar=0.4,
                                   mol=-60.0 if i % 2 else 150.0, halo=halo, levels=levels))
    fb = FootprintBatch(specs, tuning=dict(shoot_block=block, xpass_layout=0, fft_threads=0))
    fb.run()
    for i, s in enumerate(specs):
        one = FootprintBatch([s])
        one.run()
        torch.cuda.synchronize()
        for a, b in zip(fb.output(i), one.output(0)):
            assert torch.equal(a, b), i


def test_dispersion_pairs_equal_single_solves():
    """48 dispersion instances of one source in one plan."""
    import torch

    from bldfm_amd import _lib
    from bldfm_amd.solver import _geometry, _instance, _level_maps

    nx, ny, dom, n = 128, 126, (600.0, 500.0), 9
    q = np.random.default_rng(3).random((ny, nx))
    dev = _lib.device()
    src = torch.as_tensor(q, device=dev).reshape(-1)

    def plan_of(winds):
        insts, ints = [], []
        for w in winds:
            met = _lib.make_met(n, 10.0, w, 0.4, None, -70.0, 1.0, "MOST", None, None, None)
            lib = _lib.load()
            nz = _lib._I32()
            import ctypes

            _lib.check(lib.bldfm_profile_query(ctypes.byref(met), ctypes.byref(nz), None, None))
            g = _geometry((ny, nx), np.zeros(nz.value), dom, n, (nx, ny), (0.0, 0.0), False, None, "double")
            slot, idx = _level_maps(g["levels"], nz.value)
            inst = _instance(g, 1, False, False, "double", 0.5)
            inst.prof_from_met = 1
            inst.met = met
            insts.append(inst)
            ints.append(np.concatenate([slot, idx]))
        p = _lib.Plan(insts, np.concatenate(ints).astype(np.int32), dev)
        buf = lambda k, t: torch.empty(max(k, 1), dtype=t, device=dev)  # noqa: E731
        conc, flx = buf(p.out_elems, torch.float64), buf(p.out_elems, torch.float64)
        p.execute(buf(p.prof_doubles, torch.float64), src.repeat(len(winds)), conc, flx,
                  buf(p.workspace_bytes, torch.uint8))
        torch.cuda.synchronize()
        return conc.view(len(winds), ny, nx), flx.view(len(winds), ny, nx)

    winds = [(3.0 + 0.05 * i, 1.0 - 0.04 * i) for i in range(48)]
    c, f = plan_of(winds)
    for i, w in enumerate(winds):
        c1, f1 = plan_of([w])
        assert torch.equal(c[i], c1[0]) and torch.equal(f[i], f1[0]), i
