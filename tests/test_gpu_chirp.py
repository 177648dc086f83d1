"""Chirp transforms of padded lengths with large prime factors, at the edges
of their lengths: windows that just fit a power of two and the next one, odd
and prime padded lengths, footprints and dispersion (all four passes, both
output types), several levels, against the numpy oracle.

Bar: rel-L2 <= 1e-10 in FP64 (the solver's), 1e-6 in single precision output.
"""

import numpy as np
import pytest

from conftest import rel_l2
from oracle import pbl as opbl
from oracle import solver as osolver

pytestmark = pytest.mark.gpu

# (nx, ny, px, py, footprint, precision, levels): padded lengths in the comments
CASES = [
    (32, 32, 1, 3, False, "double", [0, 4, 8]),       # 34 = 2*17, 38 = 2*19: one wave, M = 64 just fits 63
    (34, 64, 6, 12, False, "double", [8]),            # 46 = 2*23, 88 = 8*11; M = 128
    (64, 66, 15, 10, True, "double", [8]),            # 94 = 2*47, 86 = 2*43; windows of 128 and 132 -> M = 128, 256
    (128, 130, 33, 30, False, "single", [2, 8]),      # 194 = 2*97, 190 = 2*5*19, float32 output
    (126, 257, 40, 20, True, "double", [8]),          # odd ny: the 296-point transform of a 297-point grid
    (256, 250, 61, 62, False, "double", [8]),         # 378 = 2*27*7, 374 = 2*11*17; M = 512
    (400, 258, 47, 70, True, "double", [8]),          # 494 = 2*13*19, 398 = 2*199; M = 1024
    (516, 40, 121, 7, False, "double", [4, 8]),       # 758 = 2*379; M = 2048 along x
    (40, 1024, 7, 200, True, "double", [8]),          # 1424 = 16*89; M = 2048 just too short by one
]


@pytest.mark.parametrize("nx,ny,px,py,footprint,precision,levels", CASES)
def test_rough_padded_lengths_match_the_oracle(nx, ny, px, py, footprint, precision, levels):
    from bldfm_amd import solver

    # one halo for both axes: choose the cell sizes so that int(halo / dx) = px, int(halo / dy) = py
    halo = 100.0
    dx, dy = halo / (px + 0.25), halo / (py + 0.25)
    domain = (nx * dx, ny * dy)
    z, prof = opbl.vertical_profiles(8, 10.0, (3.0, 1.5), ustar=0.4, mol=-60.0)
    q = np.zeros((ny, nx))
    if not footprint:
        q = np.random.default_rng(nx + ny).random((ny, nx))
    kw = dict(modes=(nx - nx % 2, ny - ny % 2), meas_pt=(0.4 * domain[0], 0.6 * domain[1]) if footprint else (0.0, 0.0),
              footprint=footprint, halo=halo, precision=precision)
    c, f, _ = solver.solve_device(q, z, prof, domain, levels, **kw)
    _, oc, of = osolver.steady_state_transport_solver(q, z, prof, domain, levels, **kw)
    bar = 1e-6 if precision == "single" else 1e-10
    assert c.shape == (len(levels),) + np.shape(oc)[-2:]
    for k in range(len(levels)):
        a, b = (np.reshape(x, (len(levels),) + np.shape(oc)[-2:])[k] for x in (oc, of))
        assert rel_l2(f[k].cpu().numpy(), b) <= bar
        if np.any(a):
            assert rel_l2(c[k].cpu().numpy(), a) <= bar


def test_a_mixed_batch_equals_single_plans_bit_for_bit():
    """Chirp lines of several lengths and mixed-radix lines in one plan."""
    import torch

    from bldfm_amd.batch import FootprintBatch, FootprintSpec

    specs = [FootprintSpec(nx=nx, ny=ny, domain=(4.0 * nx, 4.0 * ny), modes=(nx - nx % 2, ny - ny % 2),
                           meas_pt=(2.0 * nx, 2.0 * ny), n=8, meas_height=10.0, wind=(3.0, 1.0), ustar=0.4, mol=-80.0,
                           halo=4.0 * h + 0.5)
             for nx, ny, h in [(64, 48, 15), (130, 65, 33), (33, 257, 20), (128, 128, 128), (300, 40, 47), (90, 94, 9)]]
    fb = FootprintBatch(specs)
    fb.run()
    for layout in (0, 1, 2):
        for i, s in enumerate(specs):
            one = FootprintBatch([s], tuning=dict(shoot_block=64, xpass_layout=layout, fft_threads=0))
            one.run()
            torch.cuda.synchronize()
            for a, b in zip(fb.output(i), one.output(0)):
                assert torch.equal(a, b), (i, layout)
