"""Padded lengths with large prime factors about the longest chirp, M = 2048:
windows of 2048 values in all, which it takes, and of 2049 and more, which stay
with the mixed-radix line, along either axis and beside chirp lines of the other
axis and of other instances, against the numpy oracle.

Bar: rel-L2 <= 1e-10 (the solver's).
"""

import numpy as np
import pytest

from conftest import rel_l2
from oracle import pbl as opbl
from oracle import solver as osolver

pytestmark = pytest.mark.gpu

# (nx, ny, px, py, footprint): the inverse pass needs inputs + outputs - 1 of the long axis
CASES = [
    (40, 1024, 3, 201, True),    # 1426 = 2*23*31: 1025 + 1024 - 1 = 2048, a chirp; x 46 = 2*23, a chirp
    (40, 1025, 3, 201, True),    # 1426 of 1427: 1025 + 1025 - 1 = 2049, mixed radix
    (40, 1026, 3, 200, True),    # 1426: 1027 + 1026 - 1 = 2052, mixed radix
    (40, 1026, 3, 200, False),   # the same with the forward passes, 2051
    (1026, 40, 200, 3, False),   # along x
    (1030, 1028, 9, 11, True),   # 1048 = 8*131, 1050 = 2*3*25*7: mixed radix along both
]


def _domain(nx, ny, px, py, halo=100.0):
    # one halo for both axes: choose the cell sizes so that int(halo / dx) = px, int(halo / dy) = py
    return nx * halo / (px + 0.25), ny * halo / (py + 0.25)


@pytest.mark.parametrize("nx,ny,px,py,footprint", CASES)
def test_windows_about_the_longest_chirp_match_the_oracle(nx, ny, px, py, footprint):
    from bldfm_amd import solver

    domain = _domain(nx, ny, px, py)
    z, prof = opbl.vertical_profiles(8, 10.0, (3.0, 1.5), ustar=0.4, mol=-60.0)
    q = np.zeros((ny, nx)) if footprint else np.random.default_rng(nx + ny).random((ny, nx))
    kw = dict(modes=(nx - nx % 2, ny - ny % 2), meas_pt=(0.4 * domain[0], 0.6 * domain[1]) if footprint else (0.0, 0.0),
              footprint=footprint, halo=100.0, precision="double")
    c, f, _ = solver.solve_device(q, z, prof, domain, [8], **kw)
    _, oc, of = osolver.steady_state_transport_solver(q, z, prof, domain, [8], **kw)
    assert rel_l2(f[0].cpu().numpy(), of) <= 1e-10
    assert rel_l2(c[0].cpu().numpy(), oc) <= 1e-10


def test_a_batch_with_and_without_chirps_equals_single_plans_bit_for_bit():
    import torch

    from bldfm_amd.batch import FootprintBatch, FootprintSpec

    specs = []
    for nx, ny, px, py in [(40, 1026, 3, 200), (40, 1024, 3, 201), (64, 66, 15, 10), (1026, 44, 200, 3), (34, 1025, 6, 201)]:
        domain = _domain(nx, ny, px, py)
        specs.append(FootprintSpec(nx=nx, ny=ny, domain=domain, modes=(nx - nx % 2, ny - ny % 2),
                                   meas_pt=(0.5 * domain[0], 0.5 * domain[1]), n=8, meas_height=10.0, wind=(3.0, 1.0),
                                   ustar=0.4, mol=-80.0, halo=100.0))
    fb = FootprintBatch(specs)
    fb.run()
    for i, s in enumerate(specs):
        one = FootprintBatch([s])
        one.run()
        torch.cuda.synchronize()
        for a, b in zip(fb.output(i), one.output(0)):
            assert torch.equal(a, b), i
