"""A solve from host profiles under graph capture: refused, as the graph would
replay a copy from host memory that has other owners by then; the next solve
is not disturbed."""

import numpy as np
import pytest

from oracle import pbl as opbl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("footprint", [True, False])
def test_solves_from_host_profiles_are_not_captured(footprint):
    import torch
    from bldfm_amd import solver

    z, prof = opbl.vertical_profiles(8, 10.0, (3.0, 1.5), ustar=0.4, mol=-60.0)
    q = torch.as_tensor(np.random.default_rng(5).random((40, 48)), device="cuda")
    kw = dict(modes=(48, 40), halo=100.0, precision="double", footprint=footprint)
    args = (q, z, prof, (480.0, 400.0), [8])
    before = solver.solve_device(*args, **kw)
    torch.cuda.synchronize()
    with pytest.raises(RuntimeError):
        with torch.cuda.graph(torch.cuda.CUDAGraph()):
            solver.solve_device(*args, **kw)
    after = solver.solve_device(*args, **kw)
    torch.cuda.synchronize()
    assert torch.equal(before[0], after[0]) and torch.equal(before[1], after[1])
