"""Profiles evaluated by four groups of a workgroup, at the edges of its 64
and 256 levels: against the oracle (rtol 1e-12), and the level table made from
them against the one made from the same profiles as caller arrays (equal
footprints bit for bit).
"""

import numpy as np
import pytest

from oracle import pbl as opbl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("closure", ["MOST", "MOSTM", "CONSTANT", "OAAHOC"])
@pytest.mark.parametrize("mol", [-40.0, 90.0])
@pytest.mark.parametrize("nlev", [2, 63, 64, 65, 256, 257, 300])
def test_profiles_at_the_group_edges(nlev, mol, closure):
    import torch

    from bldfm_amd.batch import FootprintBatch, FootprintSpec
    from bldfm_amd.pbl_model import vertical_profiles
    from bldfm_amd.solver import solve_device

    kw = dict(meas_height=10.0, wind=(3.0, 1.0), ustar=0.4, mol=mol, closure=closure,
              tke=0.8 if closure == "OAAHOC" else None)
    # the grid's length grows with n: the n whose grid has nlev levels (or the nearest above)
    n = next(k for k in range(1, 400) if len(opbl.vertical_profiles(k, **kw)[0]) >= nlev)
    z, prof = vertical_profiles(n, **kw)
    oz, oprof = opbl.vertical_profiles(n, **kw)
    np.testing.assert_allclose(z, np.ravel(oz), rtol=1e-12)
    for a, b in zip(prof, oprof):
        np.testing.assert_allclose(a, np.ravel(b), rtol=1e-12)
    level = min(n, len(z) - 1)
    spec = FootprintSpec(nx=12, ny=10, domain=(60.0, 50.0), modes=(12, 10), meas_pt=(30.0, 25.0), n=n, levels=[level], **kw)
    fb = FootprintBatch([spec])
    fb.run()
    c, f, _ = solve_device(np.zeros((10, 12)), z, prof, (60.0, 50.0), level, modes=(12, 10), meas_pt=(30.0, 25.0),
                           footprint=True, precision="double")
    torch.cuda.synchronize()
    got = fb.profiles(0)
    assert np.array_equal(got[0], z) and all(np.array_equal(a, b) for a, b in zip(got[1], prof))
    for a, b in zip(fb.output(0), (c, f)):
        assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))
