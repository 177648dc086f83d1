"""Tensors whose conjugation or negation torch has put off: the memory holds
other values than the tensor has, and the kernels read memory.

Bar of the FFT: relative L2 4e-15 (worst of the random-shape sweep is 3.4e-15).
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n0,n1", [(1, 1), (7, 300), (64, 48), (1024, 263), (3, 15015)])
def test_fft_of_lazy_double_views(n0, n1):
    import torch
    from bldfm_amd import fft_manager

    rng = np.random.default_rng(n0 + 5 * n1)
    x = rng.standard_normal((n0, n1)) + 1j * rng.standard_normal((n0, n1))
    dev = torch.as_tensor(x, device="cuda")
    before = dev.clone()
    for view, base in ((dev.conj(), x.conj()), (torch._neg_view(dev), -x), (dev.mH, x.conj().T), (dev.conj().imag, -x.imag),
                       (torch._neg_view(dev.real), -x.real), (torch._neg_view(dev.conj()), -x.conj())):
        for got, want in ((fft_manager.fft2(view), np.fft.fft2(base)), (fft_manager.ifft2(view, norm="ortho"), np.fft.ifft2(base, norm="ortho"))):
            assert got.dtype == torch.complex128
            assert np.linalg.norm(got.cpu().numpy() - want) <= 4e-15 * np.linalg.norm(want)
    assert torch.equal(dev, before)


def test_solve_of_a_negated_source():
    import torch
    from bldfm_amd import solver
    from oracle import pbl as opbl

    z, prof = opbl.vertical_profiles(8, 10.0, (3.0, 1.5), ustar=0.4, mol=-60.0)
    q = torch.as_tensor(np.random.default_rng(2).random((40, 48)), device="cuda")
    kw = dict(modes=(48, 40), halo=100.0, precision="double")
    got = solver.solve_device(torch._neg_view(q), z, prof, (480.0, 400.0), [2, 8], **kw)
    want = solver.solve_device((-q).clone(), z, prof, (480.0, 400.0), [2, 8], **kw)
    plain = solver.solve_device(q, z, prof, (480.0, 400.0), [2, 8], **kw)
    assert not torch.equal(want[1], plain[1])
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
