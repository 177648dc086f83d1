"""Column tiles of the plain 2-D FFT at their edges: one, four and eight
columns per workgroup, column counts that do not fill a tile, the longest
column of each tile width and the next longer one, against numpy.

Bar: relative L2 4e-15 (worst of the random-shape sweep is 3.4e-15).
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n0,n1,batch", [
    (1, 300, 1), (2, 257, 1), (8, 255, 1), (8, 256, 1), (7, 85, 3), (63, 261, 1), (64, 1003, 1), (1024, 263, 1),
    (1025, 129, 2), (2048, 258, 1), (2047, 33, 8), (2049, 258, 1), (1024, 5, 60), (360, 2, 129),
    (8, 8195, 1), (1, 300, 220), (63, 1041, 1), (256, 255, 1), (256, 256, 1), (97, 700, 1)])
def test_column_tiles_match_numpy(n0, n1, batch):
    from bldfm_amd import fft_manager

    rng = np.random.default_rng(n0 * 7 + n1)
    x = rng.standard_normal((batch, n0, n1)) + 1j * rng.standard_normal((batch, n0, n1))
    for got, want in ((fft_manager.fft2(x), np.fft.fft2(x)), (fft_manager.ifft2(x, norm="ortho"), np.fft.ifft2(x, norm="ortho"))):
        assert np.linalg.norm(got - want) <= 4e-15 * np.linalg.norm(want)


@pytest.mark.parametrize("n0,n1", [
    (7, 11), (13, 49), (121, 169), (343, 77), (91, 1001), (1386, 143), (2197, 14), (22, 2401), (26, 7007), (7007, 3),
    (28, 1331), (17, 1309), (4, 15015), (15015, 2)])
def test_prime_butterflies_match_numpy(n0, n1):
    """Radices 7, 11 and 13 alone, repeated, mixed with each other and with the
    generic stage (17), in rows, columns, both register sizes and split lines."""
    from bldfm_amd import fft_manager

    rng = np.random.default_rng(n0 * 3 + n1)
    x = rng.standard_normal((n0, n1)) + 1j * rng.standard_normal((n0, n1))
    for got, want in ((fft_manager.fft2(x), np.fft.fft2(x)), (fft_manager.ifft2(x, norm="ortho"), np.fft.ifft2(x, norm="ortho"))):
        assert np.linalg.norm(got - want) <= 4e-15 * np.linalg.norm(want)


@pytest.mark.parametrize("n0,n1", [
    (1, 1), (7, 300), (8, 257), (1024, 263), (1025, 260), (2049, 258), (3, 2049), (15015, 3), (3, 15015), (4100, 15015 // 5)])
def test_complex64_rounds_only_the_result(n0, n1):
    """complex64 and float32 fields through every kernel family, contiguous or
    not, conjugate and negated views, eight-byte aligned: the FP64 transform
    rounded once.  A rounding is at most 2^-24 of each part, so is their L2."""
    import torch
    from bldfm_amd import fft_manager

    rng = np.random.default_rng(n0 + 5 * n1)
    flat = (rng.standard_normal(n0 * n1 + 1) + 1j * rng.standard_normal(n0 * n1 + 1)).astype(np.complex64)
    x = flat[1:].reshape(n0, n1)
    dev = torch.as_tensor(flat, device="cuda")[1:].reshape(n0, n1)
    assert dev.data_ptr() % 16 == 8
    turned = torch.as_tensor(np.ascontiguousarray(x.T), device="cuda").T
    for got, base in ((fft_manager.fft2(x), x), (fft_manager.fft2(dev), x), (fft_manager.fft2(turned), x),
                      (fft_manager.fft2(dev.conj()), x.conj()), (fft_manager.fft2(torch._neg_view(dev)), -x),
                      (fft_manager.fft2(x.real), x.real), (fft_manager.fft2(dev.real), x.real),
                      (fft_manager.fft2(dev.conj().imag), -x.imag)):
        want = np.fft.fft2(base.astype(np.complex128))
        got = got if isinstance(got, np.ndarray) else got.cpu().numpy()
        assert got.dtype == np.complex64
        assert np.linalg.norm(got - want) <= 6e-8 * np.linalg.norm(want)
    got, want = fft_manager.ifft2(dev).cpu().numpy(), np.fft.ifft2(x.astype(np.complex128))
    assert np.linalg.norm(got - want) <= 6e-8 * np.linalg.norm(want)
