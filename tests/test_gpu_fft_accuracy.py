"""FP64 error of the plain 2-D FFT on lengths with the factors 7, 11 and 13,
against numpy's transform in extended precision.

Bars.  A line of these lengths computed with every twiddle taken from the
tables, as the generic prime stage does it, is off by 2.5 to 2.9e-16 in
relative L2; with twiddle powers formed by repeated products it is off by 4.7
to 7.3e-16 (both arithmetics repeated on the CPU).  Lines alone: 1.25 times the
former, 3.6e-16.  Columns come after rows of eight points, 1.4e-16 in L2 of
their own at most: 3.9e-16.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = [1001, 1183, 1331, 1386, 1540, 1690, 1820, 2002, 2028, 2197, 2401]


@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("rows", [True, False])
def test_prime_lengths_keep_the_generic_stages_accuracy(n, rows):
    from bldfm_amd import fft_manager

    shape, bar = ((64, 1, n), 3.6e-16) if rows else ((40, n, 8), 3.9e-16)
    rng = np.random.default_rng(n)
    x = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    xl = x.astype(np.clongdouble)
    for got, want in ((fft_manager.fft2(x), np.fft.fft2(xl)), (fft_manager.ifft2(x, norm="forward"), np.fft.ifft2(xl, norm="forward"))):
        err = float(np.linalg.norm(got - want) / np.linalg.norm(want))
        print(f"  {n} {'rows' if rows else 'columns'}: {err:.2e}", flush=True)
        assert err <= bar
