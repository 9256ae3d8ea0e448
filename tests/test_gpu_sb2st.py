"""scao_eig_sb2st (band -> tridiagonal) on matrices of any scale: the spectrum
of its tridiagonal against LAPACK's of the band."""

from __future__ import annotations

import numpy as np
import pytest
import scipy.linalg
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("exponent", [0, -498, -505, 400])
@pytest.mark.parametrize("n", [3, 17, 18, 50, 100])
def test_band_keeps_its_spectrum(hip_device, n, exponent):
    """float64 arithmetic throughout: 1e-13 n |B| at any scale whose squares a
    double holds (2^-505: 2^-1010, so that a column a thousandth of |B| still
    has 32 bits and more of its square above the smallest double)."""
    from scao_amd import _lib as L
    rng = np.random.default_rng(n)
    b = min(L.EIG_BAND, n - 1)
    lower = rng.standard_normal((b + 1, n))          # lower[d, c] = B[c + d, c]
    band = np.zeros((n, L.EIG_BANDW))
    for d in range(b + 1):
        band[d:, d] = lower[d, :n - d]               # band[r, d] = B[r, r - d]
        lower[d, n - d:] = 0.0
    dev = torch.from_numpy(np.ldexp(band, exponent))[None].to(hip_device)
    d = torch.empty(1, n, dtype=torch.float64, device=hip_device)
    e = torch.zeros(1, n, dtype=torch.float64, device=hip_device)
    L.call("scao_eig_sb2st", dev.data_ptr(), n, 1, d.data_ptr(), e.data_ptr(),
           L.stream_ptr(hip_device))
    got = scipy.linalg.eigvalsh_tridiagonal(np.ldexp(d.cpu().numpy()[0], -exponent),
                                            np.ldexp(e.cpu().numpy()[0, :n - 1], -exponent))
    want = scipy.linalg.eig_banded(lower, lower=True, eigvals_only=True)
    assert np.abs(got - want).max() <= 1e-13 * n * np.abs(want).max()
