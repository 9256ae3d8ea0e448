"""scao_eig_bisect on tridiagonal matrices against LAPACK in float64: sizes
around its groups of eight steps, both splits of the work (few and many
matrices), zero diagonals, decoupled blocks, repeated eigenvalues, scales."""

from __future__ import annotations

import numpy as np
import pytest
import scipy.linalg
import torch

pytestmark = pytest.mark.gpu


def _bisect(dev, d, e, kq):
    from scao_amd import _lib as L
    B, n = d.shape
    dd, ee = torch.from_numpy(d).to(dev), torch.from_numpy(e).to(dev)
    w = torch.empty(B, kq, dtype=torch.float64, device=dev)
    tot = torch.empty(B, dtype=torch.float64, device=dev)
    work = torch.empty(L.lib().scao_eig_bisect_work(n, B), dtype=torch.uint8, device=dev)
    L.call("scao_eig_bisect", dd.data_ptr(), ee.data_ptr(), n, B, kq, w.data_ptr(),
           tot.data_ptr(), work.data_ptr(), L.stream_ptr(dev))
    return w.cpu().numpy(), tot.cpu().numpy()


def _matrices(n, rng):
    d, e = rng.standard_normal(n), rng.standard_normal(n)
    yield d, e
    yield d * 1e-12, e * 1e-12
    yield d * 1e12, e * 1e12
    yield np.zeros(n), np.ones(n)                      # zero minors at x = 0
    yield np.repeat(rng.standard_normal(-(-n // 4)), 4)[:n], np.zeros(n)   # repeated, all decoupled
    yield d, np.where(np.arange(n) % 5 == 4, 0.0, e)   # blocks of five
    yield np.abs(d) + 3.0, e * 1e-200                  # positive, e^2 underflows
    yield np.where(np.arange(n) % 2 == 0, 1e-30, 1.0) * d, e * 1e-15


@pytest.mark.parametrize("n,kq", [(1, 1), (2, 2), (8, 3), (9, 9), (16, 5), (17, 16), (65, 33),
                                  (300, 64)])
@pytest.mark.parametrize("copies", [1, 300])
def test_bisect_matches_lapack(hip_device, n, kq, copies):
    """The kq largest within 1e-14 n |T|; the clamped sum within n times the
    negative ones' resolution (1e-12 |T| each)."""
    rng = np.random.default_rng(n)
    mats = list(_matrices(n, rng))
    d = np.stack([m[0] for m in mats] * copies)
    e = np.stack([m[1] for m in mats] * copies)
    w, tot = _bisect(hip_device, d, e, kq)
    for i, (dd, ee) in enumerate(mats):
        ev = scipy.linalg.eigvalsh_tridiagonal(dd, ee[:n - 1]) if n > 1 else dd.copy()
        scale = max(np.abs(ev).max(), 1e-300)
        for r in (0, len(mats) * (copies - 1)):
            got, s = w[r + i], tot[r + i]
            assert np.abs(got - ev[::-1][:kq]).max() <= 1e-14 * n * scale, (i, r)
            assert abs(s - np.maximum(ev, 0).sum()) <= 2e-12 * n * scale, (i, r)


@pytest.mark.parametrize("exponent", [-900, -333, -230, 230, 333, 900])
@pytest.mark.parametrize("n,kq", [(9, 9), (65, 33), (300, 64)])
@pytest.mark.parametrize("copies", [1, 300])
def test_bisect_is_scale_free(hip_device, n, kq, exponent, copies):
    """Multiplying T by a power of two multiplies the results by it, bit for
    bit (the test above holds T itself to LAPACK): the counts run on T brought
    to one size, and no product of a few entries leaves the range of a double.
    The clamped sum is the given trace minus the negative ones: exact too."""
    rng = np.random.default_rng(n)
    mats = [m for m in _matrices(n, rng) if np.abs(m[1])[np.abs(m[1]) > 0].min(initial=1.0) > 1e-20]
    d = np.stack([m[0] for m in mats] * copies)
    e = np.stack([m[1] for m in mats] * copies)
    d = np.where(np.abs(d) < 1e-20, 0.0, d)     # nothing of the scaled T is denormal
    w, tot = _bisect(hip_device, d, e, kq)
    ws, tots = _bisect(hip_device, np.ldexp(d, exponent), np.ldexp(e, exponent), kq)
    assert np.array_equal(ws, np.ldexp(w, exponent))
    assert np.array_equal(tots, np.ldexp(tot, exponent))


def test_bisect_zero_matrix(hip_device):
    w, tot = _bisect(hip_device, np.zeros((3, 65)), np.zeros((3, 65)), 33)
    assert np.abs(w).max() <= 1e-300 and np.abs(tot).max() <= 1e-300
