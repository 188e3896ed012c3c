"""The spectrum's row kernel on rows longer than 257 modes, with four rows at
a time and (many bins) two, in both LDS sizes: the occupation of every bin
exactly, the means of k and k^2 over all modes of a bin to 1e-12, and the
power of single modes at the wavefront boundaries and the ends of a row.
Against numpy with the estimator's expressions."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bins_of(k2, k2max, nb):
    return np.floor(nb * np.sqrt(k2 / k2max)).astype(np.int64)


def all_modes(N, nb):
    """(occupation, sum of k, sum of k^2) of every bin over the N^3 modes; the
    k row ky = 0 .. N/2 stands for ky and N - ky, kz likewise."""
    H = N // 2
    t = (2.0 * np.pi * np.arange(H + 1)) ** 2
    k2max = 3.0 * t[H]
    wx = np.where((np.arange(H + 1) == 0) | (np.arange(H + 1) == H), 1, 2)
    occ, sk, sk2 = np.zeros(nb, dtype=np.int64), np.zeros(nb), np.zeros(nb)
    w2 = wx[:, None] * wx  # (ky, kx)
    for kz in range(H + 1):
        k2 = t + t[:, None] + t[kz]
        b = bins_of(k2, k2max, nb)
        w = w2 * wx[kz]
        if kz == 0:
            w[0, 0] = 0
        live = b < nb
        b, w, k2 = b[live], w[live], k2[live]
        occ += np.bincount(b, weights=w, minlength=nb).astype(np.int64)
        sk += np.bincount(b, weights=w * np.sqrt(k2), minlength=nb)
        sk2 += np.bincount(b, weights=w * k2, minlength=nb)
    return occ, sk, sk2, t, k2max


def test_the_reference_counts_every_mode():
    occ = all_modes(16, 7)[0]
    assert occ.sum() == 16 ** 3 - 2  # all but k = 0 and the corner k = k_max


@pytest.mark.parametrize("N,form,numbins", [(768, 0, (384,)), (768, 1, (16, 1024)), (1024, 1, (64, 512, 1024))])
def test_long_rows(gev, N, form, numbins):
    H = N // 2
    rng = np.random.default_rng(N)
    kxs = [0, 1, 62, 63, 64, 65, 127, 128, 255, 256, 257, 319, H - 1, H]
    modes = [(int(rng.integers(1, N)), int(rng.integers(0, N)), kx, complex(rng.integers(1, 9), rng.integers(-8, 9)))
             for kx in kxs for _ in range(2)]
    F = np.zeros((N, N, H + 1), dtype=np.complex128)
    for kz, ky, kx, a in modes:
        F[kz, ky, kx] = a
    with gev.Box(N, 0, form=form) as b:
        b.upload_field(gev.SCALARFT, F)
        got = {nb: b.extractPowerSpectrum(gev.SCALARFT, nb, False, 1) for nb in numbins}
    for nb in numbins:
        kb, pw, ks, ps, oc = got[nb]
        occ, sk, sk2, t, k2max = all_modes(N, nb)
        assert np.array_equal(oc, occ), nb
        live = occ > 0
        assert np.allclose(kb[live], sk[live] / occ[live], rtol=1e-12, atol=0), nb
        mean2 = ks[live] ** 2 + kb[live] ** 2
        assert np.allclose(mean2, sk2[live] / occ[live], rtol=1e-12, atol=0), nb
        want = np.zeros(nb)
        for kz, ky, kx, a in modes:
            k2 = t[kx] + t[min(ky, N - ky)] + t[min(kz, N - kz)]
            i = int(bins_of(k2, k2max, nb))
            want[i] += (1 if kx in (0, H) else 2) * abs(a) ** 2 * k2 * np.sqrt(k2)
        want[live] /= occ[live]
        assert np.allclose(pw, want, rtol=1e-12, atol=0), nb
