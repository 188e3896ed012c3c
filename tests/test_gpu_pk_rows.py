"""The spectrum's row kernel where its tiling has edges: fewer rows per
workgroup than wavefronts, rows longer than one or four wavefronts, each
LDS size of the kernel, one bin, more bins than modes of a row, and the
largest table.  Against the oracle's sequential estimator: the means agree
to 1e-12 (sums of up to 1e7 positive terms in a fixed order, a few ulps per
term), the mode counts exactly; twice the same bits."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,numbins,deconvolve,ktype", [
    (8, 1, 1, 1), (12, 16, 0, 0), (32, 1024, 1, 1), (48, 7, 1, 0), (128, 64, 1, 1), (192, 257, 0, 1), (256, 1024, 1, 1)])
def test_rows_against_the_oracle(gev, N, numbins, deconvolve, ktype):
    rng = np.random.default_rng(N + numbins)
    F = rng.standard_normal((N, N, N // 2 + 1)) + 1j * rng.standard_normal((N, N, N // 2 + 1))
    kb, pw, ks, ps, oc = O.extract_cross_spectrum(F, numbins=numbins, deconvolve=deconvolve, ktype=ktype)
    with gev.Box(N, 0) as b:
        b.upload_field(gev.SCALARFT, F)
        got = b.extractPowerSpectrum(gev.SCALARFT, numbins, bool(deconvolve), ktype)
        again = b.extractPowerSpectrum(gev.SCALARFT, numbins, bool(deconvolve), ktype)
    for g, a in zip(got, again):
        assert np.array_equal(g, a)
    assert np.array_equal(got[4], oc)
    assert np.allclose(got[0], kb, rtol=1e-12, atol=0)
    assert np.allclose(got[1], pw, rtol=1e-12, atol=0)


def test_largest_table_on_a_long_row(gev):
    """N = 768 (the largest LDS rows) with 1024 bins: a field whose only mode
    is A at (kz, ky, kx) = (1, 2, 3) has its power in one bin; every mode is counted."""
    N, nb = 768, 1024
    with gev.Box(N, 0, form=gev.FORM_FP32) as b:
        F = np.zeros((N, N, N // 2 + 1), dtype=np.complex128)
        F[1, 2, 3] = 3.0 - 4.0j
        b.upload_field(gev.SCALARFT, F)
        kb, pw, ks, ps, oc = b.extractPowerSpectrum(gev.SCALARFT, nb, False, 1)
    k2 = (2 * np.pi) ** 2 * 14.0
    i = int(np.floor(nb * np.sqrt(k2 / (3 * (np.pi * N) ** 2))))
    assert int((pw > 0).sum()) == 1 and pw[i] > 0
    assert np.isclose(pw[i], 2 * 25.0 * k2 ** 1.5 / oc[i], rtol=1e-12)
    assert oc.sum() > 0.99 * N ** 3
