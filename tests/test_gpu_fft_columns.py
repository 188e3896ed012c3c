"""The 3D transforms at every compiled grid size up to 256 in both forms, over
one and several components: single-stage columns (N = 8), columns whose
butterflies do not fill a wavefront, every mix of radices, and the launches
that take several components at once.  Against numpy in float64: the rounding
error of an FFT grows with its number of stages, bounded here by
8 eps log2(N^3) in the 2-norm (eps of the form's element)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [8, 12, 16, 24, 32, 48, 64, 96, 128, 192, 256]


@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("N", SIZES)
def test_transforms_of_one_and_several_components(gev, N, form):
    rng = np.random.default_rng(100 * N + form)
    tol = 8 * (2.0 ** -53 if form == gev.FORM_FP64 else 2.0 ** -24) * np.log2(float(N) ** 3)
    plans = [(gev.PLAN_PHI, gev.PHI, gev.SCALARFT, 1)]
    plans.append((gev.PLAN_SIJ, gev.SIJ, gev.SIJFT, 6) if N <= 128 else (gev.PLAN_BI, gev.BI, gev.BIFT, 3))
    with gev.Box(N, 0, form=form) as b:
        for plan, real, kf, nc in plans:
            f = rng.standard_normal((nc, N, N, N)).astype(np.float32).astype(np.float64)
            b.upload_field(real, f if nc > 1 else f[0])
            b.fft(plan, gev.FFT_FORWARD)
            got = b.download_field(kf).reshape(nc, N, N, N // 2 + 1)
            b.fft(plan, gev.FFT_BACKWARD)
            back = b.download_field(real).reshape(nc, N, N, N)
            for c in range(nc):
                want = np.fft.rfftn(f[c])
                assert np.linalg.norm(got[c] - want) <= tol * np.linalg.norm(want), (N, c)
                # the backward transform starts from the rounded k field
                assert np.linalg.norm(back[c] / N ** 3 - f[c]) <= 2 * tol * np.linalg.norm(f[c]), (N, c)
