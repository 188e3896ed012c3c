"""The 3D transforms from 384^3 up, where a thread of the column passes has
several first-stage butterflies, a last stage does not divide by the threads
(384 and 768: radix 3) or the workgroup is one butterfly per thread of 768.
The field is a product of three random vectors, a different value at every
point, so its transform is the product of three 1D transforms.  The bound is
that of the small grids: 8 eps log2(N^3) in the 2-norm (eps of the form's
element), per component and direction."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def vectors(rng, N):
    return [rng.standard_normal(N) for _ in range(3)]  # z, y, x


def field(v, form):
    f = v[0][:, None, None] * (v[1][:, None] * v[2])
    return f.astype(np.float32) if form else f


def rel(got, want):
    """|got - want| / |want| of two arrays of planes (want: plane -> array)."""
    d = n = 0.0
    for z in range(len(got)):
        w = want(z)
        d += np.sum(np.abs(got[z] - w) ** 2)
        n += np.sum(np.abs(w) ** 2)
    return np.sqrt(d / n)


@pytest.mark.parametrize("N,form,six", [(384, 0, True), (384, 1, True), (512, 0, False), (512, 1, False),
                                        (768, 0, False), (768, 1, False), (1024, 1, False)])
def test_transforms(gev, N, form, six):
    rng = np.random.default_rng(N + form)
    tol = 8 * (2.0 ** -24 if form else 2.0 ** -53) * np.log2(float(N) ** 3)
    vs = [vectors(rng, N) for _ in range(6 if six else 1)]
    plan, real, kf = (gev.PLAN_SIJ, gev.SIJ, gev.SIJFT) if six else (gev.PLAN_PHI, gev.PHI, gev.SCALARFT)
    with gev.Box(N, 0, form=form) as b:
        f = np.stack([field(v, form) for v in vs]) if six else field(vs[0], form)
        b.upload_field(real, f.astype(np.float64))
        del f
        b.fft(plan, gev.FFT_FORWARD)
        got = b.download_field(kf).reshape(len(vs), N, N, N // 2 + 1)
        for c, v in enumerate(vs):
            kz, kyx = np.fft.fft(v[0]), np.fft.fft(v[1])[:, None] * np.fft.rfft(v[2])
            assert rel(got[c], lambda z: kz[z] * kyx) <= tol, (N, c, "forward")
        del got
        b.fft(plan, gev.FFT_BACKWARD)
        back = b.download_field(real).reshape(len(vs), N, N, N)
        for c, v in enumerate(vs):
            yx = v[1][:, None] * v[2]
            assert rel(back[c] / float(N) ** 3, lambda z: v[0][z] * yx) <= 2 * tol, (N, c, "backward")
