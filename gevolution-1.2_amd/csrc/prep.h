// prep.h -- per-site bodies of prepareFTsource (gevolution.hpp:56-192,
// PHINONLINEAR on, ORIGINALMETRIC off), shared by the standalone stencil
// kernels (stencil.hip) and the first FFT pass that applies them on the fly
// (fftsolve.hip).  Expression order follows the reference literally; with
// -ffp-contract=off both users give the same bits.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace gev_prep {

struct Nb {
    int x, y, z, xm, xp, ym, yp, zm, zp;
};

__device__ __forceinline__ Nb nb_of(int x, int y, int z, int N) {
    Nb c;
    c.x = x;
    c.y = y;
    c.z = z;
    c.xm = x == 0 ? N - 1 : x - 1;
    c.xp = x == N - 1 ? 0 : x + 1;
    c.ym = y == 0 ? N - 1 : y - 1;
    c.yp = y == N - 1 ? 0 : y + 1;
    c.zm = z == 0 ? N - 1 : z - 1;
    c.zp = z == N - 1 ? 0 : z + 1;
    return c;
}

__device__ __forceinline__ int64_t L(int N, int x, int y, int z) {
    return (int64_t)x + (int64_t)N * ((int64_t)y + (int64_t)N * z);
}

// prepareFTsource (2), gevolution.hpp:169-192: the new source value at site i
// (phi stored as F: double, or float in the FP32 form; arithmetic in double)
template <typename F>
__device__ __forceinline__ double prep_scalar(const F *__restrict__ phi, double chi_i, double src_i,
                                              const Nb &c, int64_t i, int N, double bg, double coeff,
                                              double coeff2, double coeff3) {
    const double p = phi[i];
    const double px = phi[L(N, c.xp, c.y, c.z)], mx = phi[L(N, c.xm, c.y, c.z)];
    const double py = phi[L(N, c.x, c.yp, c.z)], my = phi[L(N, c.x, c.ym, c.z)];
    const double pz = phi[L(N, c.x, c.y, c.zp)], mz = phi[L(N, c.x, c.y, c.zm)];
    double r = coeff2 * (src_i - bg);
    r *= 1. - 2. * p;
    r += 0.125 * (mx - px) * (mx - px);
    r += 0.125 * (my - py) * (my - py);
    r += 0.125 * (mz - pz) * (mz - pz);
    r += (coeff3 - coeff) * p - coeff3 * chi_i;
    return r;
}

// The terms of prepareFTsource (1), gevolution.hpp:56-147, of one component
// with the deposited value t: i = j from phi above and below along i, i != j
// from phi on the plaquette's corners.
__device__ __forceinline__ double prep_diag(double t, double up, double dn, double coeff) {
    double s = coeff * t;
    s += 0.5 * (up - dn) * (up - dn);
    return s;
}
__device__ __forceinline__ double prep_off(double t, double p, double pa, double pb, double pab, double coeff) {
    double s = coeff * t;
    s += pa * pb - p * pab;
    s += 0.5 * p * p;
    s -= 0.5 * pa * pa;
    s -= 0.5 * pb * pb;
    s += 0.5 * pab * pab;
    return s;
}
// ... in the FP32 form: the same terms over the float fields, evaluated in float
__device__ __forceinline__ float prep_diag(float t, float up, float dn, float coeff) {
    return coeff * t + 0.5f * (up - dn) * (up - dn);
}
__device__ __forceinline__ float prep_off(float t, float p, float pa, float pb, float pab, float coeff) {
    const float hp = 0.5f * p * p, ha = 0.5f * pa * pa, hb = 0.5f * pb * pb;
    return coeff * t + (pa * pb - p * pab) + hp - ha - hb + 0.5f * pab * pab;
}

// S[6] (order 00,01,02,11,12,22) from the deposited T[6] at site i (F: the
// field element, and the type the stencils are evaluated in)
template <typename F>
__device__ __forceinline__ void prep_tensor(const F *__restrict__ phi, const F T[6], const Nb &c, int64_t i, int N,
                                            F coeff, F S[6]) {
    const F p = phi[i];
    const F px = phi[L(N, c.xp, c.y, c.z)], mx = phi[L(N, c.xm, c.y, c.z)];
    const F py = phi[L(N, c.x, c.yp, c.z)], my = phi[L(N, c.x, c.ym, c.z)];
    const F pz = phi[L(N, c.x, c.y, c.zp)], mz = phi[L(N, c.x, c.y, c.zm)];
    const F pxy = phi[L(N, c.xp, c.yp, c.z)];
    const F pxz = phi[L(N, c.xp, c.y, c.zp)];
    const F pyz = phi[L(N, c.x, c.yp, c.zp)];
    S[0] = prep_diag(T[0], px, mx, coeff);
    S[3] = prep_diag(T[3], py, my, coeff);
    S[5] = prep_diag(T[5], pz, mz, coeff);
    S[1] = prep_off(T[1], p, px, py, pxy, coeff);
    S[2] = prep_off(T[2], p, px, pz, pxz, coeff);
    S[4] = prep_off(T[4], p, py, pz, pyz, coeff);
}

// one component of it (q in the order above, the same for a whole wavefront)
template <typename F>
__device__ __forceinline__ F prep_tensor_one(const F *__restrict__ phi, F t, const Nb &c, int64_t i, int N, F coeff,
                                             int q) {
    const F p = phi[i];
    switch (q) {
    case 0: return prep_diag(t, phi[L(N, c.xp, c.y, c.z)], phi[L(N, c.xm, c.y, c.z)], coeff);
    case 3: return prep_diag(t, phi[L(N, c.x, c.yp, c.z)], phi[L(N, c.x, c.ym, c.z)], coeff);
    case 5: return prep_diag(t, phi[L(N, c.x, c.y, c.zp)], phi[L(N, c.x, c.y, c.zm)], coeff);
    case 1:
        return prep_off(t, p, phi[L(N, c.xp, c.y, c.z)], phi[L(N, c.x, c.yp, c.z)], phi[L(N, c.xp, c.yp, c.z)], coeff);
    case 2:
        return prep_off(t, p, phi[L(N, c.xp, c.y, c.z)], phi[L(N, c.x, c.y, c.zp)], phi[L(N, c.xp, c.y, c.zp)], coeff);
    default:
        return prep_off(t, p, phi[L(N, c.x, c.yp, c.z)], phi[L(N, c.x, c.y, c.zp)], phi[L(N, c.x, c.yp, c.zp)], coeff);
    }
}

}  // namespace gev_prep
