// fft.hip -- 3D real-to-complex / complex-to-real FFT for one box, replacing
// LATfield2's PlanFFT<Cplx>::execute over FFTW3 (main.cpp:238-246, 477, 488,
// 544, 563, 575, 593).  Unnormalised in both directions, forward sign -1, so
// backward(forward(f)) = N^3 f (manual.pdf sec. 4, p.14).
//
// Layout: real fields are N^3 (x fastest).  k fields are [kz][ky][kx] with kx
// in [0, N/2] stored in rows of pitch P = kpitch(N) complexes.
//
// A 3D transform is three passes, each one HBM read + one HBM write:
//   forward : r2c along x (real rows -> k rows)      k_r2c_x
//             c2c along y, in place                   k_c2c_cols
//             c2c along z, in place                   k_c2c_cols
//   backward: c2c along z (k field -> scratch)        k_c2c_cols
//             c2c along y, in place on scratch        k_c2c_cols
//             c2r along x (scratch -> real rows)      k_c2r_x
// so the backward transform leaves its k input intact (BiFT is state,
// main.cpp:586/593).
//
// Inside a pass a workgroup stages a tile in LDS and runs a Stockham
// auto-sort FFT with compile-time radix plan (8, then 4, 2, 3).  The x passes
// use the half-length complex transform: z[n] = x[2n] + i x[2n+1].  The
// strided passes load W consecutive columns (W complexes = 128 bytes per row
// in FP64) so every global access is a full cache line.
#include <algorithm>

#include "gev_internal.h"
#include "fft_core.h"

namespace {

using namespace gev_fft;
constexpr int TPB = 256;

// Components (and boxes of a batch) of one launch, in blockIdx.z: component
// fastest; cs / bs: elements from one component / box to the next.
struct Comps {
    int nc;
    int64_t in_cs, in_bs, out_cs, out_bs;
    __device__ __forceinline__ int comp() const { return (int)blockIdx.z % nc; }
    __device__ __forceinline__ int box() const { return (int)blockIdx.z / nc; }
    __device__ __forceinline__ int64_t in_offset() const { return box() * in_bs + comp() * in_cs; }
    __device__ __forceinline__ int64_t out_offset() const { return box() * out_bs + comp() * out_cs; }
};

// ---------------------------------------------------------------- kernels

// r2c along x: nrows real rows of N -> nrows k rows (pitch P) of N/2+1.
template <typename T, int N>
__global__ __launch_bounds__(TPB) void k_r2c_x(const T *__restrict__ in,
                                               typename cplx_of<T>::type *__restrict__ out, int P,
                                               int64_t nrows,
                                               const typename cplx_of<T>::type *__restrict__ twN,
                                               Comps cc, gev::Batch bt) {
    using C = typename cplx_of<T>::type;
    if (!gev::box_on(bt, cc.box())) return;
    in += cc.in_offset();
    out += cc.out_offset();
    constexpr int M = N / 2;
    constexpr int LINES = x_lines<N>();
    __shared__ C buf[LINES * xstride<M>()];
    __shared__ C tw[M];
    const int64_t row0 = (int64_t)blockIdx.x * LINES;
    for (int t = threadIdx.x; t < M; t += TPB) tw[t] = twN[2 * t];
    {
        // all loads of this thread in flight before the first LDS write
        constexpr int PER = (LINES * M + TPB - 1) / TPB;
        C v[PER];
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int idx = threadIdx.x + k * TPB;
            const int line = idx / M, n = idx % M;
            const int64_t row = row0 + line;
            v[k] = mk2<C>(0, 0);
            if ((PER * TPB == LINES * M || idx < LINES * M) && row < nrows)
                v[k] = reinterpret_cast<const C *>(in + row * N)[n];
        }
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int idx = threadIdx.x + k * TPB;
            if (PER * TPB == LINES * M || idx < LINES * M) buf[eaddr<M, LINES, false>(idx / M, idx % M)] = v[k];
        }
    }
    __syncthreads();
    stages<C, M, LINES, false, 1>(buf, tw);
    for (int idx = threadIdx.x; idx < LINES * (M + 1); idx += TPB) {
        const int line = idx / (M + 1), k = idx % (M + 1);
        const int64_t row = row0 + line;
        if (row >= nrows) continue;
        C A = buf[eaddr<M, LINES, false>(line, k == M ? 0 : k)];
        C B = cconj(buf[eaddr<M, LINES, false>(line, k == 0 ? 0 : M - k)]);
        C E = mk2<C>((A.x + B.x) * (T)0.5, (A.y + B.y) * (T)0.5);
        C D = mk2<C>((A.x - B.x) * (T)0.5, (A.y - B.y) * (T)0.5);
        C O = mul_mi(D);
        out[row * P + k] = cadd(E, cmul(twN[k], O));
    }
}

// c2r along x: nrows k rows (pitch P) -> nrows real rows of N.  out_rest (may
// be null): where the components after the first go.  The imaginary
// parts of kx = 0 and kx = N/2 are ignored (FFTW / numpy c2r convention).
template <typename T, int N>
__global__ __launch_bounds__(TPB) void k_c2r_x(const typename cplx_of<T>::type *__restrict__ in,
                                               T *__restrict__ out, int P, int64_t nrows,
                                               const typename cplx_of<T>::type *__restrict__ twN,
                                               T *__restrict__ out_rest, Comps cc, gev::Batch bt) {
    using C = typename cplx_of<T>::type;
    if (!gev::box_on(bt, cc.box())) return;
    in += cc.in_offset();
    if (out_rest && cc.comp() > 0) out = out_rest + cc.box() * cc.out_bs + (int64_t)(cc.comp() - 1) * cc.out_cs;
    else out += cc.out_offset();
    constexpr int M = N / 2;
    constexpr int LINES = x_lines<N>();
    __shared__ C buf[LINES * xstride<M>()];
    __shared__ C tw[M];
    const int64_t row0 = (int64_t)blockIdx.x * LINES;
    for (int t = threadIdx.x; t < M; t += TPB) tw[t] = twN[2 * t];
    {
        // all loads of this thread in flight before the first LDS write
        constexpr int PER = (LINES * M + TPB - 1) / TPB;
        C xa[PER], xb[PER], wk[PER];
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const int idx = threadIdx.x + j * TPB;
            const int line = idx / M, k = idx % M;
            const int64_t row = row0 + line;
            xa[j] = xb[j] = wk[j] = mk2<C>(0, 0);
            if ((PER * TPB == LINES * M || idx < LINES * M) && row < nrows) {
                xa[j] = in[row * P + k];
                xb[j] = in[row * P + (M - k)];
                wk[j] = twN[k];
            }
        }
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const int idx = threadIdx.x + j * TPB;
            if (!(PER * TPB == LINES * M || idx < LINES * M)) continue;
            const int k = idx % M;
            C Xk = xa[j], Xm = xb[j];
            if (k == 0) {
                Xk.y = 0;
                Xm.y = 0;
            }
            C S = cadd(Xk, cconj(Xm));
            C D = csub(Xk, cconj(Xm));
            C Z = cadd(S, mul_pi(cmul(cconj(wk[j]), D)));
            buf[eaddr<M, LINES, false>(idx / M, k)] = cconj(Z);  // inverse transform through the forward one
        }
    }
    __syncthreads();
    stages<C, M, LINES, false, 1>(buf, tw);
    for (int idx = threadIdx.x; idx < LINES * M; idx += TPB) {
        const int line = idx / M, n = idx % M;
        const int64_t row = row0 + line;
        if (row >= nrows) continue;
        C z = cconj(buf[eaddr<M, LINES, false>(line, n)]);
        reinterpret_cast<C *>(out + row * N)[n] = z;
    }
}

// c2c along a strided axis.  Column c = (outer index, kx0 + w): elements at
// in[outer*os + kx + e*es], e < N.  INV = backward (sign +1).  RB: the
// tile's row bytes (0: the form's default; every column is transformed the
// same way whatever the tile).  blockIdx.z: component (fastest) and box.
//
// Bound by HBM and how it takes the pattern (128-byte pieces of rows 4 KB
// apart, read and written): 2.16 GB in 0.46 ms at 512^3 (FP64, 4.7 TB/s of
// the 5.7 a plain copy reaches; 0.48 with the first and last stage through
// LDS as well), 1.08 GB in 0.22 ms (FP32; 0.24).  Measured no faster at
// 512^3: workgroups that walk several tiles with the next one's loads in
// flight (0.51), 256-byte rows (0.48, one workgroup per CU), 512 threads.
template <typename T, int N, bool INV, int RB = 0>
__global__ __launch_bounds__((col_tpb<T, N, RB>()), 2) void k_c2c_cols(const typename cplx_of<T>::type *in,
                                                  typename cplx_of<T>::type *out, int H,
                                                  int64_t es, int64_t os,
                                                  const typename cplx_of<T>::type *__restrict__ twN,
                                                  int ntx, Comps cc, gev::Batch bt) {
    using C = typename cplx_of<T>::type;
    constexpr int TPB = col_tpb<T, N, RB>();
    if (!gev::box_on(bt, cc.box())) return;
    in += cc.in_offset();
    out += cc.out_offset();
    constexpr int W = col_tile<T, N, RB>();
    using Tile = ColumnTile<C, N, W, TPB>;
    __shared__ C buf[Tile::SINGLE ? 1 : N * W];
    __shared__ C tw[Tile::SINGLE ? 1 : N];
    if (!Tile::SINGLE)
        for (int t = threadIdx.x; t < N; t += TPB) tw[t] = twN[t];
    // XCD-aware order: workgroup ids go round-robin over the 8 XCDs, so each
    // XCD walks a run of neighbouring tiles
    int l = blockIdx.x;
    if (gridDim.x % 8 == 0) l = (l % 8) * (gridDim.x / 8) + l / 8;
    const int kx0 = (l % ntx) * W, w = Tile::column();
    const int64_t base = (int64_t)(l / ntx) * os + kx0;
    // this thread's byte offset from a tile's element eu (below 2^32: N / 8 rows)
    const uint32_t off = (uint32_t)(((int64_t)Tile::ev() * es + w) * (int64_t)sizeof(C));
    const bool ok = kx0 + w < H;
    Tile tile;
    tile.load([&](int eu) {
        C x = mk2<C>(0, 0);
        if (ok) x = *reinterpret_cast<const C *>(reinterpret_cast<const char *>(in + base + eu * es) + off);
        return x;
    });
    auto store = [&](int eu, C x) {
        if (ok) *reinterpret_cast<C *>(reinterpret_cast<char *>(out + base + eu * es) + off) = INV ? cconj(x) : x;
    };
    if constexpr (Tile::SINGLE) {
        tile.template finish_single<INV>(store);
    } else {
        tile.template first<INV>(buf);
        __syncthreads();
        Tile::finish(buf, tw, store);
    }
}

// Timer names of a pass launched over n components (n <= MAXC): the plain
// name for one, name[n] for several (the per-launch byte count scales by n).
constexpr int MAXC = 6;
enum { P_R2C_X, P_C2C_Y, P_C2C_Z, P_C2C_Z_INV, P_C2C_Y_INV, P_C2R_X };
const char *pass_name(int pass, int n) {
#define GEV_NAMES(s) {s, s "[2]", s "[3]", s "[4]", s "[5]", s "[6]"}
    static const char *const names[6][MAXC] = {GEV_NAMES("fft_r2c_x"),     GEV_NAMES("fft_c2c_y"),
                                               GEV_NAMES("fft_c2c_z"),     GEV_NAMES("fft_c2c_z_inv"),
                                               GEV_NAMES("fft_c2c_y_inv"), GEV_NAMES("fft_c2r_x")};
#undef GEV_NAMES
    return names[pass][n - 1];
}

// One strided pass (axis: 0 = y, 1 = z) over nc components (cs elements
// apart) of nb boxes (bs apart) with the context's tile for that axis:
// ctx->col_rb[axis] row bytes (0: the default).  The row variants exist for
// N <= 256, the grids batches run.
template <typename T, int N, bool INV, int RB>
void launch_cols_rb(gev_ctx *ctx, int axis, int nc, unsigned nb, const typename cplx_of<T>::type *in,
                    typename cplx_of<T>::type *out, const typename cplx_of<T>::type *tw, int64_t cs, int64_t bs,
                    const gev::Batch &bt) {
    constexpr int W = col_tile<T, N, RB>();
    const int H = N / 2 + 1, ntx = (H + W - 1) / W;
    const int64_t P = ctx->P, es = axis == 0 ? P : P * N, os = axis == 0 ? P * N : P;
    hipLaunchKernelGGL((k_c2c_cols<T, N, INV, RB>), dim3(ntx * N, 1, nc * nb), dim3(col_tpb<T, N, RB>()), 0,
                       ctx->stream, in, out, H, es, os, tw, ntx, Comps{nc, cs, bs, cs, bs}, bt);
}

template <typename T, int N, bool INV>
void launch_cols(gev_ctx *ctx, int axis, int nc, unsigned nb, const typename cplx_of<T>::type *in,
                 typename cplx_of<T>::type *out, const typename cplx_of<T>::type *tw, int64_t cs, int64_t bs,
                 const gev::Batch &bt) {
    const int rb = N <= 256 ? ctx->col_rb[axis] : 0;
    if constexpr (N <= 256) {
        if (rb == 64) return launch_cols_rb<T, N, INV, 64>(ctx, axis, nc, nb, in, out, tw, cs, bs, bt);
        if (rb == 256) return launch_cols_rb<T, N, INV, 256>(ctx, axis, nc, nb, in, out, tw, cs, bs, bt);
    }
    launch_cols_rb<T, N, INV, 0>(ctx, axis, nc, nb, in, out, tw, cs, bs, bt);
}

// Components that share one launch of a strided pass: all of them, unless one
// component alone is about a GB.  Small grids gain the launches (64^3: six y
// passes 45 -> 9 us, a GR cycle 207 -> 178 us), larger ones the tails (256^3
// FP32: 32 -> 25 us per component; 512^3 FP32 229 -> 224, 384^3 FP64 equal);
// at 512^3 FP64 one launch per component is the faster one (465 against 473 us).
template <typename T, int N> constexpr int cols_per_launch(int ncomp) {
    return (int64_t)N * N * (N / 2 + 1) * 2 * (int64_t)sizeof(T) < (600ll << 20) ? ncomp : 1;
}

template <typename T, int N, bool INV>
void cols_pass(gev_ctx *ctx, int pass, int axis, int ncomp, unsigned nb, const typename cplx_of<T>::type *in,
               typename cplx_of<T>::type *out, const typename cplx_of<T>::type *tw, int64_t cs, int64_t bs,
               const gev::Batch &bt) {
    const int step = cols_per_launch<T, N>(ncomp);
    for (int c = 0; c < ncomp; c += step) {
        gev::ScopedTimer t(ctx, pass_name(pass, step));
        launch_cols<T, N, INV>(ctx, axis, step, nb, in + c * cs, out + c * cs, tw, cs, bs, bt);
    }
}

// passes: bit 0 = x (r2c), bit 1 = y, bit 2 = z, up to MAXC components pass
// by pass.  The x pass is one launch over the components (and the boxes of a
// batch).
template <typename T, int N>
int run_forward(gev_ctx *ctx, const T *real, typename cplx_of<T>::type *k, int ncomp,
                const typename cplx_of<T>::type *tw, int passes, const gev::Batch &bt) {
    using C = typename cplx_of<T>::type;
    const int P = ctx->P;
    const int64_t nrows = (int64_t)N * N;
    const int64_t n3v = (int64_t)N * N * N, nkv = (int64_t)P * N * N;
    constexpr int LINES = x_lines<N>();
    const bool batch = bt.cyc != nullptr;
    const unsigned nb = batch ? (unsigned)ctx->nbox : 1u;
    const int64_t rs = batch ? ctx->stride / (int64_t)sizeof(T) : 0, ks = batch ? ctx->stride / (int64_t)sizeof(C) : 0;
    for (int c0 = 0; c0 < ncomp; c0 += MAXC) {
        const int nc = ncomp - c0 < MAXC ? ncomp - c0 : MAXC;
        C *const kc = k + c0 * nkv;
        if (passes & 1) {
            gev::ScopedTimer t(ctx, pass_name(P_R2C_X, nc));
            hipLaunchKernelGGL((k_r2c_x<T, N>), dim3(gev::grid_for(nrows, LINES), 1, nc * nb), dim3(TPB), 0,
                               ctx->stream, real + c0 * n3v, kc, P, nrows, tw, Comps{nc, n3v, rs, nkv, ks}, bt);
        }
        if (passes & 2) cols_pass<T, N, false>(ctx, P_C2C_Y, 0, nc, nb, kc, kc, tw, nkv, ks, bt);
        if (passes & 4) cols_pass<T, N, false>(ctx, P_C2C_Z, 1, nc, nb, kc, kc, tw, nkv, ks, bt);
    }
    return gev::check_hip(ctx, hipGetLastError(), "fft forward launch");
}

// from_y: k already went through the inverse z pass; the remaining passes run
// in place on k itself (tmp unused), the x pass as one launch over the
// components (up to MAXC); real_rest (may be null) takes the components after
// the first.  Otherwise every component goes z, y, x through tmp.
template <typename T, int N>
int run_backward(gev_ctx *ctx, const typename cplx_of<T>::type *k, T *real, T *real_rest, int ncomp,
                 typename cplx_of<T>::type *tmp, const typename cplx_of<T>::type *tw, bool from_y,
                 const gev::Batch &bt) {
    using C = typename cplx_of<T>::type;
    const int P = ctx->P;
    const int64_t nrows = (int64_t)N * N;
    const int64_t n3v = (int64_t)N * N * N, nkv = (int64_t)P * N * N;
    constexpr int LINES = x_lines<N>();
    const bool batch = bt.cyc != nullptr;
    const unsigned nb = batch ? (unsigned)ctx->nbox : 1u;
    const int64_t rs = batch ? ctx->stride / (int64_t)sizeof(T) : 0, ks = batch ? ctx->stride / (int64_t)sizeof(C) : 0;
    auto c2r = [&](const C *from, T *to, T *to_rest, int nc) {
        gev::ScopedTimer t(ctx, pass_name(P_C2R_X, nc));
        hipLaunchKernelGGL((k_c2r_x<T, N>), dim3(gev::grid_for(nrows, LINES), 1, nc * nb), dim3(TPB), 0, ctx->stream,
                           from, to, P, nrows, tw, to_rest, Comps{nc, nkv, ks, n3v, rs}, bt);
    };
    if (from_y) {
        if (ncomp > MAXC) return gev::fail(ctx, GEV_EINVAL, "too many components in one transform");
        auto *kk = const_cast<C *>(k);
        cols_pass<T, N, true>(ctx, P_C2C_Y_INV, 0, ncomp, nb, kk, kk, tw, nkv, ks, bt);
        c2r(kk, real, real_rest, ncomp);
        return gev::check_hip(ctx, hipGetLastError(), "fft backward launch");
    }
    for (int c = 0; c < ncomp; c++) {
        cols_pass<T, N, true>(ctx, P_C2C_Z_INV, 1, 1, nb, k + c * nkv, tmp, tw, nkv, ks, bt);
        cols_pass<T, N, true>(ctx, P_C2C_Y_INV, 0, 1, nb, tmp, tmp, tw, nkv, ks, bt);
        c2r(tmp, real + c * n3v, nullptr, 1);
    }
    return gev::check_hip(ctx, hipGetLastError(), "fft backward launch");
}

}  // namespace

namespace gev {

bool fft_size_supported(int N) {
    switch (N) {
#define CASE(n) case n:
        GEV_FFT_SIZES(CASE)
#undef CASE
        return true;
    default:
        return false;
    }
}

// the passes in the context's form: FP64, or FP32 (float fields, float2 k fields)
static int forward(gev_ctx *ctx, const double *real, double2 *kfield, int ncomp, int passes,
                   const Batch &bt = Batch{}) {
    switch (ctx->N) {
#define CASE(n)                                                                                                  \
    case n:                                                                                                      \
        return ctx->fp32 ? run_forward<float, n>(ctx, fld<float>(real), cfld<float2>(kfield), ncomp, ctx->twiddle_f, \
                                                 passes, bt)                                                     \
                         : run_forward<double, n>(ctx, real, kfield, ncomp, ctx->twiddle, passes, bt);
        GEV_FFT_SIZES(CASE)
#undef CASE
    default:
        return fail(ctx, GEV_EINVAL, "unsupported FFT size");
    }
}

static int backward(gev_ctx *ctx, const double2 *kfield, double *real, double *real_rest, int ncomp, bool from_y,
                    const Batch &bt = Batch{}) {
    switch (ctx->N) {
#define CASE(n)                                                                                             \
    case n:                                                                                                 \
        return ctx->fp32 ? run_backward<float, n>(ctx, cfld<float2>(kfield), fld<float>(real), fld<float>(real_rest), \
                                                  ncomp, cfld<float2>(ctx->fft_tmp), ctx->twiddle_f, from_y, bt) \
                         : run_backward<double, n>(ctx, kfield, real, real_rest, ncomp, ctx->fft_tmp,       \
                                                   ctx->twiddle, from_y, bt);
        GEV_FFT_SIZES(CASE)
#undef CASE
    default:
        return fail(ctx, GEV_EINVAL, "unsupported FFT size");
    }
}

int fft_forward(gev_ctx *ctx, const double *real, double2 *kfield, int ncomp) {
    return forward(ctx, real, kfield, ncomp, 7);
}

int fft_backward(gev_ctx *ctx, const double2 *kfield, double *real, int ncomp) {
    return backward(ctx, kfield, real, nullptr, ncomp, false);
}

int fft_forward_xy(gev_ctx *ctx, const double *real, double2 *kfield, int ncomp, const Batch &bt) {
    return forward(ctx, real, kfield, ncomp, 3, bt);
}

int fft_forward_y(gev_ctx *ctx, double2 *kfield, int ncomp, const Batch &bt) {
    return forward(ctx, nullptr, kfield, ncomp, 2, bt);
}

int fft_forward_z(gev_ctx *ctx, double2 *kfield, int ncomp, const Batch &bt) {
    return forward(ctx, nullptr, kfield, ncomp, 4, bt);
}

int fft_backward_yx(gev_ctx *ctx, double2 *kfield, double *real, int ncomp, const Batch &bt, double *real_rest) {
    return backward(ctx, kfield, real, real_rest, ncomp, true, bt);
}

}  // namespace gev
