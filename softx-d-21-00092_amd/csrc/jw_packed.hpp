// jw_packed.hpp -- the unfused passes of the generator-basis step, templated on
// the storage type C (double2: FP64 form, float2: mixed form): the 2-D FFT
// row and column passes and the per-site kernels (noise, kernel multiply,
// U xi U^dagger, update).  Site algebra is FP64 in both forms, but for U xi U^dagger of
// the mixed form at N = 8192.  Used where the fused passes are not (N outside 64..2048, the LINEAR kernel's 9-component
// transforms, jw_set_fused(ctx, 0)).
#pragma once

#include "jw_common.hpp"
#include "jw_engine.hpp"

namespace jw {

// ===========================================================================
// FFT passes
// ===========================================================================
// Rows per workgroup (at most N: a workgroup never reaches past its plane) and
// columns per workgroup (at most N), each a divisor of N.  Column strips are
// as wide as about 150 KB of LDS allows (at most 16 columns).
template <int N, typename C = double2>
struct RowCfg {
    static constexpr int RPW0 = (N >= 1024) ? 1 : (1024 / N);
    static constexpr int RPW = RPW0 < N ? RPW0 : N;
    static constexpr int ELEMS = RPW * N;
    static constexpr int NT = (ELEMS / 8 < 64) ? 64 : ((ELEMS / 8 > 1024) ? 1024 : ELEMS / 8);
    static_assert(RPW >= 1 && RPW <= N && N % RPW == 0, "row tiling must divide the plane");
};
template <int N, typename C = double2>
struct ColCfg {
    static constexpr int BUDGET = 150 * 1024;
    static constexpr int W1 = BUDGET / (padded<N, 3>::value * (int)sizeof(C));
    static constexpr int W0 = W1 >= 16 ? 16 : (W1 >= 8 ? 8 : (W1 >= 4 ? 4 : (W1 >= 2 ? 2 : 1)));
    static constexpr int W = W0 < N ? W0 : N;
    static constexpr int ELEMS = W * N;
    static constexpr int NT = (ELEMS / 8 < 64) ? 64 : ((ELEMS / 8 > 1024) ? 1024 : ELEMS / 8);
    static_assert(W >= 1 && W <= N && N % W == 0, "column tiling must divide the plane");
};

template <int N, int DIR, typename C>
__global__ __launch_bounds__((RowCfg<N, C>::NT)) void k_fft_rows(C* __restrict__ data, size_t plane_stride,
                                                              const C* __restrict__ tw, double scale) {
    typedef typename scalar_of<C>::type T;
    using G = RowCfg<N, C>;
    constexpr int PN = padded<N, 4>::value;            // padded row length in LDS
    __shared__ C lds[G::RPW * PN];
    const int tid = threadIdx.x;
    C* base = data + blockIdx.y * plane_stride + (size_t)blockIdx.x * G::ELEMS;
    for (int i = tid; i < G::ELEMS; i += G::NT) lds[lpos<1, PN, 4>(i % N, i / N)] = base[i];
    __syncthreads();
    lds_fft<N, G::RPW, 1, PN, G::NT, DIR, 4>(lds, tw, tid);
    for (int i = tid; i < G::ELEMS; i += G::NT) base[i] = cscale(lds[lpos<1, PN, 4>(i % N, i / N)], (T)scale);
}

template <int N, int DIR, typename C>
__global__ __launch_bounds__((ColCfg<N, C>::NT)) void k_fft_cols(C* __restrict__ data, size_t plane_stride,
                                                              const C* __restrict__ tw, double scale) {
    typedef typename scalar_of<C>::type T;
    using G = ColCfg<N, C>;
    __shared__ C lds[padded<N, 3>::value * G::W];
    const int tid = threadIdx.x;
    C* base = data + blockIdx.y * plane_stride + (size_t)blockIdx.x * G::W;
    for (int i = tid; i < G::ELEMS; i += G::NT)
        lds[lpos<G::W, 1, 3>(i / G::W, i % G::W)] = base[(size_t)(i / G::W) * N + (i % G::W)];
    __syncthreads();
    lds_fft<N, G::W, G::W, 1, G::NT, DIR, 3>(lds, tw, tid);
    for (int i = tid; i < G::ELEMS; i += G::NT)
        base[(size_t)(i / G::W) * N + (i % G::W)] = cscale(lds[lpos<G::W, 1, 3>(i / G::W, i % G::W)], (T)scale);
}

// From N = 64 on the FP64 transforms run in registers (jw_regfft.hpp), T threads a row or a
// column, and LDS is touched by one exchange over the workgroup and one inside a wave
// instead of by every radix-8 stage; a column strip is a 64-byte segment wide.  Bound by
// memory: nine planes of FP64 at N = 512 (2 x 38 MB), rows 17.0 -> 16.8 us, columns 22.0 ->
// 14.5; four at N = 8192 8.9 -> 6.6 ms (columns).
template <int N, int DIR, typename C>
__global__ __launch_bounds__(RowN<N>::NT) void k_fft_rows_reg(C* __restrict__ data, size_t plane_stride,
                                                              const C* __restrict__ tw, double scale) {
    typedef typename scalar_of<C>::type T;
    typedef RegFft<N> F;
    __shared__ C lds[RowN<N>::RPW * RowT<N, C>::PL];
    C* row = data + blockIdx.y * plane_stride + ((size_t)blockIdx.x * RowN<N>::RPW + threadIdx.x / F::T) * N;
    C* buf = lds + (threadIdx.x / F::T) * RowT<N, C>::PL;
    const int j = threadIdx.x % F::T;
    C v[F::PT];
    auto site = [&](int r) { return opaque_v(j) + r * F::T; };
    auto freq = [&](int q) {
        const int i = opaque_v(j);
        return reg_freq<N>(i / F::N3, i % F::N3, 0) + reg_freq_q<N>(q);
    };
#pragma unroll
    for (int r = 0; r < F::PT; r++) v[r] = row[DIR < 0 ? site(r) : freq(r)];
    if constexpr (DIR < 0) reg_fft_fwd<N, 1, true>(v, buf, tw_fft(tw), opaque_v(j));
    else reg_fft_inv<N, 1, true>(v, buf, tw_fft(tw), opaque_v(j));
#pragma unroll
    for (int r = 0; r < F::PT; r++) row[DIR < 0 ? freq(r) : site(r)] = cscale(v[r], (T)scale);
}

// inverse row transforms of tiled planes (Tile) into row-major ones; the rows of a tile
// run on one XCD.  Bound by memory; four FP32 planes at N = 8192 1.13 ms (1.05 in place on
// row-major ones, whose column passes took 6.2 ms longer a step).
template <int N, typename C>
__global__ __launch_bounds__(RowN<N>::NT) void k_rows_inv_tiled(C* __restrict__ out, const C* __restrict__ in, size_t V,
                                                                const C* __restrict__ tw) {
    typedef RegFft<N> F;
    __shared__ C lds[RowN<N>::RPW * RowT<N, C>::PL];
    const int x = xcd_strip(blockIdx.x, N / RowN<N>::RPW) * RowN<N>::RPW + threadIdx.x / F::T;
    C* buf = lds + (threadIdx.x / F::T) * RowT<N, C>::PL;
    const int j = threadIdx.x % F::T;
    C v[F::PT];
    const C* src = in + blockIdx.y * V + Tile<N, C>::at(x, reg_freq<N>(j / F::N3, j % F::N3, 0));
#pragma unroll
    for (int q = 0; q < F::PT; q++) v[q] = src[reg_freq_q<N>(q) * Tile<N, C>::TR];
    reg_fft_inv<N, 1, true>(v, buf, tw_fft(tw), opaque_v(j));
    C* dst = out + blockIdx.y * V + (size_t)x * N + j;
#pragma unroll
    for (int r = 0; r < F::PT; r++) dst[r * F::T] = v[r];
}

template <int N, int DIR, typename C>
__global__ __launch_bounds__((ColR<N, C>::NT)) void k_fft_cols_reg(C* __restrict__ data, size_t plane_stride,
                                                                   const C* __restrict__ tw, double scale) {
    typedef typename scalar_of<C>::type T;
    typedef RegFft<N> F;
    constexpr int W = ColR<N, C>::W;
    __shared__ C lds[ColR<N, C>::ELEMS];
    data += blockIdx.y * plane_stride + (size_t)xcd_strip(blockIdx.x, N / W) * W;
    auto site = [&]() { const int t = opaque_v((int)threadIdx.x); return (unsigned)(t / W * N + t % W); };
    auto freq = [&]() {
        const int t = opaque_v((int)threadIdx.x), j = t / W;
        return (unsigned)(reg_freq<N>(j / F::N3, j % F::N3, 0) * N + t % W);
    };
    constexpr size_t RS = (size_t)F::T * N;
    auto rq = [](int q) { return (size_t)reg_freq_q<N>(q) * N; };
    C v[F::PT];
    const unsigned o = DIR < 0 ? site() : freq();
#pragma unroll
    for (int r = 0; r < F::PT; r++) v[r] = (data + (DIR < 0 ? r * RS : rq(r)))[o];
    if constexpr (DIR < 0) reg_fft_fwd<N, W, true>(v, lds, tw_fft(tw), opaque_v((int)threadIdx.x));
    else reg_fft_inv<N, W, true>(v, lds, tw_fft(tw), opaque_v((int)threadIdx.x));
    const unsigned e = DIR < 0 ? freq() : site();
#pragma unroll
    for (int r = 0; r < F::PT; r++) (data + (DIR < 0 ? rq(r) : r * RS))[e] = cscale(v[r], (T)scale);
}

// REG: the transforms in registers.  The FP32 2-D transforms (the unfused sequence of the
// mixed form) and the row passes beside the 16-byte column strips keep the radix-8 passes in
// LDS: the 16- and 32-point factors' constants, rounded to FP32, cost more error there than
// the passes saved (rms of forward, multiply, inverse, LDS / registers: N = 1024 2.23e-7 /
// 2.29e-7, 2048 2.34e-7 / 2.41e-7, 4096 2.48e-7 / 2.59e-7; FP64 4.38e-16 / 4.11e-16,
// 4.57e-16 / 4.51e-16, 5.04e-16 / 4.69e-16).
template <int N, bool REG, typename C>
static hipError_t launch_rows(jw_ctx* c, C* p, int np, int dir, double scale, const C* tw) {
    KTimer t(c, K_FFT_ROWS);
    if constexpr (REG && N >= 64) {
        dim3 grid(N / RowN<N>::RPW, np), block(RowN<N>::NT);
        if (dir) hipLaunchKernelGGL((k_fft_rows_reg<N, -1, C>), grid, block, 0, c->stream, p, c->V, tw, scale);
        else hipLaunchKernelGGL((k_fft_rows_reg<N, +1, C>), grid, block, 0, c->stream, p, c->V, tw, scale);
    } else {
        using G = RowCfg<N, C>;
        dim3 grid(N / G::RPW, np);
        if (dir) hipLaunchKernelGGL((k_fft_rows<N, -1, C>), grid, dim3(G::NT), 0, c->stream, p, c->V, tw, scale);
        else hipLaunchKernelGGL((k_fft_rows<N, +1, C>), grid, dim3(G::NT), 0, c->stream, p, c->V, tw, scale);
    }
    return hipGetLastError();
}

template <int N, bool REG, typename C>
static hipError_t launch_cols(jw_ctx* c, C* p, int np, int dir, double scale, const C* tw) {
    KTimer t(c, K_FFT_COLS);
    if constexpr (REG && N >= 64) {
        dim3 grid(N / ColR<N, C>::W, np), block(ColR<N, C>::NT);
        if (dir) hipLaunchKernelGGL((k_fft_cols_reg<N, -1, C>), grid, block, 0, c->stream, p, c->V, tw, scale);
        else hipLaunchKernelGGL((k_fft_cols_reg<N, +1, C>), grid, block, 0, c->stream, p, c->V, tw, scale);
    } else {
        using G = ColCfg<N, C>;
        dim3 grid(N / G::W, np);
        if (dir) hipLaunchKernelGGL((k_fft_cols<N, -1, C>), grid, dim3(G::NT), 0, c->stream, p, c->V, tw, scale);
        else hipLaunchKernelGGL((k_fft_cols<N, +1, C>), grid, dim3(G::NT), 0, c->stream, p, c->V, tw, scale);
    }
    return hipGetLastError();
}

#define JW_SIZE_SWITCH(N, CALL)                         \
    switch (N) {                                        \
        case 4: return CALL(4);                         \
        case 8: return CALL(8);                         \
        case 16: return CALL(16);                       \
        case 32: return CALL(32);                       \
        case 64: return CALL(64);                       \
        case 128: return CALL(128);                     \
        case 256: return CALL(256);                     \
        case 512: return CALL(512);                     \
        case 1024: return CALL(1024);                   \
        case 2048: return CALL(2048);                   \
        case 4096: return CALL(4096);                   \
        case 8192: return CALL(8192);                   \
        default: return hipErrorInvalidValue;           \
    }

template <typename C>
static const C* twiddles_of(const jw_ctx* c) {
    if constexpr (sizeof(C) == sizeof(double2)) return c->tw;
    else return c->twf;
}

template <typename C>
static hipError_t fft_rows_t(jw_ctx* c, C* planes, int nplanes, int dir, double scale) {
#define CALL_ROWS(n) launch_rows<n, sizeof(C) == sizeof(double2), C>(c, planes, nplanes, dir, scale, twiddles_of<C>(c))
    JW_SIZE_SWITCH(c->N, CALL_ROWS)
#undef CALL_ROWS
}

template <typename C>
static hipError_t fft_cols_t(jw_ctx* c, C* planes, int nplanes, int dir, double scale) {
#define CALL_COLS(n) launch_cols<n, sizeof(C) == sizeof(double2), C>(c, planes, nplanes, dir, scale, twiddles_of<C>(c))
    JW_SIZE_SWITCH(c->N, CALL_COLS)
#undef CALL_COLS
}

// unitary 2-D transform of nplanes planes: dir 1 -> exp(-i k.x), dir 0 -> exp(+i k.x),
// scaled by `scale` once (1/N for the reference's 1/sqrt(V))
template <typename C>
static hipError_t fft2d_t(jw_ctx* c, C* planes, int nplanes, int dir, double scale) {
    hipError_t e = fft_rows_t(c, planes, nplanes, dir, 1.0);
    if (e != hipSuccess) return e;
    return fft_cols_t(c, planes, nplanes, dir, scale);
}

// ===========================================================================
// generator-basis engine (packed planes)
//   Xi planes 0..3: (n0,n1),(n2,n3),(n4,n5),(n6,n7) of xi_x; planes 4..7: same for xi_y
//   Vv planes: the same layout for V_x, V_y;  ZA, ZB: 4 planes (A, B)
// ===========================================================================
template <typename C>
__global__ __launch_bounds__(256) void k_gen_noise_packed(C* __restrict__ Xi, size_t V, NoiseSrc ns,
                                                          const double* __restrict__ sa_pos) {
    typedef typename scalar_of<C>::type T;
    GRID_STRIDE(i, V) {
        T z[16];
        normals16_t(ns, i, z);
        const double s = sa_pos ? sa_pos[i] : 1.0;
#pragma unroll
        for (int p = 0; p < 4; p++) {
            Xi[p * V + i] = mkc<C>(z[4 * p] * s, z[4 * p + 2] * s);           // n_{2p}, n_{2p+1}
            Xi[(4 + p) * V + i] = mkc<C>(z[4 * p + 1] * s, z[4 * p + 3] * s); // m_{2p}, m_{2p+1}
        }
    }
}

// Z[p] = i (kx(k) X[p] + ky(k) Y[p]),  kx = -2 pi c pbarX / phat2, zero at k = 0;
// scale_inputs: X, Y *= sa(k) first (and written back) for per-mode correlated noise.
template <typename C>
__global__ __launch_bounds__(256) void k_kernel_mult_packed(C* __restrict__ Z, C* __restrict__ X, C* __restrict__ Y,
                                                            int N, int coupling, const double* __restrict__ q4,
                                                            const double* __restrict__ sb,
                                                            const double* __restrict__ sa, int scale_inputs) {
    typedef typename scalar_of<C>::type T;
    const size_t V = (size_t)N * N;
    GRID_STRIDE(i, V) {
        const int ix = (int)(i / N), iy = (int)(i % N);
        const double ph = q4[ix] + q4[iy];
        const double sc = (coupling == 0) ? sa[i] : 1.0;
        const double kxv = (i == 0) ? 0.0 : -2.0 * M_PI * sc * sb[ix] / ph;
        const double kyv = (i == 0) ? 0.0 : -2.0 * M_PI * sc * sb[iy] / ph;
        const double si = scale_inputs ? sa[i] : 1.0;
#pragma unroll
        for (int p = 0; p < 4; p++) {
            C x = X[p * V + i], y = Y[p * V + i];
            if (scale_inputs) {
                x = cscale(x, (T)si);
                y = cscale(y, (T)si);
                X[p * V + i] = x;
                Y[p * V + i] = y;
            }
            Z[p * V + i] = mkc<C>(-(kxv * x.y + kyv * y.y), kxv * x.x + kyv * y.x);   // i (kx x + ky y)
        }
    }
}

// U for the FP64 site algebra of the packed kernels: all nine planes, or (U6,
// the large-lattice step) rows 0 and 1 with row 2 rebuilt as conj(row 0 x row 1)
template <int U6, typename C>
__device__ __forceinline__ void load_u_d(m3& u, const C* __restrict__ U, size_t V, size_t i) {
#pragma unroll
    for (int k = 0; k < (U6 ? 6 : 9); k++) u.m[k] = to_d(U[k * V + i]);
    if constexpr (U6 != 0) {
        row2_of(u.m);
    }
}

template <typename C, int U6 = 0>
__global__ __launch_bounds__(256) void k_uxiu_packed(C* __restrict__ Vv, const C* __restrict__ U,
                                                     const C* __restrict__ Xi_pos, size_t V, NoiseSrc ns,
                                                     const double* __restrict__ sa_pos) {
    typedef typename scalar_of<C>::type T;
    GRID_STRIDE(i, V) {
        double hx[8], hy[8];
        if (Xi_pos) {
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const C a = Xi_pos[p * V + i], b = Xi_pos[(4 + p) * V + i];
                hx[2 * p] = a.x; hx[2 * p + 1] = a.y;
                hy[2 * p] = b.x; hy[2 * p + 1] = b.y;
            }
        } else {
            T z[16];
            normals16_t(ns, i, z);
            const double s = sa_pos ? sa_pos[i] : 1.0;
#pragma unroll
            for (int k = 0; k < 8; k++) { hx[k] = z[2 * k] * s; hy[k] = z[2 * k + 1] * s; }
        }
        m3 u;
        load_u_d<U6>(u, U, V, i);
        double vx[8], vy[8];
        uxiu_gen(u, hx, vx);
        uxiu_gen(u, hy, vy);
#pragma unroll
        for (int p = 0; p < 4; p++) {
            Vv[p * V + i] = mkc<C>(vx[2 * p], vx[2 * p + 1]);
            Vv[(4 + p) * V + i] = mkc<C>(vy[2 * p], vy[2 * p + 1]);
        }
    }
}

// whole: a call's last step leaves all nine planes there, in FP64 (U itself, or the field
// of a mixed call, whose own pass back, R 6 FP32 W 9 FP64, took 2.4 ms at N = 8192 after 2.5 here)
template <typename C, int U6 = 0>
__global__ __launch_bounds__(256) void k_update_packed(C* U, const C* __restrict__ ZA, const C* __restrict__ ZB, size_t V,
                                                       double ss, int reunit, cplx* whole) {
    GRID_STRIDE(i, V) {
        double ha[8], hb[8];
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const C a = ZA[p * V + i], b = ZB[p * V + i];
            ha[2 * p] = a.x; ha[2 * p + 1] = a.y;
            hb[2 * p] = b.x; hb[2 * p + 1] = b.y;
        }
        const m3 eb = exp_i_gen(hb, ss);
        const m3 ea = exp_i_gen(ha, -ss);
        m3 u;
        load_u_d<U6>(u, U, V, i);
        m3 r = mmul(mmul(eb, u), ea);
        if (reunit) r = su3_project(r);
        if (U6 && whole) {      // rows 0 and 1 as the storage type holds them
#pragma unroll
            for (int k = 0; k < 6; k++) r.m[k] = to_d(mkc<C>(r.m[k].x, r.m[k].y));
            row2_of(r.m);
#pragma unroll
            for (int k = 0; k < 9; k++) whole[k * V + i] = r.m[k];
        } else {
#pragma unroll
            for (int k = 0; k < (U6 ? 6 : 9); k++) U[k * V + i] = mkc<C>(r.m[k].x, r.m[k].y);
        }
    }
}

// the unfused step in either precision: noise, 2-D FFTs, kernel multiplies,
// U xi U^dagger, update (reunit: project U onto SU(3) after it)
template <typename C>
static hipError_t step_unfused_t(jw_ctx* c, C* U, C* Xi, C* Vv, C* ZA, C* ZB, const NoiseSrc& ns,
                                 const double* sa_pos, const double* sa_k, int kc, int corr, double ss, int reunit) {
    const size_t V = c->V;
    const double s = 1.0 / c->N;
    const unsigned g = grid_for(V, 256);
    hipError_t e;
#define JW_TRY(x) if ((e = (x)) != hipSuccess) return e
    {
        KTimer t(c, K_GEN_NOISE);
        hipLaunchKernelGGL(k_gen_noise_packed<C>, dim3(g), dim3(256), 0, c->stream, Xi, V, ns, sa_pos);
        JW_TRY(hipGetLastError());
    }
    JW_TRY(fft2d_t(c, Xi, 8, 1, s));
    {
        KTimer t(c, K_KMULT);
        hipLaunchKernelGGL(k_kernel_mult_packed<C>, dim3(g), dim3(256), 0, c->stream, ZA, Xi, Xi + 4 * V, c->N, kc,
                           c->q4, c->sb, sa_k, corr);
        JW_TRY(hipGetLastError());
    }
    JW_TRY(fft2d_t(c, ZA, 4, 0, s));
    if (corr) JW_TRY(fft2d_t(c, Xi, 8, 0, s));
    {
        KTimer t(c, K_UXIU);
        hipLaunchKernelGGL(k_uxiu_packed<C>, dim3(g), dim3(256), 0, c->stream, Vv, U, corr ? Xi : nullptr, V, ns,
                           sa_pos);
        JW_TRY(hipGetLastError());
    }
    JW_TRY(fft2d_t(c, Vv, 8, 1, s));
    {
        KTimer t(c, K_KMULT);
        hipLaunchKernelGGL(k_kernel_mult_packed<C>, dim3(g), dim3(256), 0, c->stream, ZB, Vv, Vv + 4 * V, c->N, kc,
                           c->q4, c->sb, sa_k, 0);
        JW_TRY(hipGetLastError());
    }
    JW_TRY(fft2d_t(c, ZB, 4, 0, s));
    {
        KTimer t(c, K_UPDATE);
        hipLaunchKernelGGL(k_update_packed<C>, dim3(g), dim3(256), 0, c->stream, U, ZA, ZB, V, ss, reunit, (cplx*)nullptr);
        JW_TRY(hipGetLastError());
    }
#undef JW_TRY
    return hipSuccess;
}


// ===========================================================================
// Large lattices (N = 4096, 8192): the fused column passes of jw_engine.hpp
// (forward column FFT, kernel multiply, inverse column FFT per strip;
// the momentum-space noise drawn there) with the row transforms and the site
// algebra as separate passes, since one lattice row of four planes no longer
// fits LDS (FP64 at N = 4096 needs 256 KB).  U is held as rows 0 and 1 (row 2
// rebuilt on load), as in the fused step.  Per step, in complex planes moved:
//   [position-space noise: noise W 8, forward row FFT R 8 W 8]
//   column A                     R 8 (0 drawn) W 4 (+8 correlated or drawn)
//   inverse row FFT of A         R 4 W 4   (after U xi U^dagger where A is in tiles)
//   correlated or drawn noise, k_row_uxiu_1p (not in FP64 at N = 8192):
//     inverse row FFT of xi~, U xi~ U^dagger, forward row FFT of V  R 20 W 8
//   otherwise: [inverse row FFT of xi~ R 8 W 8]
//     U xi U^dagger              R 6 (+8) W 8
//     forward row FFT of V       R 8 W 8
//   column B                     R 8 W 4
//   inverse row FFT of B         R 4 W 4
//   update                       R 14 W 6
// 88 planes with the noise drawn per mode (114 in FP64 at N = 8192),
// against 66 for the fused step of N <= 2048.  Column strips: k_col_reg on planes in
// natural order (layout 3 of its parameter), 16-byte row segments in FP32 at N = 8192, 32 at
// N = 4096, which writes tiles of 64 bytes (Tile) where row passes read; one plane at a
// time over 16-byte segments (BF = 32) in FP64 at N = 8192.
// ===========================================================================
// U xi~ U^dagger of the large-lattice step as one pass over a lattice row, where
// four planes of a row do not fit LDS: the four planes of a direction are in the
// registers of T threads each (jw_regfft.hpp), and every exchange goes through LDS
// for the real parts and then for the imaginary parts (4 N elements of 4 bytes:
// 132 KB at N = 8192).  The transformed planes are exchanged once more so that each
// thread holds the four of its own sites for V = U xi~ U^dagger (U as rows 0 and 1,
// read once per direction), and back.  In place of the inverse row FFT of xi~ (R 8 W 8),
// the site pass (R 14 W 8) and the forward row FFT of V (R 8 W 8): R 20 W 8.
// Bound by memory and by its own exchanges in turn (one workgroup a CU): FP32 at N = 8192
// 4.6 ms (10.7 GB; 5.0 from tiles), where a plane at a time through LDS stages took 7.7 ms.  Against the
// three passes, two steps at N = 4096 with drawn correlated noise: FP64 18.3 -> 15.5 ms, mixed
// 10.8 -> 10.0 (with FP64 products here as there: 4.3 ms a step, 4.2 with FP32 ones, which
// put a long step 5% further from FP64).  FP64 at N = 8192 fits neither LDS nor registers and keeps the three passes.
template <int N, typename C>
struct Row1P {
    typedef RegFft<N> F;
    typedef typename scalar_of<C>::type T;
    static constexpr int NT = 4 * F::T, SPT = N / NT;
    static constexpr int SUB = RegLds<N, 1, T>::SUB, PL = RegLds<N, 1, T>::ELEMS;
    static constexpr bool ok = sizeof(C) == sizeof(float2) || N == 4096;
    // the products' type: FP64 at N = 4096 in both forms, as in the separate passes; FP32 at 8192
    static constexpr bool FP64 = N == 4096;
    typedef typename std::conditional<FP64, m3, m3f>::type M;
    typedef typename std::conditional<FP64, double, float>::type S;
};
// v[k] -> LDS at to(k), v[k] <- LDS from from(k), the real parts and then the imaginary
// parts; WG: over the workgroup (otherwise inside each wave).  Ends with its reads.
template <int PT, bool WG, typename C, typename TO, typename FROM>
__device__ __forceinline__ void split_exchange(C* v, TO&& to, FROM&& from) {
    auto wait = [] {
        if constexpr (WG) __syncthreads();
        else wave_lds_fence();
    };
#pragma unroll
    for (int half = 0; half < 2; half++) {
        wait();
#pragma unroll
        for (int k = 0; k < PT; k++) *to(k) = half ? v[k].y : v[k].x;
        wait();
#pragma unroll
        for (int k = 0; k < PT; k++) (half ? v[k].y : v[k].x) = *from(k);
    }
}
// TILED: xi~ in tiles (Tile), the rows of a tile on one XCD.
template <int N, int TILED, typename C>
__global__ __launch_bounds__((Row1P<N, C>::NT), 1) void k_row_uxiu_1p(C* __restrict__ Vv, const C* __restrict__ U,
                                                                      const C* __restrict__ Xs, size_t V,
                                                                      const C* __restrict__ tw) {
    typedef typename scalar_of<C>::type T;
    typedef RegFft<N> F;
    typedef Row1P<N, C> R;
    constexpr int PT = F::PT, N3 = F::N3, SPT = R::SPT, SUB = R::SUB;
    static_assert(SPT * R::NT == N && 4 * SPT == PT, "row tiling");
    __shared__ T lds[4 * R::PL];
    const int x = TILED ? xcd_strip(blockIdx.x, N) : (int)blockIdx.x;
    const size_t row0 = (size_t)x * N;
    // the slots of the exchanges: a thread's points j + T r, its sub-sequence, the order inside it,
    // and a thread's sites (site y of plane p at (y / T) SUB + y mod T)
    auto pl = [&] { return lds + opaque_v((int)threadIdx.x) / F::T * R::PL; };
    auto idx = [] { return opaque_v((int)threadIdx.x) % F::T; };
#pragma unroll 1
    for (int half = 0; half < 2; half++) {
        C v[PT];
        {
            const int t = opaque_v((int)threadIdx.x), j = t % F::T;
            const int f = reg_freq<N>(j / N3, j % N3, 0);
            const C* src = Xs + (size_t)(4 * half + t / F::T) * V + (TILED ? Tile<N, C>::at(x, f) : row0 + f);
#pragma unroll
            for (int q = 0; q < PT; q++) v[q] = src[reg_freq_q<N>(q) * (TILED ? Tile<N, C>::TR : 1)];
        }
        {
            const int j = idx(), g = j / N3, m = j % N3;
            T* sub = pl() + g * SUB;
            T* own = pl() + j;
            if (half) __syncthreads();
#pragma unroll
            for (int u = 0; u < F::NU; u++) dft_reg<N3, +1>(v + u * N3);
            split_exchange<PT, false>(
                v, [&](int k) { return sub + (m + N3 * (k / N3)) * N3 + ((k % N3) ^ m); },
                [&](int b) { return sub + b * N3 + (m ^ (b % N3)); });
            twiddle<N, 3, +1>(v, tw_fft(tw), m);
            dft_reg<PT, +1>(v);
            split_exchange<PT, true>(
                v, [&](int a) { return sub + m + N3 * a; }, [&](int k) { return own + k * SUB; });
            twiddle<N, 1, +1>(v, tw_fft(tw), j);
            dft_reg<PT, +1>(v);
        }
        {
            T* own = pl() + idx();
            const int t = opaque_v((int)threadIdx.x);
            T* site = lds + t / F::T * SUB + t % F::T;
            split_exchange<PT, true>(
                v, [&](int r) { return own + r * SUB; },
                [&](int k) { return site + k % 4 * R::PL + k / 4 * 4 * SUB; });
        }
        // v[4 q + p]: plane p of site threadIdx + q NT
        const int tu = opaque_v((int)threadIdx.x);
#pragma unroll
        for (int q = 0; q < SPT; q++) {
            const size_t i = row0 + tu + q * R::NT;
            typename R::S hh[8], w[8];
#pragma unroll
            for (int p = 0; p < 4; p++) {
                hh[2 * p] = v[4 * q + p].x;
                hh[2 * p + 1] = v[4 * q + p].y;
            }
            typename R::M u;
            if constexpr (R::FP64) load_u_d<1>(u, U, V, i);
            else load_u(u, U, V, i);
            uxiu_gen(u, hh, w);
#pragma unroll
            for (int p = 0; p < 4; p++) v[4 * q + p] = mkc<C>(w[2 * p], w[2 * p + 1]);
        }
        {
            T* own = pl() + idx();
            const int t = opaque_v((int)threadIdx.x);
            T* site = lds + t / F::T * SUB + t % F::T;
            split_exchange<PT, true>(
                v, [&](int k) { return site + k % 4 * R::PL + k / 4 * 4 * SUB; },
                [&](int r) { return own + r * SUB; });
        }
        {
            const int j = idx(), g = j / N3, m = j % N3;
            T* sub = pl() + g * SUB;
            T* own = pl() + j;
            dft_reg<PT, -1>(v);
            twiddle<N, 1, -1>(v, tw_fft(tw), j);
            split_exchange<PT, true>(
                v, [&](int k) { return own + k * SUB; }, [&](int a) { return sub + m + N3 * a; });
            dft_reg<PT, -1>(v);
            twiddle<N, 3, -1>(v, tw_fft(tw), m);
            split_exchange<PT, false>(
                v, [&](int b) { return sub + b * N3 + (m ^ (b % N3)); },
                [&](int k) { return sub + (m + N3 * (k / N3)) * N3 + ((k % N3) ^ m); });
#pragma unroll
            for (int u = 0; u < F::NU; u++) dft_reg<N3, -1>(v + u * N3);
        }
        {
            const int t = opaque_v((int)threadIdx.x), j = t % F::T;
            C* dst = Vv + (size_t)(4 * half + t / F::T) * V + row0 + reg_freq<N>(j / N3, j % N3, 0);
#pragma unroll
            for (int q = 0; q < PT; q++) dst[reg_freq_q<N>(q)] = v[q];
        }
    }
}

template <int N, int BF, typename C>
static hipError_t step_large_n(jw_ctx* c, C* U, C* Xi, C* Vv, C* ZA, C* ZB, const StepArgs& a) {
    const size_t V = c->V;
    const C* tw = twiddles_of<C>(c);
    const unsigned g = grid_for(V, 256);
    const int wb = a.corr || a.kspace;      // xi~ written back by column A
    constexpr bool REG = BF == 3 || sizeof(C) == sizeof(double2);
    hipError_t e;
#define JW_TRY(x) if ((e = (x)) != hipSuccess) return e
    if (!a.kspace) {
        {
            KTimer t(c, K_GEN_NOISE);
            hipLaunchKernelGGL(k_gen_noise_packed<C>, dim3(g), dim3(256), 0, c->stream, Xi, V, a.ns, a.sa_pos);
            JW_TRY(hipGetLastError());
        }
        JW_TRY((launch_rows<N, REG, C>(c, Xi, 8, 1, 1.0, tw)));
    }
    {
        KTimer t(c, K_COL_KMULT);
        JW_TRY((col_pass<N, BF>(c, ZA, Xi, Xi + 4 * V, a.sa_k, a.sqrt_coupling, a.corr, 1, a.ns, a.kspace, a.corr)));
    }
    // BF = 3: column passes write tiles, which the row transforms take out of place, into
    // the planes of xi~ once U xi~ U^dagger has read them
    const C *HA = ZA, *HB = ZB;
    auto rows_inv = [&](C* Z, C* to, const C*& H) -> hipError_t {
        if constexpr (BF == 3) {
            KTimer t(c, K_FFT_ROWS);
            hipLaunchKernelGGL((k_rows_inv_tiled<N, C>), dim3(N / RowN<N>::RPW, 4), dim3(RowN<N>::NT), 0, c->stream, to, Z, V, tw);
            H = to;
            return hipGetLastError();
        } else {
            return launch_rows<N, REG, C>(c, Z, 4, 0, 1.0, tw);
        }
    };
    bool one_pass = false;
    if constexpr (Row1P<N, C>::ok) {
        if (wb) {
            KTimer t(c, K_UXIU);
            if (BF == 3 && a.kspace)
                hipLaunchKernelGGL((k_row_uxiu_1p<N, BF == 3, C>), dim3(N), dim3(Row1P<N, C>::NT), 0, c->stream, Vv, U, Xi, V, tw);
            else
                hipLaunchKernelGGL((k_row_uxiu_1p<N, 0, C>), dim3(N), dim3(Row1P<N, C>::NT), 0, c->stream, Vv, U, Xi, V, tw);
            JW_TRY(hipGetLastError());
            one_pass = true;
        }
    }
    if (!one_pass) {
        if (wb) JW_TRY((launch_rows<N, REG, C>(c, Xi, 8, 0, 1.0, tw)));
        {
            KTimer t(c, K_UXIU);
            hipLaunchKernelGGL((k_uxiu_packed<C, 1>), dim3(g), dim3(256), 0, c->stream, Vv, U, wb ? Xi : nullptr, V,
                               a.ns, a.sa_pos);
            JW_TRY(hipGetLastError());
        }
        JW_TRY((launch_rows<N, REG, C>(c, Vv, 8, 1, 1.0, tw)));
    }
    JW_TRY(rows_inv(ZA, Xi, HA));
    {
        KTimer t(c, K_COL_KMULT);
        JW_TRY((col_pass<N, BF>(c, ZB, Vv, Vv + 4 * V, a.sa_k, a.sqrt_coupling, 0, 1, a.ns, 0, 0)));
    }
    JW_TRY(rows_inv(ZB, Xi + 4 * V, HB));
    {
        KTimer t(c, K_UPDATE);
        hipLaunchKernelGGL((k_update_packed<C, 1>), dim3(g), dim3(256), 0, c->stream, U, HA, HB, V, a.sqrt_step,
                           a.reunit, a.whole);
        JW_TRY(hipGetLastError());
    }
#undef JW_TRY
    return hipSuccess;
}

// the column strips of a large lattice: the register-held strips of layout 0 (FP32
// at both sizes, FP64 at N = 4096), X and Y in LDS for the matrix-core stages on layout 0 (mixed,
// N = 4096), or one plane at a time over 16-byte segments (layout 32; FP64 at N = 8192 has
// no other)
template <typename C>
static hipError_t step_large_t(jw_ctx* c, C* U, C* Xi, C* Vv, C* ZA, C* ZB, const StepArgs& a) {
    if (a.nbatch != 1) return hipErrorInvalidValue;
    if (c->N == 8192) {
        if constexpr (sizeof(C) == sizeof(float2))
            if (c->layout == 0) return step_large_n<8192, 3>(c, U, Xi, Vv, ZA, ZB, a);
        return step_large_n<8192, 32>(c, U, Xi, Vv, ZA, ZB, a);
    }
    if (c->N == 4096) {
        if (c->layout == 32) return step_large_n<4096, 32>(c, U, Xi, Vv, ZA, ZB, a);
        if constexpr (sizeof(C) == sizeof(float2))
            if (c->fft_mfma) return step_large_n<4096, 5>(c, U, Xi, Vv, ZA, ZB, a);
        return step_large_n<4096, 3>(c, U, Xi, Vv, ZA, ZB, a);
    }
    return hipErrorInvalidValue;
}

}  // namespace jw
