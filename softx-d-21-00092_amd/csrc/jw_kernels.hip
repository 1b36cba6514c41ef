// jw_kernels.hip -- HIP kernels of the MI355X JIMWLK solver (gfx950) and their
// launchers.  Device storage: every field is a set of SoA planes of V complex
// doubles; plane k of a 9-component field holds matrix entry k = 3*row + col;
// site (x, y) sits at index x*N + y in every plane (field.h:199-209 order).
//
// Two families of kernels:
//  * the reference's per-function operations on 9-component fields
//    (generate_gaussian, prepare_A_local, uxiulocal, update_uf, ...).  Those
//    whose arithmetic can be reproduced operation for operation are compiled
//    without FMA contraction so that they agree with the reference to the bit;
//  * the generator-basis engine: every su(3) field (xi_x, xi_y, A, V_x, V_y, B)
//    is carried as 8 real generator planes packed two per complex plane, which
//    turns the reference's 72 complex plane FFTs per step into 24.
#include "jw_packed.hpp"

#include <math.h>

namespace jw {

// ===========================================================================
// FFT passes (jw_packed.hpp), FP64 instances
// ===========================================================================
hipError_t fft_rows(jw_ctx* c, cplx* planes, int nplanes, int dir, double scale) {
    return fft_rows_t(c, planes, nplanes, dir, scale);
}

hipError_t fft_cols(jw_ctx* c, cplx* planes, int nplanes, int dir, double scale) {
    return fft_cols_t(c, planes, nplanes, dir, scale);
}

hipError_t fft2d(jw_ctx* c, cplx* planes, int nplanes, int dir, double scale) {
    return fft2d_t(c, planes, nplanes, dir, scale);
}

// ===========================================================================
// host transfers: field planes <-> the reference's AoS order, on pinned host memory
// (consecutive lanes touch consecutive 16-byte words of it: whole bus transactions; bound
// by the bus)
// ===========================================================================
template <int T>
__global__ __launch_bounds__(256) void k_planes_to_aos(cplx* __restrict__ aos, const cplx* __restrict__ f, size_t V, size_t s0,
                                                       size_t n) {
    GRID_STRIDE(e, n * T) aos[e] = f[(e % T) * V + s0 + e / T];
}
template <int T>
__global__ __launch_bounds__(256) void k_aos_to_planes(cplx* __restrict__ f, const cplx* __restrict__ aos, size_t V, size_t s0,
                                                       size_t n) {
    GRID_STRIDE(e, n * T) f[(e % T) * V + s0 + e / T] = aos[e];
}

hipError_t planes_to_aos(jw_ctx* c, cplx* aos, const cplx* f, int t, size_t s0, size_t n) {
    const dim3 g(grid_for(n * t, 256)), b(256);
    if (t == 9) hipLaunchKernelGGL(k_planes_to_aos<9>, g, b, 0, c->stream, aos, f, c->V, s0, n);
    else if (t == 1) hipLaunchKernelGGL(k_planes_to_aos<1>, g, b, 0, c->stream, aos, f, c->V, s0, n);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t aos_to_planes(jw_ctx* c, cplx* f, const cplx* aos, int t, size_t s0, size_t n) {
    const dim3 g(grid_for(n * t, 256)), b(256);
    if (t == 9) hipLaunchKernelGGL(k_aos_to_planes<9>, g, b, 0, c->stream, f, aos, c->V, s0, n);
    else if (t == 1) hipLaunchKernelGGL(k_aos_to_planes<1>, g, b, 0, c->stream, f, aos, c->V, s0, n);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

// ===========================================================================
// tables
// ===========================================================================
// variant 0: sqrt(alpha) with prepare_A_local's operation order (field.h:2045-2046)
// variant 1: with generate_gaussian_with_noise_coupling_constant's (field.h:2257-2273)
__global__ __launch_bounds__(256) void k_sqrt_alpha(double* __restrict__ sa, const double* __restrict__ q4, int N, int variant, Alpha a) {
    const size_t V = (size_t)N * N;
    GRID_STRIDE(i, V) {
        const double ph = q4[i / N] + q4[i % N];
        const double inner = pow(pow(a.mu0_over_lambda * a.mu0_over_lambda, 1.0 / a.freeze_c) +
                                 pow((ph * N * N) / a.lambda_L / a.lambda_L, 1.0 / a.freeze_c), a.freeze_c);
        double v;
        if (variant == 0) v = sqrt(4.0 * M_PI / (a.beta0 * log(inner)));
        else v = sqrt((4.0 * M_PI / a.beta0) / log(inner));
        sa[i] = v;
    }
}

hipError_t build_sqrt_alpha(jw_ctx* c, double* sa, int variant, const Alpha& a) {
    hipLaunchKernelGGL(k_sqrt_alpha, dim3(grid_for(c->V, 256)), dim3(256), 0, c->stream, sa, c->q4, c->N,
                       variant, a);
    return hipGetLastError();
}

// ===========================================================================
// reference per-function kernels (9-component fields)
// ===========================================================================
__global__ __launch_bounds__(256) void k_set_unit(cplx* __restrict__ U, size_t V) {
    GRID_STRIDE(i, V) {
#pragma unroll
        for (int k = 0; k < 9; k++) U[k * V + i] = mk((k == 0 || k == 4 || k == 8) ? 1.0 : 0.0, 0.0);
    }
}

hipError_t set_unit(jw_ctx* c, cplx* U) {
    KTimer t(c, K_DROPIN);
    hipLaunchKernelGGL(k_set_unit, dim3(grid_for(c->V, 256)), dim3(256), 0, c->stream, U, c->V);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_generate_gaussian(cplx* __restrict__ xx, cplx* __restrict__ xy, size_t V, NoiseSrc ns,
                                    const double* __restrict__ sa_pos) {
#pragma clang fp contract(off)
    GRID_STRIDE(i, V) {
        double z[16];
        normals16(ns, i, z);
        double n[8], m[8];
        const double s = sa_pos ? sa_pos[i] : 1.0;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            n[k] = sa_pos ? z[2 * k] * s : z[2 * k];
            m[k] = sa_pos ? z[2 * k + 1] * s : z[2 * k + 1];
        }
        cplx a[9], b[9];
        lambda_entries(n, a);
        lambda_entries(m, b);
#pragma unroll
        for (int k = 0; k < 9; k++) { xx[k * V + i] = a[k]; xy[k * V + i] = b[k]; }
    }
}

hipError_t generate_gaussian(jw_ctx* c, cplx* xix, cplx* xiy, const NoiseSrc& ns, const double* sa_pos) {
    KTimer t(c, K_DROPIN);
    hipLaunchKernelGGL(k_generate_gaussian, dim3(grid_for(c->V, 256)), dim3(256), 0, c->stream, xix, xiy, c->V,
                       ns, sa_pos);
    return hipGetLastError();
}

// prepare_A_local (field.h:1998-2075), operation for operation
__global__ __launch_bounds__(256) void k_prepare_A_local(cplx* __restrict__ A, const cplx* __restrict__ xx, const cplx* __restrict__ xy,
                                  int N, int coupling, int kernel, const double* __restrict__ q4,
                                  const double* __restrict__ sb, const double* __restrict__ sa_k, Alpha al) {
#pragma clang fp contract(off)
    const size_t V = (size_t)N * N;
    GRID_STRIDE(i, V) {
        const int ix = (int)(i / N), iy = (int)(i % N);
        int xxm = ix, yym = iy;
        if (xxm >= N / 2) xxm -= N;
        if (yym >= N / 2) yym -= N;
        const double px = 2.0 * M_PI * xxm / (1.0 * N);
        const double py = 2.0 * M_PI * yym / (1.0 * N);
        cplx E[9];
#pragma unroll
        for (int k = 0; k < 9; k++) E[k] = mk(0.0, 0.0);
        if (fabs(px * px + py * py) > 10e-9) {
            double kxv, kyv;
            if (kernel == 0) {
                // LINEAR kernel: alpha at the continuum momentum (field.h:2032-2033)
                double sc = 1.0;
                if (coupling == 0)
                    sc = sqrt(4.0 * M_PI / (al.beta0 * log(pow(pow(al.mu0_over_lambda * al.mu0_over_lambda,
                                                                   1.0 / al.freeze_c) +
                                                               pow(((px * px + py * py) * N * N) / al.lambda_L /
                                                                   al.lambda_L, 1.0 / al.freeze_c),
                                                               al.freeze_c))));
                kxv = -2.0 * M_PI * sc * px / (px * px + py * py);
                kyv = -2.0 * M_PI * sc * py / (px * px + py * py);
            } else {
                const double ph = q4[ix] + q4[iy];
                const double sc = coupling == 0 ? sa_k[i] : 1.0;
                kxv = -2.0 * M_PI * sc * sb[ix] / ph;
                kyv = -2.0 * M_PI * sc * sb[iy] / ph;
            }
            const cplx KX = mk(0.0, kxv), KY = mk(0.0, kyv);
#pragma unroll
            for (int k = 0; k < 9; k++) E[k] = xadd(xmul(KX, xx[k * V + i]), xmul(KY, xy[k * V + i]));
        }
#pragma unroll
        for (int k = 0; k < 9; k++) A[k * V + i] = E[k];
    }
}

hipError_t prepare_A_local(jw_ctx* c, cplx* A, const cplx* xix, const cplx* xiy, int coupling, int kernel,
                           const double* sa_k, const Alpha& al) {
    KTimer t(c, K_DROPIN);
    hipLaunchKernelGGL(k_prepare_A_local, dim3(grid_for(c->V, 256)), dim3(256), 0, c->stream, A, xix, xiy, c->N,
                       coupling, kernel, c->q4, c->sb, sa_k, al);
    return hipGetLastError();
}

// uxiulocal (field.h:1892-1933): (U xi) U^dagger, operation for operation
__global__ __launch_bounds__(256) void k_uxiulocal(cplx* __restrict__ vx, cplx* __restrict__ vy, const cplx* __restrict__ U,
                            const cplx* __restrict__ xx, const cplx* __restrict__ xy, size_t V) {
    GRID_STRIDE(i, V) {
        const m3 u = load9(U, V, i);
        m3 d;
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
            for (int cc = 0; cc < 3; cc++) d.m[3 * r + cc] = conjg(u.m[3 * cc + r]);
        store9(vx, V, i, xmmul(xmmul(u, load9(xx, V, i)), d));
        store9(vy, V, i, xmmul(xmmul(u, load9(xy, V, i)), d));
    }
}

hipError_t uxiulocal(jw_ctx* c, cplx* Vx, cplx* Vy, const cplx* U, const cplx* xix, const cplx* xiy) {
    KTimer t(c, K_DROPIN);
    hipLaunchKernelGGL(k_uxiulocal, dim3(grid_for(c->V, 256)), dim3(256), 0, c->stream, Vx, Vy, U, xix, xiy, c->V);
    return hipGetLastError();
}

// update_uf (field.h:1966-1996): U <- exp(i sqrt(ds) B) U exp(-i sqrt(ds) A), both
// exponents read through their upper triangles
__global__ __launch_bounds__(256) void k_update_uf(cplx* __restrict__ U, const cplx* __restrict__ B, const cplx* __restrict__ A, size_t V,
                            double ss) {
    GRID_STRIDE(i, V) {
        double hb[8], ha[8];
        gen_from_upper(load9(B, V, i), hb);
        gen_from_upper(load9(A, V, i), ha);
        const m3 eb = exp_i_gen(hb, ss);
        const m3 ea = exp_i_gen(ha, -ss);
        store9(U, V, i, mmul(mmul(eb, load9(U, V, i)), ea));
    }
}

hipError_t update_uf(jw_ctx* c, cplx* U, const cplx* B, const cplx* A, double step) {
    KTimer t(c, K_DROPIN);
    hipLaunchKernelGGL(k_update_uf, dim3(grid_for(c->V, 256)), dim3(256), 0, c->stream, U, B, A, c->V, sqrt(step));
    return hipGetLastError();
}

// setMVModel (field.h:683-757): n = z*sigma + 0, lambda-basis map
__global__ __launch_bounds__(256) void k_set_mv_model(cplx* __restrict__ f, size_t V, NoiseSrc ns, double sigma) {
#pragma clang fp contract(off)
    GRID_STRIDE(i, V) {
        double z[8], n[8];
        normals8(ns, i, z);
#pragma unroll
        for (int k = 0; k < 8; k++) n[k] = z[k] * sigma + 0.0;
        cplx a[9];
        lambda_entries(n, a);
#pragma unroll
        for (int k = 0; k < 9; k++) f[k * V + i] = a[k];
    }
}

hipError_t set_mv_model(jw_ctx* c, cplx* f, const NoiseSrc& ns, double sigma) {
    KTimer t(c, K_DROPIN);
    hipLaunchKernelGGL(k_set_mv_model, dim3(grid_for(c->V, 256)), dim3(256), 0, c->stream, f, c->V, ns, sigma);
    return hipGetLastError();
}

// solvePoisson (field.h:867-877): f(k) *= -g/(-phat2(k) + mass^2).  The
// reference multiplies the k = 0 mode by -g/mass^2 (no guard); with zero_mode
// set it is set to zero instead (the option of projecting out the zero mode).
__global__ __launch_bounds__(256) void k_solve_poisson(cplx* __restrict__ f, int t, int N, const double* __restrict__ q4, double mass,
                                double g, int zero_mode) {
#pragma clang fp contract(off)
    const size_t V = (size_t)N * N;
    GRID_STRIDE(i, V) {
        const double ph = q4[i / N] + q4[i % N];
        const double fac = -1.0 * g / (-ph + mass * mass);
        for (int k = 0; k < t; k++) {
            const cplx v = f[k * V + i];
            f[k * V + i] = (zero_mode && i == 0) ? mk(0.0, 0.0) : xmul(v, mk(fac, 0.0));
        }
    }
}

hipError_t solve_poisson(jw_ctx* c, cplx* f, int t, double mass, double g) {
    KTimer t_(c, K_DROPIN);
    hipLaunchKernelGGL(k_solve_poisson, dim3(grid_for(c->V, 256)), dim3(256), 0, c->stream, f, t, c->N, c->q4,
                       mass, g, c->mv_zero_mode);
    return hipGetLastError();
}

// operator*= (field.h:337-365): U <- U exp(i f)
__global__ __launch_bounds__(256) void k_mul_exp(cplx* __restrict__ U, const cplx* __restrict__ f, size_t V) {
    GRID_STRIDE(i, V) {
        double h[8];
        gen_from_upper(load9(f, V, i), h);
        store9(U, V, i, mmul(load9(U, V, i), exp_i_gen(h, 1.0)));
    }
}

hipError_t mul_exp(jw_ctx* c, cplx* U, const cplx* f) {
    KTimer t(c, K_DROPIN);
    hipLaunchKernelGGL(k_mul_exp, dim3(grid_for(c->V, 256)), dim3(256), 0, c->stream, U, f, c->V);
    return hipGetLastError();
}

// lfield::trace (field.h:1375-1432): tr[(U/V)(U/V)^dagger], operation for operation
__device__ __forceinline__ double trace_site(const cplx* __restrict__ U, size_t V, size_t i, double vol) {
#pragma clang fp contract(off)
    double diag[3];
#pragma unroll
    for (int r = 0; r < 3; r++) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const cplx u = U[(3 * r + k) * V + i];
            const double ax = u.x / vol, ay = u.y / vol;
            s = s + (ax * ax - ay * (-ay));
        }
        diag[r] = s;
    }
    return (diag[0] + diag[1]) + diag[2];
}

__global__ __launch_bounds__(256) void k_trace(const cplx* __restrict__ U, cplx* __restrict__ corr, size_t V, double vol) {
    GRID_STRIDE(i, V) corr[i] = mk(trace_site(U, V, i, vol), 0.0);
}

hipError_t trace(jw_ctx* c, const cplx* U, cplx* corr) {
    KTimer t(c, K_OBS);
    hipLaunchKernelGGL(k_trace, dim3(grid_for(c->V, 256)), dim3(256), 0, c->stream, U, corr, c->V,
                       1.0 * c->N * c->N);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// tr[(F U / V)(F U / V)^dagger] over the lattice as reals: forward row transforms of
// the nine planes of U out of place (R 9 W 9), then the nine column transforms of a
// strip with the trace summed in registers (R 9 W 1/2), in trace_site's order of sums.
// Against the copy of U, two in-place transforms and the trace as passes of their own
// (R 36 W 28): N = 1024 60 + 65 us against 53 + 63 + 24 and the copy.  64 <= N <= 2048; others
// take those passes.
// ---------------------------------------------------------------------------
template <int N>
__global__ __launch_bounds__(RowN<N>::NT, 2) void k_corr_rows(cplx* __restrict__ out, const cplx* __restrict__ U, size_t V,
                                                             const cplx* __restrict__ tw) {
    constexpr int PT = RegFft<N>::PT, T = RegFft<N>::T;
    __shared__ cplx lds[RowN<N>::RPW * RowT<N, cplx>::PL];
    const int x = blockIdx.x * RowN<N>::RPW + threadIdx.x / T, j = threadIdx.x % T;
    const size_t row = (size_t)blockIdx.y * V + (size_t)x * N;
    cplx v[PT];
#pragma unroll
    for (int r = 0; r < PT; r++) v[r] = U[row + j + r * T];
    reg_fft_fwd<N, 1, true>(v, lds + (threadIdx.x / T) * RowT<N, cplx>::PL, tw_fft(tw), opaque_v(j));
    const int k0 = pos0<N, 0>(opaque_v(j));
#pragma unroll
    for (int q = 0; q < PT; q++) out[row + k0 + posq<N, 0>(q)] = v[q];
}

template <int N>
__global__ __launch_bounds__((ColR<N, cplx>::NT), (ColR<N, cplx>::WAVES)) void k_corr_cols(double* __restrict__ corr,
                                                                                          const cplx* __restrict__ R, size_t V,
                                                                                          const cplx* __restrict__ tw) {
#pragma clang fp contract(off)
    typedef RegFft<N> F;
    constexpr int PT = F::PT, W = ColR<N, cplx>::W;
    constexpr size_t RS = (size_t)F::T * N;
    __shared__ cplx lds[ColR<N, cplx>::ELEMS];
    const int col0 = xcd_strip(blockIdx.x, N / W) * W;
    const unsigned o = (unsigned)((int)(threadIdx.x / W) * N + col0 + (int)threadIdx.x % W);
    double sum[PT], diag[PT];
    // 1 / (N V): the unitary transform and the trace's division by V, a power of two
    const double s = 1.0 / ((double)N * (double)N * (double)N);
    // the next plane in flight under a transform where the registers allow it (small
    // lattices: few workgroups, latency)
    constexpr bool AHEAD = PT <= 8;
    cplx v[PT], w[AHEAD ? PT : 1];
    auto load = [&](cplx* d, int k) {
#pragma unroll
        for (int r = 0; r < PT; r++) d[r] = (R + k * V + r * RS)[o];
    };
    if constexpr (AHEAD) load(w, 0);
#pragma unroll 1
    for (int k = 0; k < 9; k++) {
        if constexpr (AHEAD) {
#pragma unroll
            for (int r = 0; r < PT; r++) v[r] = w[r];
            if (k < 8) load(w, k + 1);
        } else {
            load(v, k);
        }
        reg_fft_fwd<N, W, false>(v, lds, tw_fft(tw), opaque_v((int)threadIdx.x));
#pragma unroll
        for (int q = 0; q < PT; q++) {
            const double ax = v[q].x * s, ay = v[q].y * s, e = ax * ax + ay * ay;
            diag[q] = k % 3 == 0 ? e : diag[q] + e;
            if (k == 2) sum[q] = diag[q];
            if (k == 5 || k == 8) sum[q] = sum[q] + diag[q];
        }
    }
    const int j = threadIdx.x / W, ky = freq_of_pos<N, 0>(col0 + (int)threadIdx.x % W);
    const int kx0 = reg_freq<N>(j / F::N3, j % F::N3, 0);
#pragma unroll
    for (int q = 0; q < PT; q++) corr[(size_t)(kx0 + reg_freq_q<N>(q)) * N + ky] = sum[q];
}

template <int N>
static hipError_t corr_n(jw_ctx* c, const cplx* U, cplx* planes, double* corr) {
    KTimer t(c, K_OBS);
    hipLaunchKernelGGL(k_corr_rows<N>, dim3(N / RowN<N>::RPW, 9), dim3(RowN<N>::NT), 0, c->stream, planes, U, c->V, c->tw);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_corr_cols<N>, dim3(N / ColR<N, cplx>::W), dim3(ColR<N, cplx>::NT), 0, c->stream, corr, planes, c->V,
                       c->tw);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_corr_from_Uk(const cplx* __restrict__ U, double* __restrict__ corr, size_t V, double vol) {
    GRID_STRIDE(i, V) corr[i] = trace_site(U, V, i, vol);
}

hipError_t correlator(jw_ctx* c, const cplx* U, cplx* planes, double* corr) {
#define JW_CORR(n, C) case n: return corr_n<n>(c, U, planes, corr);
    switch (c->N) {
        JW_FUSED_SIZES(JW_CORR, cplx)
        default: break;
    }
#undef JW_CORR
    hipError_t e = hipMemcpyAsync(planes, U, 9 * c->V * sizeof(cplx), hipMemcpyDeviceToDevice, c->stream);
    if (e != hipSuccess) return e;
    if ((e = fft2d(c, planes, 9, 1, 1.0 / c->N)) != hipSuccess) return e;
    KTimer t(c, K_OBS);
    hipLaunchKernelGGL(k_corr_from_Uk, dim3(grid_for(c->V, 256)), dim3(256), 0, c->stream, planes, corr, c->V, 1.0 * c->N * c->N);
    return hipGetLastError();
}

// average_and_symmetrize on reals, sites s0 .. s0 + n - 1 into host memory (same operations).
// Launched from the lanes' host threads, so untimed: a KTimer writes the context's counters.
__global__ __launch_bounds__(256) void k_symmetrize_real(const double* __restrict__ in, double* __restrict__ out, int N, size_t s0,
                                                         size_t n) {
#pragma clang fp contract(off)
    GRID_STRIDE(e, n) {
        const size_t idx = s0 + e;
        const int i = (int)(idx / N), j = (int)(idx % N);
        const int a = (N - i) % N, b = (N - j) % N;
        auto tmp = [&](int x, int y) { return 0.5 * (in[(size_t)x * N + y] + in[(size_t)y * N + x]); };
        const double t1 = tmp(i, j), t2 = tmp(a, j), t3 = tmp(i, b), t4 = tmp(a, b);
        out[e] = 0.25 * (((t1 + t2) + t3) + t4);
    }
}

hipError_t symmetrize_real(jw_ctx* c, const double* in, double* out, size_t s0, size_t n) {
    hipLaunchKernelGGL(k_symmetrize_real, dim3(grid_for(n, 256)), dim3(256), 0, c->stream, in, out, c->N, s0, n);
    return hipGetLastError();
}

// reals to a complex plane, and the real part of one, scaled, back
__global__ __launch_bounds__(256) void k_plane_from_real(cplx* __restrict__ f, const double* __restrict__ in, size_t n) {
    GRID_STRIDE(i, n) f[i] = mk(in[i], 0.0);
}
__global__ __launch_bounds__(256) void k_real_from_plane(double* __restrict__ out, const cplx* __restrict__ f, size_t n, double s) {
    GRID_STRIDE(i, n) out[i] = s * f[i].x;
}
hipError_t plane_from_real(jw_ctx* c, cplx* f, const double* in, size_t n) {
    hipLaunchKernelGGL(k_plane_from_real, dim3(grid_for(n, 256)), dim3(256), 0, c->stream, f, in, n);
    return hipGetLastError();
}
hipError_t real_from_plane(jw_ctx* c, double* out, const cplx* f, size_t n, double s) {
    hipLaunchKernelGGL(k_real_from_plane, dim3(grid_for(n, 256)), dim3(256), 0, c->stream, out, f, n, s);
    return hipGetLastError();
}

// average_and_symmetrize (field.h:1460-1492): transpose average, then the
// (+-kx, +-ky) reflection average, operation for operation (out of place)
__global__ __launch_bounds__(256) void k_symmetrize(const cplx* __restrict__ in, cplx* __restrict__ out, int N) {
#pragma clang fp contract(off)
    const size_t V = (size_t)N * N;
    GRID_STRIDE(idx, V) {
        const int i = (int)(idx / N), j = (int)(idx % N);
        const int a = abs(i - N) % N, b = abs(j - N) % N;
        auto tmp = [&](int x, int y) {
            const cplx p = in[(size_t)x * N + y], q = in[(size_t)y * N + x];
            return mk(0.5 * (p.x + q.x), 0.5 * (p.y + q.y));
        };
        const cplx t1 = tmp(i, j), t2 = tmp(a, j), t3 = tmp(i, b), t4 = tmp(a, b);
        const cplx s = xadd(xadd(xadd(t1, t2), t3), t4);
        out[idx] = mk(0.25 * s.x, 0.25 * s.y);
    }
}

hipError_t average_and_symmetrize(jw_ctx* c, const cplx* in, cplx* out) {
    KTimer t(c, K_OBS);
    hipLaunchKernelGGL(k_symmetrize, dim3(grid_for(c->V, 256)), dim3(256), 0, c->stream, in, out, c->N);
    return hipGetLastError();
}

// reduce (field.h:1521-1536): sum += c, err += c^2
__global__ __launch_bounds__(256) void k_reduce(const cplx* __restrict__ corr, cplx* __restrict__ sum, cplx* __restrict__ err, size_t V) {
#pragma clang fp contract(off)
    GRID_STRIDE(i, V) {
        const cplx v = corr[i];
        sum[i] = mk(sum[i].x + v.x, sum[i].y + v.y);
        const cplx sq = (v.y == 0.0 && v.x > 0.0) ? mk(v.x * v.x, 0.0) : xmul(v, v);
        err[i] = mk(err[i].x + sq.x, err[i].y + sq.y);
    }
}

hipError_t reduce(jw_ctx* c, const cplx* corr, cplx* sum, cplx* err) {
    KTimer t(c, K_OBS);
    hipLaunchKernelGGL(k_reduce, dim3(grid_for(c->V, 256)), dim3(256), 0, c->stream, corr, sum, err, c->V);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_accumulate_real(const double* __restrict__ corr, double* __restrict__ sum, double* __restrict__ err,
                                  size_t V) {
#pragma clang fp contract(off)
    GRID_STRIDE(i, V) {
        const double v = corr[i];
        sum[i] += v;
        err[i] += v * v;
    }
}

hipError_t accumulate_real(jw_ctx* c, const double* corr, double* sum, double* err) {
    KTimer t(c, K_OBS);
    hipLaunchKernelGGL(k_accumulate_real, dim3(grid_for(c->V, 256)), dim3(256), 0, c->stream, corr, sum, err, c->V);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_scale(cplx* __restrict__ p, size_t n, double s) {
    GRID_STRIDE(i, n) p[i] = cscale(p[i], s);
}

hipError_t scale_planes(jw_ctx* c, cplx* p, size_t n, double s) {
    hipLaunchKernelGGL(k_scale, dim3(grid_for(n, 256)), dim3(256), 0, c->stream, p, n, s);
    return hipGetLastError();
}

// ===========================================================================
// POSITION_EVOLUTION (main_optimized.cpp:271-297, field.h:2368-2519): the
// position-space kernel sums at every site by brute force, O(V^2):
//   A(x) = sum_y wa(x - y) xi_x(y) + wb(x - y) xi_y(y)
//   B(x) = sum_y wa(x - y) V_x(y) + wb(x - y) V_y(y),   V_i = U xi_i U^dagger
// (the reference forms U E U^dagger per pair; with V_i precomputed the sum is
// the same to rounding).  One thread per target site; the sources pass through
// LDS in tiles of JW_POS_TILE (xi_x, xi_y, V_x, V_y: 36 complex values each).
// Each term is rounded as the reference rounds C = a xi_x, D = b xi_y, E = C + D.
// ===========================================================================
#define JW_POS_TILE 32

__global__ __launch_bounds__(256) void k_position_sums(cplx* __restrict__ A, cplx* __restrict__ B,
                                                       const cplx* __restrict__ X, const cplx* __restrict__ Y,
                                                       const cplx* __restrict__ VX, const cplx* __restrict__ VY,
                                                       const double* __restrict__ wa, const double* __restrict__ wb,
                                                       int N) {
#pragma clang fp contract(off)
    const size_t V = (size_t)N * N;
    __shared__ cplx tile[4][9][JW_POS_TILE];
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = t < V;
    const int tx = (int)(t / N), ty = (int)(t % N);
    cplx a[9], b[9];
#pragma unroll
    for (int k = 0; k < 9; k++) a[k] = b[k] = mk(0.0, 0.0);
    for (size_t y0 = 0; y0 < V; y0 += JW_POS_TILE) {
        for (int e = threadIdx.x; e < 4 * 9 * JW_POS_TILE; e += blockDim.x) {
            const int f = e / (9 * JW_POS_TILE), k = (e / JW_POS_TILE) % 9, j = e % JW_POS_TILE;
            const size_t src = y0 + j;
            const cplx* P = f == 0 ? X : f == 1 ? Y : f == 2 ? VX : VY;
            tile[f][k][j] = src < V ? P[k * V + src] : mk(0.0, 0.0);
        }
        __syncthreads();
        const int nj = (int)(V - y0 < JW_POS_TILE ? V - y0 : JW_POS_TILE);
        if (active)
            for (int j = 0; j < nj; j++) {
                const size_t src = y0 + j;
                const int sx = (int)(src / N), sy = (int)(src % N);
                const size_t r = (size_t)((tx - sx + N) % N) * N + (size_t)((ty - sy + N) % N);
                const double wx = wa[r], wy = wb[r];
#pragma unroll
                for (int k = 0; k < 9; k++) {
                    const cplx e1 = xadd(xmul(mk(wx, 0.0), tile[0][k][j]), xmul(mk(wy, 0.0), tile[1][k][j]));
                    const cplx e2 = xadd(xmul(mk(wx, 0.0), tile[2][k][j]), xmul(mk(wy, 0.0), tile[3][k][j]));
                    a[k] = xadd(a[k], e1);
                    b[k] = xadd(b[k], e2);
                }
            }
        __syncthreads();
    }
    if (active)
#pragma unroll
        for (int k = 0; k < 9; k++) {
            A[k * V + t] = a[k];
            B[k * V + t] = b[k];
        }
}

hipError_t position_sums(jw_ctx* c, cplx* A, cplx* B, const cplx* X, const cplx* Y, const cplx* VX, const cplx* VY,
                         const double* wa, const double* wb) {
    KTimer t(c, K_DROPIN);
    hipLaunchKernelGGL(k_position_sums, dim3((unsigned)((c->V + 255) / 256)), dim3(256), 0, c->stream, A, B, X, Y, VX,
                       VY, wa, wb, c->N);
    return hipGetLastError();
}

// f(k) *= s(k) on t planes (the per-mode noise correlation)
__global__ __launch_bounds__(256) void k_scale_by_table(cplx* __restrict__ f, int t, const double* __restrict__ s,
                                                        size_t V) {
    GRID_STRIDE(i, V) {
        const double v = s[i];
        for (int k = 0; k < t; k++) f[k * V + i] = cscale(f[k * V + i], v);
    }
}

hipError_t scale_by_table(jw_ctx* c, cplx* f, int t, const double* s) {
    KTimer t_(c, K_DROPIN);
    hipLaunchKernelGGL(k_scale_by_table, dim3(grid_for(c->V, 256)), dim3(256), 0, c->stream, f, t, s, c->V);
    return hipGetLastError();
}

// ===========================================================================
// generator-basis engine (jw_packed.hpp), the unfused FP64 step
// ===========================================================================
hipError_t step_unfused(jw_ctx* c, cplx* U, cplx* Xi, cplx* Vv, cplx* ZA, cplx* ZB, const NoiseSrc& ns,
                        const double* sa_pos, const double* sa_k, int kc, int corr, double ss) {
    return step_unfused_t(c, U, Xi, Vv, ZA, ZB, ns, sa_pos, sa_k, kc, corr, ss, 0);
}

// MV sheets in the generator basis
__global__ __launch_bounds__(256) void k_mv_noise_packed(cplx* __restrict__ R, size_t V, NoiseSrc ns, double sigma) {
    GRID_STRIDE(i, V) {
        double z[8];
        normals8(ns, i, z);
#pragma unroll
        for (int p = 0; p < 4; p++) R[p * V + i] = mk(z[2 * p] * sigma + 0.0, z[2 * p + 1] * sigma + 0.0);
    }
}

static hipError_t mv_noise_packed(jw_ctx* c, cplx* R, const NoiseSrc& ns, double sigma) {
    KTimer t(c, K_MV);
    hipLaunchKernelGGL(k_mv_noise_packed, dim3(grid_for(c->V, 256)), dim3(256), 0, c->stream, R, c->V, ns, sigma);
    return hipGetLastError();
}

static hipError_t poisson_packed(jw_ctx* c, cplx* R, double mass, double g) { return solve_poisson(c, R, 4, mass, g); }

__global__ __launch_bounds__(256) void k_mul_exp_packed(cplx* __restrict__ U, const cplx* __restrict__ R, size_t V) {
    GRID_STRIDE(i, V) {
        double h[8];
#pragma unroll
        for (int p = 0; p < 4; p++) { const cplx a = R[p * V + i]; h[2 * p] = a.x; h[2 * p + 1] = a.y; }
        store9(U, V, i, mmul(load9(U, V, i), exp_i_gen(h, 1.0)));
    }
}

static hipError_t mul_exp_packed(jw_ctx* c, cplx* U, const cplx* R) {
    KTimer t(c, K_MV);
    hipLaunchKernelGGL(k_mul_exp_packed, dim3(grid_for(c->V, 256)), dim3(256), 0, c->stream, U, R, c->V);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// MV sheets, 64 <= N <= 2048, in three passes of the fused step's make (jw_engine.hpp,
// jw_regfft.hpp) instead of noise, row and column transforms, Poisson, two transforms
// back and the exponential (28 complex planes moved a sheet instead of 70):
//   k_mv_noise_row : charges drawn in registers, forward row FFT              W 4
//   k_mv_col       : column FFT, -g / (-phat2 + m^2), inverse column FFT       R 4 W 4
//   k_mv_row_exp   : inverse row FFT, U <- U exp(i A)                           R 10 W 6
// (U as rows 0 and 1; the first sheet reads no U, the last writes all nine
// entries.)  Bound by memory but for the charges, whose logarithms and sines are.
// N = 1024: 222 -> 125 us a sheet.
// ---------------------------------------------------------------------------
template <int N>
__global__ __launch_bounds__(RowN<N>::NT, 2) void k_mv_noise_row(cplx* __restrict__ R, size_t V, NoiseSrc ns, double sigma,
                                                                const cplx* __restrict__ tw) {
    constexpr int PT = RegFft<N>::PT, T = RegFft<N>::T;
    __shared__ cplx lds[RowN<N>::RPW * RowT<N, cplx>::PL];
    const int x = blockIdx.x * RowN<N>::RPW + threadIdx.x / T, p = blockIdx.y;
    const int j = opaque_v((int)threadIdx.x % T);
    const unsigned row0 = (unsigned)x * N;
    cplx a[PT];
#pragma unroll
    for (int r = 0; r < PT; r++) {
        const unsigned i = row0 + j + r * T;
        if (ns.inj) {
            a[r] = reinterpret_cast<const double2*>(ns.inj + 8 * (size_t)i)[p];
        } else {
            box_muller_pair(i, ns.step, ns.tag, (uint32_t)p, ns.seed, ns.traj, a[r].x, a[r].y);
        }
        a[r] = cscale(a[r], sigma);
        fence(a[r]);
    }
    reg_fft_fwd<N, 1, true>(a, lds + (threadIdx.x / T) * RowT<N, cplx>::PL, tw_fft(tw), opaque_v((int)threadIdx.x % T));
    const int k0 = pos0<N, 0>(opaque_v((int)threadIdx.x % T));
#pragma unroll
    for (int q = 0; q < PT; q++) R[pat<N, 0>(p, x, k0 + posq<N, 0>(q), V)] = a[q];
}

template <int N>
__global__ __launch_bounds__((ColR<N, cplx>::NT), (ColR<N, cplx>::WAVES)) void k_mv_col(cplx* __restrict__ R, size_t V,
                                                                                       const double* __restrict__ q4,
                                                                                       double mass, double g, int zero_mode,
                                                                                       const cplx* __restrict__ tw) {
    typedef RegFft<N> F;
    constexpr int PT = F::PT, W = ColR<N, cplx>::W;
    constexpr size_t RS = (size_t)F::T * N;
    __shared__ cplx lds[ColR<N, cplx>::ELEMS];
    const int col0 = xcd_strip(blockIdx.x, N / W) * W;
    R += (size_t)blockIdx.y * V;
    const unsigned o = (unsigned)((int)(threadIdx.x / W) * N + col0 + (int)threadIdx.x % W);
    cplx v[PT];
#pragma unroll
    for (int r = 0; r < PT; r++) v[r] = (R + r * RS)[o];
    reg_fft_fwd<N, W, true>(v, lds, tw_fft(tw), opaque_v((int)threadIdx.x));
    const int t = after((int)threadIdx.x, v[PT - 1].x);
    const int j = t / W, ky = freq_of_pos<N, 0>(col0 + t % W);
    const int kx0 = reg_freq<N>(j / F::N3, j % F::N3, 0);
    const double q4y = q4[ky], num = -1.0 * g * (1.0 / ((double)N * (double)N));
#pragma unroll
    for (int q = 0; q < PT; q++) {
        const double f = num / (-((q4 + reg_freq_q<N>(q))[kx0] + q4y) + mass * mass);
        v[q] = zero_mode && q == 0 && kx0 == 0 && ky == 0 ? mk(0.0, 0.0) : cscale(v[q], f);
    }
    reg_fft_inv<N, W, true>(v, lds, tw_fft(tw), opaque_v((int)threadIdx.x));
#pragma unroll
    for (int r = 0; r < PT; r++) (R + r * RS)[o] = v[r];
}

template <int N>
__global__ __launch_bounds__(RowE<N>::NT, 2) void k_mv_row_exp(cplx* __restrict__ U, const cplx* __restrict__ R, size_t V,
                                                              int first, int last, const cplx* __restrict__ tw) {
    constexpr int NT = RowE<N>::NT, SPT = RowE<N>::SPT, PL = RowT<N, cplx>::PL;
    __shared__ cplx lds[4 * PL];
    const int tid = threadIdx.x, x = blockIdx.x;
    const size_t row0 = (size_t)x * N;
    cplx a[RowE<N>::PT];
    row_load<N, 0>(a, tid, [&](int p, int k) { return R[pat<N, 0>(p, x, k, V)]; });
    row_inv<N, true>(a, lds, tw, tid);
    __syncthreads();
#pragma unroll 1
    for (int q = 0; q < SPT; q++) {
        const int y = tid + q * NT;
        const size_t i = row0 + y;
        double h[8];
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const cplx b = lds[p * PL + row_slot_of<N, cplx>(y)];
            h[2 * p] = b.x;
            h[2 * p + 1] = b.y;
        }
        m3 e = exp_i_gen(h, 1.0);
        if (!first) {
            m3 u;
            load_u(u, U, V, i);
            e = mmul(u, e);
        }
        if (last) store9(U, V, i, e);
        else store_u(U, V, i, e);
    }
}

template <int N>
static hipError_t mv_sheet_n(jw_ctx* c, cplx* U, cplx* R, const NoiseSrc& ns, double sigma, double mass, double g, int first,
                             int last) {
    KTimer t(c, K_MV);
    const size_t V = c->V;
    hipError_t e;
    hipLaunchKernelGGL(k_mv_noise_row<N>, dim3(N / RowN<N>::RPW, 4), dim3(RowN<N>::NT), 0, c->stream, R, V, ns, sigma, c->tw);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_mv_col<N>, dim3(N / ColR<N, cplx>::W, 4), dim3(ColR<N, cplx>::NT), 0, c->stream, R, V, c->q4, mass, g,
                       c->mv_zero_mode, c->tw);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_mv_row_exp<N>, dim3(N), dim3(RowE<N>::NT), 0, c->stream, U, R, V, first, last, c->tw);
    return hipGetLastError();
}

// one sheet on the planes R (four): the fused passes for 64 <= N <= 2048, else the
// separate ones (the first sheet starts from U = 1)
hipError_t mv_sheet(jw_ctx* c, cplx* U, cplx* R, const NoiseSrc& ns, double sigma, double mass, double g, int first, int last) {
#define JW_MV(n, C) case n: return mv_sheet_n<n>(c, U, R, ns, sigma, mass, g, first, last);
    switch (c->N) {
        JW_FUSED_SIZES(JW_MV, cplx)
        default: break;
    }
#undef JW_MV
    hipError_t e;
#define JW_TRY(x) if ((e = (x)) != hipSuccess) return e
    if (first) JW_TRY(set_unit(c, U));
    JW_TRY(mv_noise_packed(c, R, ns, sigma));
    JW_TRY(fft2d(c, R, 4, 1, 1.0 / c->N));
    JW_TRY(poisson_packed(c, R, mass, g));
    JW_TRY(fft2d(c, R, 4, 0, 1.0 / c->N));
    JW_TRY(mul_exp_packed(c, U, R));
#undef JW_TRY
    return hipSuccess;
}

// ===========================================================================
// calibration: a plain copy of n double2 (16 n bytes read, 16 n written), used
// to scale the HBM traffic counters of the other kernels
// ===========================================================================
__global__ __launch_bounds__(256) void k_calibration_copy(const cplx* __restrict__ a, cplx* __restrict__ b, size_t n) {
    GRID_STRIDE(i, n) b[i] = a[i];
}

hipError_t calibration_copy(jw_ctx* c, const cplx* a, cplx* b, size_t n) {
    hipLaunchKernelGGL(k_calibration_copy, dim3(grid_for(n, 256)), dim3(256), 0, c->stream, a, b, n);
    return hipGetLastError();
}

// ===========================================================================
// unit-test hook: exp(i s H(h)) for a batch of generator vectors
// ===========================================================================
__global__ __launch_bounds__(256) void k_exp_batch(const double* __restrict__ h8, double s, double* __restrict__ out, int n) {
    GRID_STRIDE(i, (size_t)n) {
        double h[8];
#pragma unroll
        for (int a = 0; a < 8; a++) h[a] = h8[8 * i + a];
        const m3 e = exp_i_gen(h, s);
#pragma unroll
        for (int k = 0; k < 9; k++) { out[18 * i + 2 * k] = e.m[k].x; out[18 * i + 2 * k + 1] = e.m[k].y; }
    }
}

hipError_t exp_batch(jw_ctx* c, const double* h8, double s, double* out18, int n) {
    hipLaunchKernelGGL(k_exp_batch, dim3(grid_for((size_t)n, 256)), dim3(256), 0, c->stream, h8, s, out18, n);
    return hipGetLastError();
}

// the normals of given Philox words, four to a call: 53-bit pair in FP64 and FP32, the two
// 32-bit pairs in FP64 and FP32
__global__ __launch_bounds__(256) void k_box_muller_batch(const uint32_t* __restrict__ words, double* __restrict__ out, int n) {
    GRID_STRIDE(i, (size_t)n) {
        const uint32_t c[4] = {words[4 * i], words[4 * i + 1], words[4 * i + 2], words[4 * i + 3]};
        double* o = out + 12 * i;
        float f[2];
        box_muller53(c, o[0], o[1]);
        box_muller53(c, f[0], f[1]);
        o[2] = f[0];
        o[3] = f[1];
#pragma unroll
        for (int p = 0; p < 2; p++) {
            box_muller32(c[2 * p], c[2 * p + 1], o[4 + 2 * p], o[5 + 2 * p]);
            box_muller32(c[2 * p], c[2 * p + 1], f[0], f[1]);
            o[8 + 2 * p] = f[0];
            o[9 + 2 * p] = f[1];
        }
    }
}

hipError_t box_muller_batch(jw_ctx* c, const uint32_t* words, double* out12, int n) {
    hipLaunchKernelGGL(k_box_muller_batch, dim3(grid_for((size_t)n, 256)), dim3(256), 0, c->stream, words, out12, n);
    return hipGetLastError();
}

}  // namespace jw
