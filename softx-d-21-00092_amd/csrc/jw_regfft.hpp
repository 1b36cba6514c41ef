// jw_regfft.hpp -- the FFT of the column passes with its data in registers.
//
// A length-N transform is split as N = PT * N2, N2 = PT * N3 and shared by
// T = N / PT threads of PT points each.  Forward (decimation in frequency):
//   1. thread j < T holds x[j + T r], r < PT, and takes the PT-point DFT over r;
//      result k1 is multiplied by w_N^(j k1);
//   2. exchange over the workgroup: thread (g, m) = (j / N3, j % N3) receives the
//      sub-sequence k1 = g at n2 = m + N3 a, a < PT;
//   3. PT-point DFT over a; result b1 is multiplied by w_N2^(m b1);
//   4. exchange among the N3 threads of a sub-sequence: thread (g, m) receives
//      b1 = m + N3 u, u < PT / N3, for all N3 values of the other digit;
//   5. PT / N3 DFTs of N3 points.
// The thread then holds the frequencies reg_freq(g, m, u, b2) =
// g + PT (m + N3 u) + PT^2 b2 in v[u N3 + b2].  The inverse runs the steps
// backwards and ends with the positions j + T r it started from, so that a
// pointwise factor between the two needs no reordering.
//
// W sequences (columns) side by side, column fastest over the lanes.  The
// N3 * W threads of a sub-sequence sit in one wave, so step 4 needs no workgroup
// barrier, and it stays inside the part of LDS that the same threads read
// in step 2.  One LDS element per point: step 4 swizzles the
// position inside a row of N3 by exclusive or with the row; step 2 pads short runs (RegLds).
#pragma once

#include "jw_device.hpp"

namespace jw {

// In what follows no multiplication is fused with an addition except where it is
// written out (the same bits wherever a transform is inlined).

// a * e^{DIR 2 pi i k / 16} for the constant twiddles of the 16-point DFT
template <int DIR, typename C>
__device__ __forceinline__ C rot16(C a, int k) {
#pragma clang fp contract(off)
    typedef decltype(a.x) T;
    const T c1 = (T)0.92387953251128675612818318939679, s1 = (T)0.38268343236508977172845998403040;
    const T h = (T)0.70710678118654752440084436210485;
    switch (k) {
        case 0: return a;
        case 4: return rot_q<DIR>(a);
        case 2: return DIR < 0 ? C{(a.x + a.y) * h, (a.y - a.x) * h} : C{(a.x - a.y) * h, (a.y + a.x) * h};
        case 6: return DIR < 0 ? C{(a.y - a.x) * h, -(a.x + a.y) * h} : C{-(a.x + a.y) * h, (a.x - a.y) * h};
        default: break;
    }
    const T c = (k == 1) ? c1 : (k == 3) ? s1 : -c1;                       // 1, 3, 9
    const T s = (T)(DIR < 0 ? -1 : 1) * ((k == 1) ? s1 : (k == 3) ? c1 : -s1);
    return cmul(a, C{c, s});
}

// 8 points: two 4-point halves; the odd outputs' 1 / sqrt 2 rides on the last additions
template <int DIR, typename C>
__device__ __forceinline__ void dft8_reg(C* v) {
#pragma clang fp contract(off)
    typedef decltype(v[0].x) T;
    C e[4] = {v[0], v[2], v[4], v[6]};
    C o[4] = {v[1], v[3], v[5], v[7]};
    dft_small<4, DIR>(e);
    dft_small<4, DIR>(o);
    const T h = (T)0.70710678118654752440084436210485;
    // o1 (1 + DIR i), o3 (-1 + DIR i), each to be scaled by h; o2 DIR i
    const C o1 = DIR < 0 ? C{o[1].x + o[1].y, o[1].y - o[1].x} : C{o[1].x - o[1].y, o[1].y + o[1].x};
    const C o3 = DIR < 0 ? C{o[3].y - o[3].x, -o[3].y - o[3].x} : C{-o[3].x - o[3].y, o[3].x - o[3].y};
    const C o2 = rot_q<DIR>(o[2]);
    v[0] = cadd(e[0], o[0]);
    v[4] = csub(e[0], o[0]);
    v[1] = C{fma_t(h, o1.x, e[1].x), fma_t(h, o1.y, e[1].y)};
    v[5] = C{fma_t(-h, o1.x, e[1].x), fma_t(-h, o1.y, e[1].y)};
    v[2] = cadd(e[2], o2);
    v[6] = csub(e[2], o2);
    v[3] = C{fma_t(h, o3.x, e[3].x), fma_t(h, o3.y, e[3].y)};
    v[7] = C{fma_t(-h, o3.x, e[3].x), fma_t(-h, o3.y, e[3].y)};
}

// in-register DFT of R points, natural order in and out
template <int R, int DIR, typename C>
__device__ __forceinline__ void dft_reg(C* v) {
#pragma clang fp contract(off)
    if constexpr (R == 8) {
        dft8_reg<DIR>(v);
    } else if constexpr (R < 8) {
        if constexpr (R > 1) dft_small<R, DIR>(v);
    } else if constexpr (R == 16) {
        // n = 4 n1 + n2, k = k1 + 4 k2
        C t[4][4];
#pragma unroll
        for (int n2 = 0; n2 < 4; n2++) {
#pragma unroll
            for (int n1 = 0; n1 < 4; n1++) t[n2][n1] = v[4 * n1 + n2];
            dft_small<4, DIR>(t[n2]);
#pragma unroll
            for (int k1 = 1; k1 < 4; k1++) t[n2][k1] = rot16<DIR>(t[n2][k1], n2 * k1);
        }
#pragma unroll
        for (int k1 = 0; k1 < 4; k1++) {
            C u[4] = {t[0][k1], t[1][k1], t[2][k1], t[3][k1]};
            dft_small<4, DIR>(u);
#pragma unroll
            for (int k2 = 0; k2 < 4; k2++) v[k1 + 4 * k2] = u[k2];
        }
    } else {
        static_assert(R == 32, "radix");
        // n = 2 n1 + n2, k = k1 + 16 k2
        typedef decltype(v[0].x) T;
        const T c32[8] = {(T)1.0, (T)0.98078528040323044912618223613424, (T)0.92387953251128675612818318939679,
                          (T)0.83146961230254523707878837761791, (T)0.70710678118654752440084436210485,
                          (T)0.55557023301960222474283081394853, (T)0.38268343236508977172845998403040,
                          (T)0.19509032201612826784828486847702};
        C e[16], o[16];
#pragma unroll
        for (int n = 0; n < 16; n++) { e[n] = v[2 * n]; o[n] = v[2 * n + 1]; }
        dft_reg<16, DIR>(e);
        dft_reg<16, DIR>(o);
#pragma unroll
        for (int k = 0; k < 16; k++) {
            C w = o[k];
            if (k & 7) {
                // e^{DIR 2 pi i k / 32}: cosine and sine of the first quadrant
                const int q = k & 7;
                const T c = c32[q], s = (T)(DIR < 0 ? -1 : 1) * c32[8 - q];
                w = cmul(w, C{c, s});
            }
            if (k >= 8) w = rot_q<DIR>(w);
            v[k] = cadd(e[k], w);
            v[k + 16] = csub(e[k], w);
        }
    }
}

// Points per thread.  Up to N = 512 one lattice has too few sequences to fill the chip,
// and 8 points with one more exchange beat 16 with half the waves (loaded column
// pass, one lattice, FP64 / FP32 us: N = 256 6.7 / 6.2 against 8.1 / 7.2; N = 512 16.0 / 9.4
// against 20.1 / 11.1; twelve lattices at once are within 8% either way).  From 1024
// on 16 points need one exchange less; 8192 = 32 * 32 * 8 keeps three factors; 64 = 4 * 4 * 4
// gives the row passes a whole wave per row.
template <int N>
struct RegFft {
    static constexpr int PT = N == 64 ? 4 : (N <= 512 ? 8 : (N <= 4096 ? 16 : 32));
    static constexpr int N2 = N / PT;
    static constexpr int N3 = N2 / PT;       // threads of a sub-sequence
    static constexpr int T = N / PT;         // threads of a sequence
    static constexpr int NU = PT / N3;
    static_assert(N3 >= 1 && N3 <= PT && PT * PT * N3 == N, "register FFT split");
};

// frequency of v[q] in thread (g, m): the thread's part and the point's
template <int N>
__device__ __forceinline__ constexpr int reg_freq_q(int q) {
    typedef RegFft<N> F;
    return F::PT * F::N3 * (q / F::N3) + F::PT * F::PT * (q % F::N3);
}
template <int N>
__device__ __forceinline__ constexpr int reg_freq(int g, int m, int q) {
    return g + RegFft<N>::PT * m + reg_freq_q<N>(q);
}

// v[k] *= w^k (DIR > 0: conjugate), k = 1 .. PT - 1, w = tw[idx].  Up to 8 points in FP64
// every power is read from the table; otherwise w^(4 a + b) is the product of two entries
// (15 loads of a stage instead of 6 cost the FP64 row passes at N = 2048 8% and the FP32
// ones 30%).  rms error of forward, multiply, inverse against extended precision, before
// (radix 8 through LDS) and now: N = 256 2.67e-16, 2.62e-16; 512 3.00e-16, 2.80e-16; 1024
// 3.01e-16, 3.22e-16; 2048 4.0e-16, 4.5e-16; in FP32 2.0e-7, 1.8e-7 at N = 2048.
template <int PT, int DIR, typename C>
__device__ __forceinline__ void twiddle_powers(C* v, const C* __restrict__ tw, int idx) {
    if constexpr (PT <= 8 && sizeof(C) == sizeof(double2)) {
#pragma unroll
        for (int k = 1; k < PT; k++) {
            C w = tw[k * idx];
            if (DIR > 0) w.y = -w.y;
            v[k] = cmul(v[k], w);
        }
        return;
    }
    C w[4];
#pragma unroll
    for (int b = 1; b < 4; b++) {
        w[b] = tw[b * idx];
        if (DIR > 0) w[b].y = -w[b].y;
        v[b] = cmul(v[b], w[b]);
    }
#pragma unroll
    for (int a = 4; a < PT; a += 4) {
        C wa = tw[a * idx];
        if (DIR > 0) wa.y = -wa.y;
        v[a] = cmul(v[a], wa);
#pragma unroll
        for (int b = 1; b < 4; b++) v[a + b] = cmul(v[a + b], cmul(wa, w[b]));
    }
}

// LDS order inside a wave: the compiler keeps the accesses in program order;
// a wave's own LDS operations complete in order
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// elements from one sub-sequence to the next in LDS: where the N3 * W elements that
// neighbouring lanes read together are less than 128 bytes, one such run of padding
// moves the next sub-sequence's run to other banks
template <int N, int W, typename C>
struct RegLds {
    static constexpr int RUN = RegFft<N>::N3 * W;
    static constexpr int SUB = RegFft<N>::N2 * W + (RUN * (int)sizeof(C) < 128 ? RUN : 0);
    static constexpr int ELEMS = RegFft<N>::PT * SUB;
};

// steps 1 to 5.  tid = j W + c: the thread's index in its sequence and its column.
// FIRST: no other wave's access of the buffer is pending (otherwise a barrier
// precedes the writes).
template <int N, int W, bool FIRST, typename C>
__device__ __forceinline__ void reg_fft_fwd(C* v, C* lds, const C* __restrict__ tw, int tid) {
    const int j = tid / W, c = tid % W;
    typedef RegFft<N> F;
    constexpr int PT = F::PT, N3 = F::N3, NU = F::NU, SUB = RegLds<N, W, C>::SUB;
    static_assert(N3 * W <= 64, "a sub-sequence sits in one wave");
    dft_reg<PT, -1>(v);
    __builtin_amdgcn_sched_barrier(0);
    twiddle_powers<PT, -1>(v, tw, j);
    if (!FIRST) __syncthreads();
    {
        C* p = lds + j * W + c;
#pragma unroll
        for (int k = 0; k < PT; k++) p[k * SUB] = v[k];
    }
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    const int g = j / N3, m = j % N3;
    C* sub = lds + g * SUB + c;
#pragma unroll
    for (int a = 0; a < PT; a++) v[a] = sub[(m + N3 * a) * W];
    dft_reg<PT, -1>(v);
    if constexpr (N3 > 1) {
        __builtin_amdgcn_sched_barrier(0);
        twiddle_powers<PT, -1>(v, tw, PT * m);
        wave_lds_fence();
#pragma unroll
        for (int b = 0; b < PT; b++) sub[(b * N3 + (m ^ (b % N3))) * W] = v[b];
        wave_lds_fence();
#pragma unroll
        for (int u = 0; u < NU; u++) {
#pragma unroll
            for (int q = 0; q < N3; q++) v[u * N3 + q] = sub[((m + N3 * u) * N3 + (q ^ m)) * W];
            dft_reg<N3, -1>(v + u * N3);
        }
    }
}

// the steps backwards; v from reg_freq order to positions j + T r, unscaled
template <int N, int W, bool FIRST, typename C>
__device__ __forceinline__ void reg_fft_inv(C* v, C* lds, const C* __restrict__ tw, int tid) {
    const int j = tid / W, c = tid % W;
    typedef RegFft<N> F;
    constexpr int PT = F::PT, N3 = F::N3, NU = F::NU, SUB = RegLds<N, W, C>::SUB;
    static_assert(N3 * W <= 64, "a sub-sequence sits in one wave");
    const int g = j / N3, m = j % N3;
    C* sub = lds + g * SUB + c;
    if (!FIRST) __syncthreads();
    if constexpr (N3 > 1) {
#pragma unroll
        for (int u = 0; u < NU; u++) {
            dft_reg<N3, +1>(v + u * N3);
#pragma unroll
            for (int q = 0; q < N3; q++) sub[((m + N3 * u) * N3 + (q ^ m)) * W] = v[u * N3 + q];
        }
        wave_lds_fence();
#pragma unroll
        for (int b = 0; b < PT; b++) v[b] = sub[(b * N3 + (m ^ (b % N3))) * W];
        twiddle_powers<PT, +1>(v, tw, PT * m);
        wave_lds_fence();
    }
    dft_reg<PT, +1>(v);
#pragma unroll
    for (int a = 0; a < PT; a++) sub[(m + N3 * a) * W] = v[a];
    __syncthreads();
    {
        const C* p = lds + j * W + c;
#pragma unroll
        for (int k = 0; k < PT; k++) v[k] = p[k * SUB];
    }
    twiddle_powers<PT, +1>(v, tw, j);
    dft_reg<PT, +1>(v);
}

}  // namespace jw
