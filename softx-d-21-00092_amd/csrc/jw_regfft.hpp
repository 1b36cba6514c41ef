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
#include "jw_internal.hpp"

namespace jw {

// In what follows no multiplication is fused with an addition except where it is
// written out (the same bits wherever a transform is inlined).

// s + h a (h real), a (1 + DIR i), a (-1 + DIR i)
template <typename T, typename C>
__device__ __forceinline__ C cmadr(C s, T h, C a) { return C{fma_t(h, a.x, s.x), fma_t(h, a.y, s.y)}; }
template <int DIR, typename C>
__device__ __forceinline__ C rot_p(C a) { return DIR < 0 ? C{a.x + a.y, a.y - a.x} : C{a.x - a.y, a.y + a.x}; }
template <int DIR, typename C>
__device__ __forceinline__ C rot_m(C a) { return DIR < 0 ? C{a.y - a.x, -a.y - a.x} : C{-a.x - a.y, a.x - a.y}; }

// The constant factors between two stages ride on the second one's additions as fused
// multiply-adds: as many instructions, one rounding less a point.

// 4 points, v[1], v[2], v[3] multiplied by w1, w2, w3 first
template <int DIR, typename C>
__device__ __forceinline__ void dft4_tw(C* v, C w1, C w2, C w3) {
#pragma clang fp contract(off)
    const C t0 = cmad(v[0], v[2], w2), t1 = cmad(v[0], v[2], C{-w2.x, -w2.y});
    const C b = cmul(v[1], w1);
    const C t2 = cmad(b, v[3], w3), t3 = rot_q<DIR>(cmad(b, v[3], C{-w3.x, -w3.y}));
    v[0] = cadd(t0, t2);
    v[2] = csub(t0, t2);
    v[1] = cadd(t1, t3);
    v[3] = csub(t1, t3);
}

// the same for w1 = e^{DIR 2 pi i / 8}, its square and its cube: h (1 + DIR i), DIR i, h (-1 + DIR i)
template <int DIR, typename C>
__device__ __forceinline__ void dft4_w8(C* v) {
#pragma clang fp contract(off)
    typedef decltype(v[0].x) T;
    const T h = (T)0.70710678118654752440084436210485;
    const C r = rot_q<DIR>(v[2]), p = cadd(v[0], r), m = csub(v[0], r);
    const C x = rot_p<DIR>(v[1]), y = rot_m<DIR>(v[3]);
    const C xs = cadd(x, y), xd = rot_q<DIR>(csub(x, y));
    v[0] = cmadr(p, h, xs);
    v[2] = cmadr(p, -h, xs);
    v[1] = cmadr(m, h, xd);
    v[3] = cmadr(m, -h, xd);
}

// in-register DFT of R points, natural order in and out
template <int R, int DIR, typename C>
__device__ __forceinline__ void dft_reg(C* v) {
#pragma clang fp contract(off)
    typedef decltype(v[0].x) T;
    const T h = (T)0.70710678118654752440084436210485;
    if constexpr (R < 8) {
        if constexpr (R > 1) dft_small<R, DIR>(v);
    } else if constexpr (R == 8) {
        C e[4] = {v[0], v[2], v[4], v[6]};
        C o[4] = {v[1], v[3], v[5], v[7]};
        dft_small<4, DIR>(e);
        dft_small<4, DIR>(o);
        // o1 (1 + DIR i), o3 (-1 + DIR i), each to be scaled by h; o2 DIR i
        const C o1 = rot_p<DIR>(o[1]), o2 = rot_q<DIR>(o[2]), o3 = rot_m<DIR>(o[3]);
        v[0] = cadd(e[0], o[0]);
        v[4] = csub(e[0], o[0]);
        v[1] = cmadr(e[1], h, o1);
        v[5] = cmadr(e[1], -h, o1);
        v[2] = cadd(e[2], o2);
        v[6] = csub(e[2], o2);
        v[3] = cmadr(e[3], h, o3);
        v[7] = cmadr(e[3], -h, o3);
    } else if constexpr (R == 16) {
        // n = 4 n1 + n2, k = k1 + 4 k2; the factors e^{DIR 2 pi i n2 k1 / 16}
        const T c1 = (T)0.92387953251128675612818318939679, s1 = (T)0.38268343236508977172845998403040, d = (T)DIR;
        C t[4][4];
#pragma unroll
        for (int n2 = 0; n2 < 4; n2++) {
#pragma unroll
            for (int n1 = 0; n1 < 4; n1++) t[n2][n1] = v[4 * n1 + n2];
            dft_small<4, DIR>(t[n2]);
        }
        C u[4][4];
#pragma unroll
        for (int k1 = 0; k1 < 4; k1++)
#pragma unroll
            for (int n2 = 0; n2 < 4; n2++) u[k1][n2] = t[n2][k1];
        dft_small<4, DIR>(u[0]);
        dft4_tw<DIR>(u[1], C{c1, d * s1}, C{h, d * h}, C{s1, d * c1});
        dft4_w8<DIR>(u[2]);
        dft4_tw<DIR>(u[3], C{s1, d * c1}, C{-h, d * h}, C{-c1, -d * s1});
#pragma unroll
        for (int k1 = 0; k1 < 4; k1++)
#pragma unroll
            for (int k2 = 0; k2 < 4; k2++) v[k1 + 4 * k2] = u[k1][k2];
    } else {
        static_assert(R == 32, "radix");
        // n = 4 n1 + n2, k = k1 + 8 k2; the factors e^{DIR 2 pi i n2 k1 / 32}
        const T c32[9] = {(T)1.0, (T)0.98078528040323044912618223613424, (T)0.92387953251128675612818318939679,
                          (T)0.83146961230254523707878837761791, (T)0.70710678118654752440084436210485,
                          (T)0.55557023301960222474283081394853, (T)0.38268343236508977172845998403040,
                          (T)0.19509032201612826784828486847702, (T)0.0};
        // quarter turns and the first quadrant's cosine and sine
        auto w32 = [&](int m) {
            C w = C{c32[m & 7], (T)DIR * c32[8 - (m & 7)]};
#pragma unroll
            for (int q = 0; q < 3; q++)
                if (q < (m >> 3)) w = rot_q<DIR>(w);
            return w;
        };
        C t[4][8];
#pragma unroll
        for (int n2 = 0; n2 < 4; n2++) {
#pragma unroll
            for (int n1 = 0; n1 < 8; n1++) t[n2][n1] = v[4 * n1 + n2];
            dft_reg<8, DIR>(t[n2]);
        }
#pragma unroll
        for (int k1 = 0; k1 < 8; k1++) {
            C u[4] = {t[0][k1], t[1][k1], t[2][k1], t[3][k1]};
            if (k1 == 0) dft_small<4, DIR>(u);
            else if (k1 == 4) dft4_w8<DIR>(u);
            else dft4_tw<DIR>(u, w32(k1), w32(2 * k1), w32(3 * k1));
#pragma unroll
            for (int k2 = 0; k2 < 4; k2++) v[k1 + 8 * k2] = u[k2];
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
    static constexpr int PT = reg_points(N);
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

// The factors of steps 1 and 3 in the order in which threads read them (reg_tables in
// jw_internal.hpp), behind the N entries w_N^i: w_N^(j k) at (k - 1) T + j, then w_N2^(m k) at
// (k - 1) N3 + m, k = 1 .. PT - 1.  A wave's entries are neighbours: read from the N entries
// instead, at stride k, they cost N = 2048 1542 us a step of fixed coupling in FP64 (1453 here).
template <int N, int STEP>
struct RegTw {
    typedef RegFft<N> F;
    static constexpr int BASE = STEP == 1 ? N : N + (F::PT - 1) * F::T, RUN = STEP == 1 ? F::T : F::N3;
};
// v[k] *= w^k of thread i of the step (DIR > 0: conjugate).  TABLE: every power is read,
// rounded once; otherwise w^(4 a + b) is the product of two entries, which the FP32 passes of
// N = 1024 and 2048 can afford (bound by requests to L1: table / products 183 / 176 and 779 /
// 754 us a step of fixed coupling).  rms error of forward, multiply, inverse against
// extended precision, radix-8 passes in LDS -> here: FP64 N = 64 3.21e-16 -> 3.00e-16, 128 3.53 ->
// 3.61, 256 3.73 -> 3.76, 512 4.21 -> 4.18, 1024 4.38 -> 4.11, 2048 4.57 -> 4.51, 4096 5.04 ->
// 4.69, 8192 5.15 -> 4.87 (products of two, no fused constants: 4.48 at 1024, 4.82 at 2048);
// FP32 (LDS: two-level table) with the table 1.72e-7 -> 1.69e-7 at 64, 1.94 -> 1.85 at 128, 2.82 ->
// 2.59 at 4096, 3.00 -> 2.72 at 8192, with products 2.82 -> 2.52 at 1024, 3.00 -> 2.63 at 2048.
template <int N, typename C>
struct TwRule {
    static constexpr bool TABLE = RegFft<N>::PT <= 8 || sizeof(C) == sizeof(double2) || N >= 4096;
};
template <int N, int STEP, int DIR, typename C>
__device__ __forceinline__ void twiddle(C* v, const C* __restrict__ tw, int i) {
    typedef RegTw<N, STEP> W;
    constexpr int PT = RegFft<N>::PT;
    auto at = [&](int k) {
        C w = (tw + (W::BASE + (k - 1) * W::RUN))[i];
        if (DIR > 0) w.y = -w.y;
        return w;
    };
    if constexpr (TwRule<N, C>::TABLE) {
#pragma unroll
        for (int k = 1; k < PT; k++) {
            v[k] = cmul(v[k], at(k));
            // FP32: 31 entries in flight at once take the registers of the data
            if (sizeof(C) == sizeof(float2) && k == 15 && PT > 16) __builtin_amdgcn_sched_barrier(0);
        }
        return;
    }
    C w[4];
#pragma unroll
    for (int b = 1; b < 4; b++) {
        w[b] = at(b);
        v[b] = cmul(v[b], w[b]);
    }
#pragma unroll
    for (int a = 4; a < PT; a += 4) {
        const C wa = at(a);
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
    twiddle<N, 1, -1>(v, tw, j);
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
        twiddle<N, 3, -1>(v, tw, m);
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
        twiddle<N, 3, +1>(v, tw, m);
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
    twiddle<N, 1, +1>(v, tw, j);
    dft_reg<PT, +1>(v);
}

}  // namespace jw
