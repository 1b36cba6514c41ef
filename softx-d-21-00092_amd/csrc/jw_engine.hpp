// jw_engine.hpp -- fused generator-basis Langevin step for 64 <= N <= 2048,
// templated on the storage type C (double2: FP64 form, float2: mixed form);
// one object per size and type (jw_step_n.hip, jw_step_multi.hip).
//
// One step (main_optimized.cpp:243-304 in the generator basis) as five passes
// over HBM instead of the reference's 8 nine-component FFTs and 5 site loops:
//   row_noise_fwd  : Philox/injected noise -> xi planes, forward row FFT    W 8
//   col_kmult (A)  : forward column FFT, kernel multiply, inverse column FFT R 8 W 4
//                    (correlated noise: also writes F_col^-1[sqrt(alpha) F xi])
//   row_uxiu       : V = U xi U^dagger, forward row FFT                      R 6 W 8
//                    (correlated noise: inverse row FFT of xi~ first)     (R 14 W 8)
//   col_kmult (B)  : as for A                                                R 8 W 4
//   row_update     : inverse row FFTs of A, B; U <- exp(i s B) U exp(-i s A) R 14 W 6
// (units: complex planes of V elements, 16 B (FP64) or 8 B (FP32) per site each;
// U as its rows 0 and 1, UPlanes below).  With the spectra drawn per mode the
// noise pass goes and column A reads nothing and writes 12 planes.
//
// Transforms run with their data in registers (jw_regfft.hpp).  Row passes: one
// workgroup per lattice row and four planes, LDS holding the row between the transform
// and the site algebra.
//
// The intermediate planes (xi, V, A, B spectra) between a row pass and a
// column pass are stored in one of these layouts (template parameter BF):
//   BF = 0   row-major, row spectra in the order of freq_of_pos.  Column passes take
//            strips of W adjacent columns, X and Y in registers (k_col_reg), workgroups
//            mapped so that strips sharing cache lines run on the same XCD.
//   BF = 3   the same in frequency order: the large lattices.
//   BF = 5   row-major for the matrix-core stages (k_col_kmult).
//   BF = 2   the x and y directions interleaved site by site (k_col_kmult).
//   BF = 4, 8  blocks of BF rows: (x, y) at ((x / BF) N + y) BF + x mod BF, so
//            that one 128-byte segment holds 8 / BF adjacent columns of BF
//            consecutive rows.  A column pass then reads and writes whole
//            segments (8 / BF columns per workgroup, one plane at a time, all
//            four plane pairs in one workgroup); row passes touch BF-row
//            segments whose rows are processed on one XCD at neighbouring times.
//   BF = 1, 16, 32  row-major, one plane at a time over 64-, 32- or 16-byte strips.
// Row spectra on row-major planes up to N = 2048 are in the order of freq_of_pos.
// U always stays row-major.
#pragma once

#include "jw_common.hpp"
#include "jw_regfft.hpp"

namespace jw {

// Row passes: one lattice row and four planes a workgroup, T = N / PT threads a plane
// (jw_regfft.hpp).  A plane of the row sits in LDS in the order of the transform's
// own exchange, so that the thread that transforms reads and writes its own
// slots; site y is at slot (y / T) SUB + y mod T.
template <int N>
struct RowE {
    static constexpr int T = RegFft<N>::T, PT = RegFft<N>::PT;
    static constexpr int NT = 4 * T;
    static constexpr int SPT = N / NT;                  // sites per thread
    static_assert(SPT >= 1 && SPT * NT == N && NT >= 64, "row pass");
};
template <int N, typename C>
struct RowT {
    static constexpr int SUB = RegLds<N, 1, C>::SUB, PL = RegLds<N, 1, C>::ELEMS;      // PL: elements of a plane
};
template <int N, typename C>
__device__ __forceinline__ int row_slot_of(int y) {
    return (y / RowE<N>::T) * RowT<N, C>::SUB + y % RowE<N>::T;
}
// The column passes in LDS (k_col_kmult) hold the X and Y tiles of one W-column strip together
// in LDS (2 W N complex values plus one padding row in eight, 144 KB at most in
// FP64): W = min(16, 4096 / N) for both forms (wider FP32 strips measured
// slower: one workgroup per CU and spills in the correlated variant).
template <int N, typename C = double2, int CORR = 0>
struct ColE {
    static constexpr int NTMAX = 1024;
    static constexpr int W = (4096 / N > 16) ? 16 : 4096 / N;
    static constexpr int ELEMS = 2 * W * N;
    static constexpr int NT = (ELEMS / 8 < 64) ? 64 : ((ELEMS / 8 > NTMAX) ? NTMAX : ELEMS / 8);
    static constexpr int PER = ELEMS / NT;          // elements per thread
    static constexpr int PAIRS = (W * N) / NT;      // (X, Y) element pairs per thread
    static_assert(W >= 1 && W <= N && N % W == 0 && PER * NT == ELEMS && PAIRS * NT == W * N, "column tiling");
};

// minimum waves per SIMD requested of the row passes: two 512-thread workgroups per CU
// in FP32 (128 registers; 70 KB of LDS at N = 2048), one in FP64
template <typename C>
struct RowWaves { static constexpr int value = sizeof(C) == sizeof(double2) ? 2 : 4; };

// strip index for block b so that the strips on one XCD (blocks b, b+8, ...) are adjacent
__device__ __forceinline__ int xcd_strip(int b, int nstrips) {
    if (nstrips % 8) return b;
    return (b % 8) * (nstrips / 8) + b / 8;
}

// offset of site (x, y) in an intermediate plane of layout BF (4 and 8 row blocks, the
// others row-major)
constexpr bool row_blocks_of(int BF) { return BF == 4 || BF == 8; }
template <int N, int BF>
__device__ __forceinline__ size_t lay(int x, int y) {
    if constexpr (!row_blocks_of(BF)) return (size_t)x * N + y;
    else return ((size_t)(x / BF) * N + y) * BF + (x % BF);
}

// offset of site (x, y) of plane q (0..3: the x direction's plane pairs,
// 4..7: the y direction's) in an 8-plane spectral array.  Layout 2 interleaves
// the two directions of a plane pair site by site, (p, x, y, d) at
// 2 V p + 2 (x N + y) + d, so that a column strip of W columns of both
// directions is one 2W-element row segment.
template <int N, int BF>
__device__ __forceinline__ size_t pat(int q, int x, int y, size_t V) {
    if constexpr (BF == 2) return (size_t)(q & 3) * 2 * V + 2 * ((size_t)x * N + y) + (q >> 2);
    else return (size_t)q * V + lay<N, BF>(x, y);
}

// Row spectra on row-major planes are stored in the order in which the
// row transform ends: position s = q T + j holds the frequency of v[q] in thread j,
// so that a wave writes and reads whole contiguous runs (in frequency order its
// 64 elements are eight runs of 8; FP32 U xi~ U^dagger at N = 2048 242 against 195 us).  A column
// pass takes columns independently and needs only their frequency.  Interleaved and
// blocked planes keep frequency order, as do the large lattices.
template <int N, int BF>
struct RowOrder {
    static constexpr bool fft = N <= 2048 && (BF == 0 || BF == 1 || BF == 5 || BF == 16);
};
template <int N, int BF>
__device__ __forceinline__ int freq_of_pos(int s) {
    typedef RegFft<N> F;
    if constexpr (!RowOrder<N, BF>::fft) return s;
    else return reg_freq<N>(s % F::T / F::N3, s % F::N3, 0) + reg_freq_q<N>(s / F::T);
}
// position of v[q] in thread j: pos0(j) + posq(q)
template <int N, int BF>
__device__ __forceinline__ int pos0(int j) {
    return RowOrder<N, BF>::fft ? j : reg_freq<N>(j / RegFft<N>::N3, j % RegFft<N>::N3, 0);
}
template <int N, int BF>
__device__ __forceinline__ constexpr int posq(int q) {
    return RowOrder<N, BF>::fft ? q * RegFft<N>::T : reg_freq_q<N>(q);
}

// lattice row of row-pass block b.  Blocks are dealt round-robin to the 8 XCDs;
// with a blocked layout the BF rows sharing segments go to one XCD in
// consecutive turns (a bijection on [0, N) for N a multiple of 8 BF).
template <int N, int BF>
__device__ __forceinline__ int row_of_block(int b) {
    if constexpr (!row_blocks_of(BF)) return b;
    else {
        static_assert(N % (8 * BF) == 0, "blocked layout needs N a multiple of 8 BF");
        const int t = b >> 3, xcd = b & 7;
        return (t / BF) * (8 * BF) + xcd * BF + (t % BF);
    }
}

// Trajectory blockIdx.z of a batched launch: its planes sit at z times the
// per-trajectory size of each array, and its noise key is traj + z (the
// Philox step is read from the device counter when one is given).
__device__ __forceinline__ NoiseSrc batch_noise(NoiseSrc ns, size_t V) {
    ns.traj += blockIdx.z;
    if (ns.inj) ns.inj += (size_t)blockIdx.z * 16 * V;
    if (ns.stepp) ns.step = *ns.stepp;
    return ns;
}
__device__ __forceinline__ size_t zofs(int planes, size_t V) { return (size_t)blockIdx.z * planes * V; }
// the same for an explicit trajectory z (kernel bodies run by one workgroup or,
// in a launch over several size groups, by a part of one)
__device__ __forceinline__ NoiseSrc batch_noise_z(NoiseSrc ns, size_t V, int z) {
    ns.traj += z;
    if (ns.inj) ns.inj += (size_t)z * 16 * V;
    if (ns.stepp) ns.step = *ns.stepp;
    return ns;
}
__device__ __forceinline__ size_t zofs_z(int z, int planes, size_t V) { return (size_t)z * planes * V; }
// where a kernel body runs: its row, strip or segment (bx), plane pair (by),
// trajectory (bz) and thread index among the threads that run it (tid)
struct BlockIx {
    int bx, by, bz, tid;
};
__device__ __forceinline__ BlockIx own_block() {
    return BlockIx{(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z, (int)threadIdx.x};
}

// matrix type of the site algebra's products: FP64 in the FP64 form, FP32 in
// the mixed form (whose exponentials and projection stay FP64)
template <typename C>
struct site_mat { typedef m3 type; };
template <>
struct site_mat<float2> { typedef m3f type; };

// U planes read and written by the fused passes: rows 0 and 1 (six planes), row
// 2 rebuilt on load as conj(row 0 x row 1) -- U is in SU(3) to the rounding of
// its form (and the mixed form projects it every few steps, rebuilding row 2
// the same way) -- so that the row passes move a third less U.  The FP64 field
// keeps its nine planes; the last step of a call writes row 2 too (a pass of its own,
// R 6 W 3, took 118 us at N = 2048 and a tenth of a call of one step at N = 64).
template <typename C>
struct UPlanes { static constexpr int value = 6; };
template <typename C, typename M>
__device__ __forceinline__ void load_u(M& u, const C* __restrict__ U, size_t V, size_t i) {
#pragma unroll
    for (int k = 0; k < UPlanes<C>::value; k++) u.m[k] = U[k * V + i];
    if constexpr (UPlanes<C>::value == 6) {
        row2_of(u.m);
    }
}
template <typename C, typename M>
__device__ __forceinline__ void store_u(C* __restrict__ U, size_t V, size_t i, const M& r) {
#pragma unroll
    for (int k = 0; k < UPlanes<C>::value; k++) U[k * V + i] = r.m[k];
}

// ordering fences: values passed through them are final at the fence and
// values read after it are defined there (empty asm statements keep their order)
__device__ __forceinline__ void fence(double& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void fence(float& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void fence(float2& v) { asm volatile("" : "+v"(v.x), "+v"(v.y)); }
__device__ __forceinline__ void fence(double2& v) { asm volatile("" : "+v"(v.x), "+v"(v.y)); }

// the same pointer, opaque to the optimiser: loads through it are not merged
// with earlier loads of the same addresses (which would keep every twiddle of
// one FFT live in registers until the next)
template <typename T>
__device__ __forceinline__ const T* opaque(const T* p) {
    typedef const __attribute__((address_space(1))) T GT;     // a global-memory table
    GT* g = (GT*)p;
    asm volatile("" : "+s"(g));
    return (const T*)g;
}
// likewise for a per-thread index: values derived from it are recomputed
// rather than kept live from one phase of a kernel to the next
__device__ __forceinline__ int opaque_v(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// the points of a thread (plane tid / T) of a row spectrum: src(plane, position)
template <int N, int BF, typename C, typename F>
__device__ __forceinline__ void row_load(C* v, int tid, F&& src) {
    const int t = opaque_v(tid), p = t / RowE<N>::T, j = t % RowE<N>::T;
    const int k0 = pos0<N, BF>(j);
#pragma unroll
    for (int q = 0; q < RowE<N>::PT; q++) v[q] = src(p, k0 + posq<N, BF>(q));
}
// inverse transform of the loaded points into the plane's slots (site order).
// FIRST: no access of the slots by other threads is pending.
template <int N, bool FIRST, typename C>
__device__ __forceinline__ void row_inv(C* v, C* lds, const C* __restrict__ tw, int tid) {
    const int t = opaque_v(tid), p = t / RowE<N>::T, j = t % RowE<N>::T;
    C* pl = lds + p * RowT<N, C>::PL;
    reg_fft_inv<N, 1, FIRST>(v, pl, tw_fft(tw), j);
    const int j2 = opaque_v(tid) % RowE<N>::T;
#pragma unroll
    for (int r = 0; r < RowE<N>::PT; r++) pl[r * RowT<N, C>::SUB + j2] = v[r];
}
// forward transform of the plane's slots, stored by dst(plane, position, value)
template <int N, int BF, typename C, typename F>
__device__ __forceinline__ void row_fwd(C* lds, const C* __restrict__ tw, int tid, F&& dst) {
    C v[RowE<N>::PT];
    {
        const int t = opaque_v(tid), p = t / RowE<N>::T, j = t % RowE<N>::T;
        C* pl = lds + p * RowT<N, C>::PL;
#pragma unroll
        for (int r = 0; r < RowE<N>::PT; r++) v[r] = pl[r * RowT<N, C>::SUB + j];
        reg_fft_fwd<N, 1, true>(v, pl, tw_fft(tw), j);
    }
    const int t = opaque_v(tid), p = t / RowE<N>::T, j = t % RowE<N>::T;
    const int k0 = pos0<N, BF>(j);
#pragma unroll
    for (int q = 0; q < RowE<N>::PT; q++) dst(p, k0 + posq<N, BF>(q), v[q]);
}

// a thread's site index in a row pass's site loop, opaque, so that the compiler
// runs the sites one after another instead of interleaving their site algebra
// (FP32: registers for two workgroups per CU; FP64: fewer spills, the same
// arithmetic)
template <typename C>
__device__ __forceinline__ int site_of(int y) {
    return opaque_v(y);
}

// ---------------------------------------------------------------------------
// row pass 1: noise -> xi row spectra (planes 0..3 xi_x, 4..7 xi_y) of row x.
// The body is shared by the noise pass and by the update pass, which runs it
// for the next step after its own sites (the noise is compute-bound, the
// update memory-bound).  lds: 4 padded rows.
// ---------------------------------------------------------------------------
template <int N, int BF, typename C>
__device__ __forceinline__ void row_noise_body(C* lds, C* __restrict__ Xi, size_t V, const NoiseSrc& ns,
                                               const double* __restrict__ sa_pos, const C* __restrict__ tw, int x, int tid) {
    typedef typename scalar_of<C>::type T;
    constexpr int NT = RowE<N>::NT, SPT = RowE<N>::SPT, PL = RowT<N, C>::PL;
    const size_t row0 = (size_t)x * N;
    T m[SPT][8];
#pragma unroll
    for (int q = 0; q < SPT; q++) {
        const int y = tid + q * NT;
        T z[16];
        normals16_t(ns, row0 + y, z);
        const T s = sa_pos ? (T)sa_pos[row0 + y] : (T)1;      // in the element type: no FP64 in FP32
#pragma unroll
        for (int p = 0; p < 4; p++) lds[p * PL + row_slot_of<N, C>(y)] = C{z[4 * p] * s, z[4 * p + 2] * s};
#pragma unroll
        for (int k = 0; k < 8; k++) m[q][k] = z[2 * k + 1] * s;
    }
    __syncthreads();
    row_fwd<N, BF>(lds, tw, tid, [&](int p, int k, C v) { Xi[pat<N, BF>(p, x, k, V)] = v; });
    __syncthreads();
#pragma unroll
    for (int q = 0; q < SPT; q++)
#pragma unroll
        for (int p = 0; p < 4; p++)
            lds[p * PL + row_slot_of<N, C>(tid + q * NT)] = mkc<C>(m[q][2 * p], m[q][2 * p + 1]);
    __syncthreads();
    row_fwd<N, BF>(lds, tw, tid, [&](int p, int k, C v) { Xi[pat<N, BF>(4 + p, x, k, V)] = v; });
}

// The noise pass proper: one plane pair of a row by T threads.  Plane p of xi_x holds
// (n_2p, n_2p+1) and plane p of xi_y (m_2p, m_2p+1), the normals of Philox calls 2p
// and 2p+1 (draw order n0, m0, n1, m1, ...: call q gives n_q, m_q), so a thread draws
// the PT sites of both planes that it transforms, in registers.
template <int N>
struct RowN {
    static constexpr int T = RegFft<N>::T;
    static constexpr int NT = T < 128 ? 128 : T;        // threads: NT / T rows side by side
    static constexpr int RPW = NT / T;
};

// row x, plane pair bi.by, thread j of the row's T; lds: one plane of the row
template <int N, int BF, typename C>
__device__ __forceinline__ void row_noise_fwd_body(C* lds, BlockIx bi, C* __restrict__ Xi, size_t V, NoiseSrc ns,
                                                   const double* __restrict__ sa_pos, const C* __restrict__ tw) {
    typedef typename scalar_of<C>::type T;
    constexpr int PT = RegFft<N>::PT, TR = RegFft<N>::T;
    Xi += zofs_z(bi.bz, 8, V);
    ns = batch_noise_z(ns, V, bi.bz);
    const int x = row_of_block<N, BF>(bi.bx), p = bi.by;
    const unsigned row0 = (unsigned)x * N;
    C a[PT], b[PT];
    const int j = opaque_v(bi.tid);
#pragma unroll
    for (int r = 0; r < PT; r++) {
        const unsigned i = row0 + j + r * TR;
        T z[4];
        if (ns.inj) {
            const double* zi = ns.inj + 16 * (size_t)i + 4 * p;
#pragma unroll
            for (int k = 0; k < 4; k++) z[k] = (T)zi[k];
        } else if constexpr (sizeof(T) == sizeof(double)) {
            box_muller_pair(i, ns.step, ns.tag, (uint32_t)(2 * p), ns.seed, ns.traj, z[0], z[1]);
            box_muller_pair(i, ns.step, ns.tag, (uint32_t)(2 * p + 1), ns.seed, ns.traj, z[2], z[3]);
        } else {
            box_muller_pair_f(i, ns.step, ns.tag, (uint32_t)(2 * p), ns.seed, ns.traj, z[0], z[1]);
            box_muller_pair_f(i, ns.step, ns.tag, (uint32_t)(2 * p + 1), ns.seed, ns.traj, z[2], z[3]);
        }
        const T s = sa_pos ? (T)sa_pos[i] : (T)1;
        a[r] = C{z[0] * s, z[2] * s};
        b[r] = C{z[1] * s, z[3] * s};
        fence(a[r]);
        fence(b[r]);
    }
    auto store = [&](const C* v, int pl) {
        const int t = opaque_v(bi.tid);
        const int k0 = pos0<N, BF>(t);
#pragma unroll
        for (int q = 0; q < PT; q++) Xi[pat<N, BF>(pl, x, k0 + posq<N, BF>(q), V)] = v[q];
    };
    reg_fft_fwd<N, 1, true>(a, lds, tw_fft(tw), opaque_v(bi.tid));
    store(a, p);
    reg_fft_fwd<N, 1, false>(b, lds, tw_fft(tw), opaque_v(bi.tid));
    store(b, 4 + p);
}

template <int N, int BF, typename C>
__global__ __launch_bounds__(RowN<N>::NT, RowWaves<C>::value) void k_row_noise_fwd(C* __restrict__ Xi, size_t V, NoiseSrc ns,
                                                              const double* __restrict__ sa_pos,
                                                              const C* __restrict__ tw) {
    __shared__ C lds[RowN<N>::RPW * RowT<N, C>::PL];
    const int s = threadIdx.x / RowN<N>::T;
    const BlockIx bi{(int)blockIdx.x * RowN<N>::RPW + s, (int)blockIdx.y, (int)blockIdx.z, (int)threadIdx.x % RowN<N>::T};
    row_noise_fwd_body<N, BF, C>(lds + s * RowT<N, C>::PL, bi, Xi, V, ns, sa_pos, tw);
}

// ---------------------------------------------------------------------------
// row pass 2: V_i = U xi_i U^dagger -> V row spectra (planes 0..3 V_x, 4..7 V_y),
// xi regenerated from the noise source (white noise)
// ---------------------------------------------------------------------------
template <int N, int BF, typename C>
__device__ __forceinline__ void row_uxiu_fwd_body(C* lds, BlockIx bi, C* __restrict__ Vv, const C* __restrict__ U,
                                                             size_t V, NoiseSrc ns, const double* __restrict__ sa_pos,
                                                             const C* __restrict__ tw) {
    typedef typename scalar_of<C>::type T;
    constexpr int NT = RowE<N>::NT, SPT = RowE<N>::SPT;
    constexpr int PL = RowT<N, C>::PL;
    const int tid = bi.tid;
    Vv += zofs_z(bi.bz, 8, V);
    U += zofs_z(bi.bz, UPlanes<C>::value, V);
    ns = batch_noise_z(ns, V, bi.bz);
    const int x = row_of_block<N, BF>(bi.bx);
    const size_t row0 = (size_t)x * N;
    T vy[SPT][8];      // in the element type: they go to LDS in it
#pragma unroll
    for (int q = 0; q < SPT; q++) {
        const int y = site_of<C>(tid + q * NT);
        const size_t i = row0 + y;
        T hx[8], hy[8];
        T z[16];
        normals16_t(ns, i, z);
        const T s = sa_pos ? (T)sa_pos[i] : (T)1;
#pragma unroll
        for (int k = 0; k < 8; k++) { hx[k] = z[2 * k] * s; hy[k] = z[2 * k + 1] * s; }
        // FP64 form: FP64 products; mixed form: FP32 products
        typename site_mat<C>::type u;
        load_u(u, U, V, i);
        T vx[8], v2[8];
        uxiu_gen(u, hx, vx);
        uxiu_gen(u, hy, v2);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            vy[q][k] = (T)v2[k];
            fence(vy[q][k]);
        }
#pragma unroll
        for (int p = 0; p < 4; p++) lds[p * PL + row_slot_of<N, C>(y)] = mkc<C>(vx[2 * p], vx[2 * p + 1]);
    }
    __syncthreads();
    row_fwd<N, BF>(lds, tw, tid, [&](int p, int k, C v) { Vv[pat<N, BF>(p, x, k, V)] = v; });
    __syncthreads();
#pragma unroll
    for (int q = 0; q < SPT; q++)
#pragma unroll
        for (int p = 0; p < 4; p++)
            lds[p * PL + row_slot_of<N, C>(tid + q * NT)] = mkc<C>(vy[q][2 * p], vy[q][2 * p + 1]);
    __syncthreads();
    row_fwd<N, BF>(lds, tw, tid, [&](int p, int k, C v) { Vv[pat<N, BF>(4 + p, x, k, V)] = v; });
}

template <int N, int BF, typename C>
__global__ __launch_bounds__(RowE<N>::NT, RowWaves<C>::value) void k_row_uxiu_fwd(C* __restrict__ Vv, const C* __restrict__ U,
                                                             size_t V, NoiseSrc ns, const double* __restrict__ sa_pos,
                                                             const C* __restrict__ tw) {
    __shared__ C lds[4 * RowT<N, C>::PL];
    row_uxiu_fwd_body<N, BF, C>(lds, own_block(), Vv, U, V, ns, sa_pos, tw);
}

// ---------------------------------------------------------------------------
// row pass 2, correlated noise: reads the column-inverse spectra of xi~,
// finishes their inverse transform along the row, and forms V_i = U xi~_i U^dagger
// in two batches (i = x, then y).  In each batch a site's V coefficients
// overwrite its own xi~ slots in LDS before the forward row FFT.  U is read in
// both batches: holding xi~_x in registers to read U once needs more registers
// and measured slower (one workgroup per CU instead of two in FP32).
// ---------------------------------------------------------------------------
template <int N, int BF, typename C>
__device__ __forceinline__ void row_uxiu_corr_body(C* lds, BlockIx bi, C* __restrict__ Vv, const C* __restrict__ U,
                                                              const C* __restrict__ Xs, size_t V,
                                                              const C* __restrict__ tw) {
    typedef typename scalar_of<C>::type T;
    constexpr int NT = RowE<N>::NT, SPT = RowE<N>::SPT, PL = RowT<N, C>::PL;
    const int tid = bi.tid;
    Vv += zofs_z(bi.bz, 8, V);
    U += zofs_z(bi.bz, UPlanes<C>::value, V);
    Xs += zofs_z(bi.bz, 8, V);
    const int x = row_of_block<N, BF>(bi.bx);
    const size_t row0 = (size_t)x * N;
    C h[RowE<N>::PT];
    row_load<N, BF>(h, tid, [&](int p, int k) { return Xs[pat<N, BF>(p, x, k, V)]; });
#pragma unroll
    for (int half = 0; half < 2; half++) {
        row_inv<N, true>(h, lds, tw, tid);
        // the y direction's spectra are in flight during the x direction's site algebra
        if (half == 0) row_load<N, BF>(h, tid, [&](int p, int k) { return Xs[pat<N, BF>(4 + p, x, k, V)]; });
        __syncthreads();
        // one site at a time: keeps a single U (9 complex, row 2 rebuilt) live
#pragma unroll 1
        for (int q = 0; q < SPT; q++) {
            const int y = tid + q * NT;
            const size_t i = row0 + y;
            C* const slot = lds + row_slot_of<N, C>(y);
            T g[8];
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const C a = slot[p * PL];
                g[2 * p] = a.x;
                g[2 * p + 1] = a.y;
            }
            typename site_mat<C>::type u;
            load_u(u, U, V, i);
            T v[8];
            uxiu_gen(u, g, v);
#pragma unroll
            for (int p = 0; p < 4; p++) slot[p * PL] = mkc<C>(v[2 * p], v[2 * p + 1]);
        }
        __syncthreads();
        row_fwd<N, BF>(lds, tw, tid, [&](int p, int k, C v) { Vv[pat<N, BF>(4 * half + p, x, k, V)] = v; });
    }
}

template <int N, int BF, typename C>
__global__ __launch_bounds__(RowE<N>::NT, RowWaves<C>::value) void k_row_uxiu_corr(C* __restrict__ Vv, const C* __restrict__ U,
                                                              const C* __restrict__ Xs, size_t V,
                                                              const C* __restrict__ tw) {
    __shared__ C lds[4 * RowT<N, C>::PL];
    row_uxiu_corr_body<N, BF, C>(lds, own_block(), Vv, U, Xs, V, tw);
}

// ---------------------------------------------------------------------------
// column pass on row-major planes, transforms in registers (jw_regfft.hpp):
//   Z[p] = F_col^-1[ i (kx X^[p] + ky Y^[p]) / V ], X^ = F_col X
//   kx = -2 pi c pbarX / phat2 (c = sa(k) for MODE 1, else 1), zero at k = 0.
//   CORR: X^, Y^ are first multiplied by sa(k) (MODE 2) and F_col^-1[X^ / V] is
//   written back over X (likewise Y).
//   GEN (with CORR): X^, Y^ are not transformed from X, Y but drawn per mode
//   (kspace_normals4, plane pair p = bi.by, noise key from ns); X and Y then
//   receive the row spectra of the position-space noise.
// X, Y: row spectra of plane p; one workgroup per strip of W columns and plane
// pair.  BF = 0: columns in the order of freq_of_pos, and sa's likewise; otherwise
// (the large lattices) column c is frequency c.  A thread holds PT points of one column
// of X and of Y; LDS holds one plane of the strip for the exchanges, and the
// (4 sin^2, sin) table of kx.
//
// What bounds it: the loaded pass moves 12 planes at 2.7-2.8 TB/s (FP64 and FP32
// at N = 2048; the bare access pattern reaches 4.6 TB/s), the drawing pass is
// bound by the noise's instructions.  64-byte row segments (W = 4 FP64, 8 FP32)
// take the bare pattern from 2.7 TB/s (16 bytes) and 3.7 (32 bytes) to 4.6, and
// the registers of a CU hold four times the strip that the LDS-resident form
// (k_col_kmult) could, with 4 workgroup barriers instead of about 20.
// N = 2048, us per launch (kernel trace, averages), k_col_kmult -> this: loaded FP64 420 ->
// 298, FP32 241 -> 146; correlated FP64 660 -> 546, FP32 445 -> 234; drawing FP64 490 -> 403,
// FP32 295 -> 183.
// ---------------------------------------------------------------------------
template <int N, typename C>
struct ColR {
    static constexpr bool F64 = sizeof(C) == sizeof(double2);
    static constexpr int WSEG = 64 / (int)sizeof(C);                     // columns of a 64-byte segment
    // the widest strip whose X and Y fit the registers of one CU (FP64 8192, FP32
    // 16384 points), 64-byte segments at most
    static constexpr int WMAX = (F64 ? 8192 : 16384) / N;
    static constexpr int W = WMAX < WSEG ? WMAX : (N / RegFft<N>::PT * WSEG < 64 ? 64 / (N / RegFft<N>::PT) : WSEG);
    static constexpr int NT = N / RegFft<N>::PT * W;
    static constexpr int ELEMS = RegLds<N, W, C>::ELEMS;                 // of C in LDS
    static constexpr bool TAB = ELEMS * (int)sizeof(C) + N * 16 <= 160 * 1024;
    static constexpr int LDS = ELEMS + (TAB ? N * 16 / (int)sizeof(C) : 0);
    // registers: 256 (FP64; 32 points a thread) or 128 a thread
    static constexpr int REGS = F64 || RegFft<N>::PT > 16 ? 256 : 128;
    static constexpr int WAVES = 512 / REGS;
    static_assert(W >= 1 && NT >= 64 && NT * REGS <= 512 * 256, "column strip");
};

// Planes that a column pass of a large lattice writes for row passes (BF = 3; Z, and X, Y
// where they are drawn): tiles of TR rows by the strip's W columns, 64 bytes each, so that a
// workgroup writes whole 64-byte pieces.  In row-major planes a strip's row segments are 16
// bytes (N = 8192 in FP32; 32 at 4096), the other strips' parts of a line come after
// the line has left L2, and 2.4 times the bytes went to memory.  us per launch, row-major
// -> tiles: N = 8192 FP32 drawing 9500 -> 5010, loaded (which reads row-major planes)
// 6180 -> 4490, against U xi~ U^dagger 4600 -> 5000 on tiles.  Two drawn fixed-coupling steps
// at N = 4096, FP64 14.8 -> 13.5 ms, FP32 10.0 -> 9.1.  at(x, c) is the offset of row x's
// column c; columns W apart are TR W elements apart.
template <int N, typename C>
struct Tile {
    static constexpr int W = ColR<N, C>::W, TR = 64 / (int)sizeof(C) / W;
    static_assert(TR >= 1 && RegFft<N>::T % TR == 0, "tile");
    static __device__ __forceinline__ size_t at(int x, int c) {
        return ((size_t)(x / TR) * (N / W) + c / W) * (TR * W) + (x % TR) * W + c % W;
    }
};

// v, defined only once d is: what is computed from it is not started before
template <typename T>
__device__ __forceinline__ int after(int v, T d) {
    asm volatile("" : "+v"(v) : "v"(d));
    return v;
}

// lds: ColR::ELEMS elements; kt: N (q4, sb) pairs (TAB), filled here by the whole workgroup
template <int N, int CORR, int GEN, int MODE, int BF, typename C>
__device__ __forceinline__ void col_reg_body(C* lds, double2* kt, BlockIx bi, C* __restrict__ Z, C* __restrict__ X,
                                             C* __restrict__ Y, size_t V, const double* __restrict__ q4,
                                             const double* __restrict__ sb, const double* __restrict__ sa,
                                             const C* __restrict__ tw, NoiseSrc ns) {
    static_assert(!GEN || CORR, "drawn spectra are written back as position-space noise");
    static_assert(!CORR || GEN || MODE == 2, "transformed noise is written back only where it is scaled");
    typedef typename scalar_of<C>::type T;
    typedef RegFft<N> F;
    typedef ColR<N, C> CR;
    constexpr int PT = F::PT, W = CR::W;
    constexpr size_t RS = (size_t)F::T * N;             // elements between a thread's points
    const int col0 = xcd_strip(bi.bx, N / W) * W;
    Z += zofs_z(bi.bz, 4, V) + (size_t)bi.by * V;
    X += zofs_z(bi.bz, 8, V) + (size_t)bi.by * V;
    Y += zofs_z(bi.bz, 8, V) + (size_t)bi.by * V;
    // the thread's first element: uniform plane and row offsets, one 32-bit offset per thread
    auto at = [&]() -> unsigned {
        const int t = opaque_v(bi.tid);
        return (unsigned)((t / W) * N + col0 + t % W);
    };
    // where it goes: tiles on the large lattices' planes, except over planes that other
    // strips still read
    auto ot = [&](bool over) -> unsigned {
        const int t = opaque_v(bi.tid);
        if constexpr (BF == 3)
            if (!over) return (unsigned)Tile<N, C>::at(t / W, col0 + t % W);
        return (unsigned)((t / W) * N + col0 + t % W);
    };
    if constexpr (CR::TAB) {
        for (int i = threadIdx.x; i < N; i += blockDim.x) kt[i] = make_double2(q4[i], sb[i]);
        if constexpr (GEN) __syncthreads();             // otherwise the transforms' barriers do
    }
    C x[PT], y[PT], z[CORR ? PT : 1];
    int tk = bi.tid;
    if constexpr (!GEN) {
        const unsigned o = at();
#pragma unroll
        for (int r = 0; r < PT; r++) x[r] = (X + r * RS)[o];
#pragma unroll
        for (int r = 0; r < PT; r++) y[r] = (Y + r * RS)[o];        // in flight under the transform of X
        reg_fft_fwd<N, W, true>(x, lds, tw_fft(tw), opaque_v(bi.tid));
        reg_fft_fwd<N, W, false>(y, lds, tw_fft(tw), opaque_v(bi.tid));
        tk = after(tk, y[PT - 1].x);
    }
    const NoiseSrc nk = batch_noise_z(ns, V, bi.bz);
    const double invV = 1.0 / ((double)N * (double)N);
    const int j = tk / W, cy = col0 + tk % W, ky = freq_of_pos<N, BF>(cy);
    const int kx0 = reg_freq<N>(j / F::N3, j % F::N3, 0);
    const unsigned k0 = (unsigned)(kx0 * N + ky), s0 = (unsigned)(kx0 * N + cy);     // sa is stored by position
    const double q4y = q4[ky];
    const T sby = (T)sb[ky];
#pragma unroll
    for (int q = 0; q < PT; q++) {
        const int dk = reg_freq<N>(0, 0, q);            // kx = kx0 + dk
        if constexpr (GEN) {
            T g[4];
            kspace_normals4(k0 + (unsigned)(dk * N), nk.step, nk.tag, bi.by, nk.seed, nk.traj, g);
            x[q] = mkc<C>(g[0] * (T)N, g[1] * (T)N);            // sqrt(V) = N
            y[q] = mkc<C>(g[2] * (T)N, g[3] * (T)N);
        }
        double2 kq;
        if constexpr (CR::TAB) kq = kt[kx0 + dk];
        else kq = make_double2((q4 + dk)[kx0], (sb + dk)[kx0]);
        // kernel factors in the element type: one FP64 division per pair in FP64,
        // one FP32 division in the mixed form (whose spectra are FP32)
        const double cc = MODE == 1 ? (sa + (size_t)dk * N)[s0] : 1.0;
        T f = (T)(-2.0 * M_PI * invV * cc) / (T)(kq.x + q4y);
        if (q == 0 && k0 == 0) f = 0;
        const T fx = f * (T)kq.y, fy = f * sby;
        if constexpr (MODE == 2) {
            const T s = (T)(sa + (size_t)dk * N)[s0];
            x[q] = cscale(x[q], s);
            y[q] = cscale(y[q], s);
        }
        const C zq = C{-fma_t(fx, x[q].y, fy * y[q].y), fma_t(fx, x[q].x, fy * y[q].x)};   // i (fx x + fy y)
        // the fences end each element before the next (an interleaved order spills)
        if constexpr (CORR) {
            z[q] = zq;
            x[q] = cscale(x[q], (T)invV);
            y[q] = cscale(y[q], (T)invV);
            fence(y[q]);
            fence(z[q]);
        } else {
            x[q] = zq;
        }
        fence(x[q]);
    }
    reg_fft_inv<N, W, true>(x, lds, tw_fft(tw), opaque_v(bi.tid));
    {
        C* const O = CORR ? X : Z;
        const unsigned o = ot(CORR && !GEN);
#pragma unroll
        for (int r = 0; r < PT; r++) (O + r * RS)[o] = x[r];
    }
    if constexpr (CORR) {
        reg_fft_inv<N, W, false>(y, lds, tw_fft(tw), opaque_v(bi.tid));
        const unsigned oy = ot(!GEN);
#pragma unroll
        for (int r = 0; r < PT; r++) (Y + r * RS)[oy] = y[r];
        reg_fft_inv<N, W, false>(z, lds, tw_fft(tw), opaque_v(bi.tid));
        const unsigned oz = ot(false);
#pragma unroll
        for (int r = 0; r < PT; r++) (Z + r * RS)[oz] = z[r];
    }
}

template <int N, int CORR, int GEN, int MODE, int BF, typename C>
__global__ __launch_bounds__((ColR<N, C>::NT), (ColR<N, C>::WAVES)) void k_col_reg(
    C* __restrict__ Z, C* __restrict__ X, C* __restrict__ Y, size_t V, const double* __restrict__ q4,
    const double* __restrict__ sb, const double* __restrict__ sa, const C* __restrict__ tw, NoiseSrc ns) {
    __shared__ __align__(16) C lds[ColR<N, C>::LDS];
    col_reg_body<N, CORR, GEN, MODE, BF, C>(lds, reinterpret_cast<double2*>(lds + ColR<N, C>::ELEMS), own_block(), Z, X, Y,
                                        V, q4, sb, sa, tw, ns);
}

// ---------------------------------------------------------------------------
// column pass in LDS (the pair-interleaved layout, and the matrix-core stages on
// row-major planes): Z[p] = F_col^-1[ i (kx X^[p] + ky Y^[p]) / V ], X^ = F_col X
//   kx = -2 pi c pbarX / phat2 (c = sa(k) for SQRT, else 1), zero at k = 0.
//   CORR: X^, Y^ are first multiplied by sa(k) (per-mode correlated noise;
//   by 1 when noise_scale is 0) and F_col^-1[sa X^ / V] is written back over X
//   (likewise Y).
//   GEN (with CORR): X^, Y^ are not transformed from X, Y but drawn per mode
//   (kspace_normals4, plane pair p = blockIdx.y, noise key from ns); X and Y
//   then receive the row spectra of the position-space noise.
// X, Y: row spectra of plane p = blockIdx.y; strips of W columns.  PI: X is
// the pair-interleaved array (layout 2) holding both directions, Y unused.
// LDS row x holds [X(x, c0..c0+W-1), Y(x, c0..c0+W-1)]: 2W sequences of length N
// with element stride 2W.
// ---------------------------------------------------------------------------
// MF = 1, white noise (FP32 tiles of 74 KB, two per CU): registers of two
// workgroups asked for, as the FP32 butterfly version fits them by itself; the
// correlated variant needs more than that without spilling and runs one per CU
template <int N, int CORR, typename C, int PI = 0, int MF = 0, int GEN = 0>
__device__ __forceinline__ void col_kmult_body(C* lds, BlockIx bi, C* __restrict__ Z, C* __restrict__ X,
                                                          C* __restrict__ Y, size_t V, int sqrt_coupling,
                                                          const double* __restrict__ q4,
                                                          const double* __restrict__ sb,
                                                          const double* __restrict__ sa,
                                                          const C* __restrict__ tw, NoiseSrc ns, int noise_scale) {
    static_assert(!GEN || CORR, "drawn spectra are written back as position-space noise");
    typedef typename scalar_of<C>::type T;
    typedef ColE<N, C, CORR> CE;
    constexpr int W = CE::W, NT = CE::NT, PER = CE::PER, PAIRS = CE::PAIRS;
    constexpr int S2 = 2 * W, BF = PI ? 2 : 5;
    const int tid = bi.tid;
    const auto twl = tw_source<N, sizeof(C) == sizeof(float2)>(tw);
    const int strip = xcd_strip(bi.bx, N / W);
    const int col0 = strip * W;
    Z += zofs_z(bi.bz, 4, V);
    X += zofs_z(bi.bz, 8, V);
    Y += zofs_z(bi.bz, 8, V);
    const size_t pofs = (size_t)bi.by * V;
    const double invV = 1.0 / ((double)N * (double)N);
    // element e of the tile: row e / 2W, LDS slot s (X for s < W, Y above),
    // global offset g within X (PI: the pair-interleaved array) or Y
    auto elem = [&](int e, int& x, int& s, size_t& g) {
        x = e / S2;
        const int m = e % S2;
        if constexpr (PI) {
            s = (m & 1) * W + (m >> 1);
            g = 2 * pofs + 2 * ((size_t)x * N + col0) + m;
        } else {
            s = m;
            g = pofs + (size_t)x * N + col0 + (m % W);
        }
    };
    if constexpr (!GEN) {
#pragma unroll
        for (int q = 0; q < PER; q++) {
            int x, s;
            size_t g;
            elem(tid + q * NT, x, s, g);
            lds[lpos<S2, 1, 3>(x, s)] = (PI || s < W) ? X[g] : Y[g];
        }
        __syncthreads();
        lds_fft<N, S2, S2, 1, NT, -1, 3, MF>(lds, tw_fft(twl), opaque_v(tid));
    }
    const NoiseSrc nk = batch_noise_z(ns, V, bi.bz);
    // pair (x, c): X^ in slot c of LDS row x, Y^ in slot W + c
    C zreg[CORR ? PAIRS : 1];
    // FP32 correlated: indices recomputed per phase (opaque_v), since addresses
    // kept live across the FFTs would cost the registers of a second
    // workgroup per CU (measured 0.76 -> 0.70 ms per step at N = 2048)
    constexpr bool REIDX = CORR && sizeof(C) == sizeof(float2);
    const int tk = REIDX ? opaque_v(tid) : tid;
#pragma unroll
    for (int q = 0; q < PAIRS; q++) {
        const int pr = tk + q * NT;
        const int kx = pr / W, c = pr % W, ky = freq_of_pos<N, BF>(col0 + c);
        const size_t k = (size_t)kx * N + col0 + c;                 // sa is stored by position
        C vx, vy;
        if constexpr (GEN) {
            T g[4];
            kspace_normals4((uint32_t)(kx * N + ky), nk.step, nk.tag, bi.by, nk.seed, nk.traj, g);
            vx = mkc<C>(g[0] * (T)N, g[1] * (T)N);          // sqrt(V) = N
            vy = mkc<C>(g[2] * (T)N, g[3] * (T)N);
        } else {
            vx = lds[lpos<S2, 1, 3>(kx, c)];
            vy = lds[lpos<S2, 1, 3>(kx, W + c)];
        }
        // kernel factors in the element type: one FP64 division per pair in FP64,
        // one FP32 division in the mixed form (whose spectra are FP32)
        T fx = 0, fy = 0;
        if (kx != 0 || ky != 0) {
            const double cc = sqrt_coupling ? sa[k] : 1.0;
            const T f = (T)(-2.0 * M_PI * invV * cc) / (T)(q4[kx] + q4[ky]);
            fx = f * (T)sb[kx];
            fy = f * (T)sb[ky];
        }
        if (CORR) {
            if (noise_scale) {
                const T s = (T)sa[k];
                vx = cscale(vx, s);
                vy = cscale(vy, s);
            }
            lds[lpos<S2, 1, 3>(kx, c)] = cscale(vx, (T)invV);
            lds[lpos<S2, 1, 3>(kx, W + c)] = cscale(vy, (T)invV);
        }
        const C z = mkc<C>(-(fx * vx.y + fy * vy.y), fx * vx.x + fy * vy.x);   // i (fx vx + fy vy)
        if (CORR) zreg[q] = z;
        else lds[lpos<S2, 1, 3>(kx, c)] = z;
    }
    __syncthreads();
    if (CORR) {
        // xi~ = F_col^-1 of the scaled tiles, written back over X and Y
        lds_fft<N, S2, S2, 1, NT, +1, 3, MF>(lds, tw_fft(twl), opaque_v(tid));
        const int ts = REIDX ? opaque_v(tid) : tid;
#pragma unroll
        for (int q = 0; q < PER; q++) {
            int x, s;
            size_t g;
            elem(ts + q * NT, x, s, g);
            if (PI || s < W) X[g] = lds[lpos<S2, 1, 3>(x, s)];
            else Y[g] = lds[lpos<S2, 1, 3>(x, s)];
        }
        __syncthreads();
        const int tz = REIDX ? opaque_v(tid) : tid;
#pragma unroll
        for (int q = 0; q < PAIRS; q++) {
            const int pr = tz + q * NT;
            lds[lpos<S2, 1, 3>(pr / W, pr % W)] = zreg[q];
        }
        __syncthreads();
    }
    // Z: the W sequences in the X slots
    lds_fft<N, W, S2, 1, NT, +1, 3, MF>(lds, tw_fft(twl), opaque_v(tid));
    const int to = REIDX ? opaque_v(tid) : tid;
#pragma unroll
    for (int q = 0; q < PAIRS; q++) {
        const int pr = to + q * NT;
        const int x = pr / W, c = pr % W;
        Z[pofs + (size_t)x * N + col0 + c] = lds[lpos<S2, 1, 3>(x, c)];
    }
}

template <int N, int CORR, typename C, int PI = 0, int MF = 0, int GEN = 0>
__global__ __launch_bounds__((ColE<N, C, CORR>::NT), (MF && !CORR ? 2 * ColE<N, C, CORR>::NT / 256 : 1)) void k_col_kmult(C* __restrict__ Z, C* __restrict__ X,
                                                          C* __restrict__ Y, size_t V, int sqrt_coupling,
                                                          const double* __restrict__ q4,
                                                          const double* __restrict__ sb,
                                                          const double* __restrict__ sa,
                                                          const C* __restrict__ tw, NoiseSrc ns, int noise_scale) {
    __shared__ C lds[padded<N, 3>::value * 2 * ColE<N, C, CORR>::W];
    col_kmult_body<N, CORR, C, PI, MF, GEN>(lds, own_block(), Z, X, Y, V, sqrt_coupling, q4, sb, sa, tw, ns, noise_scale);
}

// ---------------------------------------------------------------------------
// column pass on the blocked layout: one workgroup per 128-byte column segment
// (CPB = 8 / BF adjacent columns) and plane pair p, one plane at a time in LDS:
//   X^ = F_col X[p]  ->  acc = i fx X^       (CORR: X^ *= sa, X[p] <- F_col^-1[X^ / V])
//   Y^ = F_col Y[p]  ->  acc += i fy Y^      (CORR: likewise for Y[p])
//   Z[p] = F_col^-1 acc
// with fx, fy, sa as in k_col_kmult.  Element e of a loaded segment set is
// x-block e / 8, slot e mod 8 = c BF + x mod BF: consecutive threads read
// consecutive 16-byte words.  sa16 holds sa(k) in 16-row blocks.
// ---------------------------------------------------------------------------
template <int N, int BF, typename C>
struct ColB {
    // BF = 4, 8: one 128-byte segment (SEG elements) holds CPB columns of BF rows;
    // BF = 1 (row-major): 64-byte row segments of CPB adjacent columns;
    // BF = 16 (row-major): 32-byte row segments (two workgroups per CU in FP64
    // at N = 2048); BF = 32 (row-major): 16-byte row segments, the strip that
    // fits LDS at N = 8192 (one FP64 or two FP32 columns, 139 KB)
    static constexpr int RB = (BF == 1 || BF >= 16) ? 1 : BF;     // rows per block of the layout
    static constexpr int SEG = BF == 1    ? 64 / (int)sizeof(C)
                               : BF == 16 ? 32 / (int)sizeof(C)
                               : BF == 32 ? 16 / (int)sizeof(C)
                                          : 128 / (int)sizeof(C);
    static constexpr int CPB = SEG / RB;               // columns per workgroup
    static constexpr int ELEMS = CPB * N;
    static constexpr int NTMAX = (BF == 1 || BF == 32) ? 1024 : 512;
    static constexpr int NT = (ELEMS / 8 < 64) ? 64 : ((ELEMS / 8 > NTMAX) ? NTMAX : ELEMS / 8);
    static constexpr int PER = ELEMS / NT;             // elements per thread
    static constexpr int LDS_BYTES = CPB * padded<N, 4>::value * (int)sizeof(C);
    // the row-major narrow strips ask for the registers of two workgroups per
    // CU where their LDS allows two
    static constexpr int WAVES = (BF >= 16 && 2 * LDS_BYTES <= 160 * 1024) ? (NT * 2 + 255) / 256 : 1;
    static_assert((BF == 1 || BF == 4 || BF == 8 || BF == 16 || BF == 32) && CPB >= 1 && CPB <= N &&
                      PER * NT == ELEMS && N % 16 == 0 && N % CPB == 0,
                  "blocked column tiling");
};

template <int N, int BF, int CORR, typename C, int GEN = 0, int MF = 0>
__global__ __launch_bounds__((ColB<N, BF, C>::NT), (ColB<N, BF, C>::WAVES)) void k_col_kmult_blk(C* __restrict__ Z, C* __restrict__ X,
                                                                     C* __restrict__ Y, size_t V, int sqrt_coupling,
                                                                     const double* __restrict__ q4,
                                                                     const double* __restrict__ sb,
                                                                     const double* __restrict__ sa16,
                                                                     const C* __restrict__ tw, NoiseSrc ns,
                                                                     int noise_scale) {
    static_assert(!GEN || CORR, "drawn spectra are written back as position-space noise");
    typedef typename scalar_of<C>::type T;
    constexpr int SEG = ColB<N, BF, C>::SEG, CPB = ColB<N, BF, C>::CPB, RB = ColB<N, BF, C>::RB;
    constexpr int NT = ColB<N, BF, C>::NT, PER = ColB<N, BF, C>::PER;
    constexpr int PN = padded<N, 4>::value;
    __shared__ C lds[CPB * PN];
    const int tid = threadIdx.x;
    const auto twl = tw_source<N, true>(tw);
    Z += zofs(4, V);
    X += zofs(8, V);
    Y += zofs(8, V);
    // 32-byte strips: the four strips of one 128-byte line on one XCD at neighbouring times
    const int y0 = (BF >= 16 ? xcd_strip(blockIdx.x, N / CPB) : (int)blockIdx.x) * CPB;
    const double invV = 1.0 / ((double)N * (double)N);
    // global offset within a plane / LDS slot of loaded element e: x-block
    // e / SEG, slot e mod SEG = c BF + x mod BF (row-major, BF = 1: row e / SEG,
    // column y0 + e mod SEG)
    auto goff = [&](int e) -> size_t { return (size_t)(e / SEG) * ((size_t)N * RB) + (size_t)y0 * RB + (e % SEG); };
    auto lofs = [&](int e) -> int {
        const int sl = e % SEG;
        return lpos<1, PN, 4>((e / SEG) * RB + sl % RB, sl / RB);
    };
    auto load = [&](const C* __restrict__ P) {
        const int t = opaque_v(tid);
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int e = t + q * NT;
            lds[lofs(e)] = P[goff(e)];
        }
    };
    auto store = [&](C* __restrict__ P) {
        const int t = opaque_v(tid);
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int e = t + q * NT;
            P[goff(e)] = lds[lofs(e)];
        }
    };
    // one direction d (0: x, 1: y): forward column FFT of P, accumulate
    // i f_d P^ into acc for this thread's pairs (kx = pr mod N, column c = pr / N)
    // with f_d = -2 pi cc sb[k_d] / phat^2 / V, zero at k = 0; CORR: scale P^
    // by sa (noise_scale) and write F_col^-1[sa P^ / V] back over P.  GEN: P^
    // drawn per mode instead; the x direction's draw also gives the y spectrum
    // (held in yg until then).
    const NoiseSrc nk = batch_noise(ns, V);
    C yg[GEN ? PER : 1];
    auto direction = [&](C* __restrict__ P, C acc[PER], int d) {
        const double* q4d = opaque(q4);
        const double* sbd = opaque(sb);
        const double* sad = opaque(sa16);
        if constexpr (!GEN) {
            load(P);
            __syncthreads();
            lds_fft<N, CPB, 1, PN, NT, -1, 4, MF>(lds, tw_fft(twl), opaque_v(tid));
        }
        const int t = opaque_v(tid);
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int pr = t + q * NT;
            const int kx = pr % N, c = pr / N, ky = freq_of_pos<N, BF>(y0 + c);
            const int l = lpos<1, PN, 4>(kx, c);
            const size_t k16 = ((size_t)(kx >> 4) * N + y0 + c) * 16 + (kx & 15);      // sa16 is stored by position
            C v;
            if constexpr (GEN) {
                if (d == 0) {
                    T g[4];
                    kspace_normals4((uint32_t)((size_t)kx * N + ky), nk.step, nk.tag, blockIdx.y, nk.seed, nk.traj, g);
                    v = mkc<C>(g[0] * (T)N, g[1] * (T)N);      // sqrt(V) = N
                    yg[q] = mkc<C>(g[2] * (T)N, g[3] * (T)N);
                } else {
                    v = yg[q];
                }
            } else {
                v = lds[l];
            }
            if (CORR) {
                if (noise_scale) v = cscale(v, (T)sad[k16]);
                lds[l] = cscale(v, (T)invV);
            }
            T f = 0;
            if (kx != 0 || ky != 0) {
                const double cc = sqrt_coupling ? sad[k16] : 1.0;
                f = (T)(-2.0 * M_PI * invV * cc) / (T)(q4d[kx] + q4d[ky]) * (T)sbd[d ? ky : kx];
            }
            if (d == 0) acc[q] = mkc<C>(-(f * v.y), f * v.x);
            else acc[q] = mkc<C>(acc[q].x - f * v.y, acc[q].y + f * v.x);
        }
        __syncthreads();
        if (CORR) {
            lds_fft<N, CPB, 1, PN, NT, +1, 4, MF>(lds, tw_fft(twl), opaque_v(tid));
            store(P);
            __syncthreads();
        }
    };
    // plane pair p = blockIdx.y (one pass over the pairs would let the compiler
    // hoist every twiddle and kernel factor out of the loop into registers)
    const size_t po = (size_t)blockIdx.y * V;
    C acc[PER];
    direction(X + po, acc, 0);
    direction(Y + po, acc, 1);
    const int t = opaque_v(tid);
#pragma unroll
    for (int q = 0; q < PER; q++) {
        const int pr = t + q * NT;
        lds[lpos<1, PN, 4>(pr % N, pr / N)] = acc[q];
    }
    __syncthreads();
    lds_fft<N, CPB, 1, PN, NT, +1, 4, MF>(lds, tw_fft(twl), opaque_v(tid));
    store(Z + po);
}


// ---------------------------------------------------------------------------
// row pass 3: inverse row FFTs of the A and B column-inverse spectra and the
// update U <- exp(i s B) U exp(-i s A) (field.h:1966-1996) in one pass.
// A's coefficients are kept in registers, B's stay in LDS.  The site algebra
// (exponentials, products, the optional projection onto SU(3)) is FP64 in both
// forms; U is stored in the element type C.
// ---------------------------------------------------------------------------
template <int N, int BF, typename C>
__device__ __forceinline__ void row_update_body(C* lds, BlockIx bi, C* __restrict__ U, const C* __restrict__ ZA,
                                                              const C* __restrict__ ZB, size_t V, double ss,
                                                              int reunit, int whole, const C* __restrict__ tw, int next_noise,
                                                              C* __restrict__ Xi, NoiseSrc ns,
                                                              const double* __restrict__ sa_pos) {
    typedef typename scalar_of<C>::type T;
    constexpr int NT = RowE<N>::NT, SPT = RowE<N>::SPT, PL = RowT<N, C>::PL;
    const int tid = bi.tid;
    U += zofs_z(bi.bz, UPlanes<C>::value, V);
    ZA += zofs_z(bi.bz, 4, V);
    ZB += zofs_z(bi.bz, 4, V);
    const int x = row_of_block<N, BF>(bi.bx);
    const size_t row0 = (size_t)x * N;
    C za[RowE<N>::PT], zb[RowE<N>::PT];
    row_load<N, BF>(za, tid, [&](int p, int k) { return ZA[p * V + lay<N, BF>(x, k)]; });
    row_load<N, BF>(zb, tid, [&](int p, int k) { return ZB[p * V + lay<N, BF>(x, k)]; });
    row_inv<N, true>(za, lds, tw, tid);
    __syncthreads();
    T ha[SPT][8];
#pragma unroll
    for (int q = 0; q < SPT; q++)
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const C a = lds[p * PL + row_slot_of<N, C>(tid + q * NT)];
            ha[q][2 * p] = a.x;
            ha[q][2 * p + 1] = a.y;
        }
    row_inv<N, false>(zb, lds, tw, tid);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < SPT; q++) {
        const int y = site_of<C>(tid + q * NT);
        const size_t i = row0 + y;
        T hb[8];
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const C b = lds[p * PL + row_slot_of<N, C>(y)];
            hb[2 * p] = b.x;
            hb[2 * p + 1] = b.y;
        }
        if constexpr (sizeof(C) == sizeof(double2)) {
            m3 u;
            load_u(u, U, V, i);
            m3 w = mmul(exp_i_gen(hb, ss), u);
            double hd[8];
#pragma unroll
            for (int k = 0; k < UPlanes<C>::value; k++) fence(w.m[k]);      // the rows that are stored
#pragma unroll
            for (int k = 0; k < 8; k++) {
                hd[k] = ha[q][k];
                fence(hd[k]);
            }
            m3 r = mmul(w, exp_i_gen(hd, -ss));
            if (reunit) r = su3_project(r);
            store_u(U, V, i, r);
            if (whole) {        // a call's last step leaves all nine entries
                row2_of(r.m);
#pragma unroll
                for (int k = 6; k < 9; k++) U[k * V + i] = r.m[k];
            }
        } else {
            // FP64 exponentials, FP32 products; the projection in FP64.  The
            // fences keep the two exponentials apart (fewer live registers).
            const m3f eb = exp_i_gen_f(hb, ss);
            m3f u;
            load_u(u, U, V, i);
            m3f w = mmul(eb, u);
            T hd[8];
#pragma unroll
            for (int k = 0; k < UPlanes<C>::value; k++) fence(w.m[k]);      // the rows that are stored
#pragma unroll
            for (int k = 0; k < 8; k++) {
                hd[k] = ha[q][k];
                fence(hd[k]);
            }
            m3f r = mmul(w, exp_i_gen_f(hd, -ss));
            if (reunit) r = to_f(su3_project(to_d(r)));
            store_u(U, V, i, r);
        }
    }
    if (next_noise) {        // the next step's xi row spectra
        __syncthreads();
        NoiseSrc nn = batch_noise_z(ns, V, bi.bz);
        nn.step += 1;
        row_noise_body<N, BF, C>(lds, Xi + zofs_z(bi.bz, 8, V), V, nn, sa_pos, tw, x, bi.tid);
    }
}

template <int N, int BF, typename C>
__global__ __launch_bounds__(RowE<N>::NT, RowWaves<C>::value) void k_row_update(C* __restrict__ U, const C* __restrict__ ZA,
                                                              const C* __restrict__ ZB, size_t V, double ss,
                                                              int reunit, int whole, const C* __restrict__ tw, int next_noise,
                                                              C* __restrict__ Xi, NoiseSrc ns,
                                                              const double* __restrict__ sa_pos) {
    __shared__ C lds[4 * RowT<N, C>::PL];
    row_update_body<N, BF, C>(lds, own_block(), U, ZA, ZB, V, ss, reunit, whole, tw, next_noise, Xi, ns, sa_pos);
}

// ---------------------------------------------------------------------------
// One launch per kernel class over every size group of a batch (row-major
// intermediate planes).  Block b of a launch belongs to the group whose block
// range holds it.  A group whose body needs NT threads, fewer than the T of
// the launch, runs T / NT bodies side by side in the block (rows, or column
// strips), each on its own thread range and its own part of LDS; all bodies
// of one block have the same N, so the barriers inside them coincide.
// ---------------------------------------------------------------------------
template <typename C>
struct GroupRun {
    int N, nblk;                      // lattice size, blocks of this group in the launch
    C *U, *Xi, *Vv, *ZA, *ZB;         // the group's trajectories, as for one grouped launch
    size_t V;
    NoiseSrc ns;                      // key of the group's first trajectory
    const double *sa_pos, *sa_k, *q4, *sb;
    const C* tw;
};
template <typename C>
struct MultiRun {
    int ng;
    GroupRun<C> g[JW_MAX_GROUPS];
};

// the group of launch block b; b becomes the block's index inside the group
template <typename C>
__device__ __forceinline__ const GroupRun<C>& group_of(const MultiRun<C>& m, int& b) {
    int g = 0;
    while (g < m.ng - 1 && b >= m.g[g].nblk) {
        b -= m.g[g].nblk;
        g++;
    }
    return m.g[g];
}

template <int N>
using int_c = std::integral_constant<int, N>;

// f(int_c<N>, group, block index in the group) for the block's group, N from
// the sizes a launch of T threads can hold (threads per body = MAXNT(N) <= T)
template <int T, template <int> class NTOF, typename C, typename F>
__device__ __forceinline__ void dispatch_group(const MultiRun<C>& m, F&& f) {
    int b = blockIdx.x;
    const GroupRun<C>& g = group_of(m, b);
    switch (g.N) {
        case 64: if constexpr (NTOF<64>::value <= T) f(int_c<64>{}, g, b); break;
        case 128: if constexpr (NTOF<128>::value <= T) f(int_c<128>{}, g, b); break;
        case 256: if constexpr (NTOF<256>::value <= T) f(int_c<256>{}, g, b); break;
        case 512: if constexpr (NTOF<512>::value <= T) f(int_c<512>{}, g, b); break;
        case 1024: if constexpr (NTOF<1024>::value <= T) f(int_c<1024>{}, g, b); break;
        case 2048: if constexpr (NTOF<2048>::value <= T) f(int_c<2048>{}, g, b); break;
        default: break;
    }
}
template <int N> struct RowNT { static constexpr int value = RowE<N>::NT; };
template <typename C>
struct ColNT { template <int N> struct of { static constexpr int value = ColR<N, C>::NT; }; };
// threads of a column launch: the strips of every size have at most that many,
// at the registers of ColR
template <typename C>
struct ColMultiT { static constexpr int value = sizeof(C) == sizeof(double2) ? 512 : 1024; };

// LDS of a row launch of T threads: T / NT bodies of `planes` padded rows
template <int T, int planes, typename C>
struct RowMultiLds {
    template <int N>
    static constexpr int NT() { return planes == 1 ? RegFft<N>::T : RowE<N>::NT; }
    template <int N>
    static constexpr int need() { return NT<N>() <= T ? (T / NT<N>()) * planes * RowT<N, C>::PL : 0; }
    static constexpr int a = need<64>() > need<128>() ? need<64>() : need<128>();
    static constexpr int b = need<256>() > need<512>() ? need<256>() : need<512>();
    static constexpr int c = need<1024>() > need<2048>() ? need<1024>() : need<2048>();
    static constexpr int ab = a > b ? a : b;
    static constexpr int value = ab > c ? ab : c;
};
// LDS of a column launch: the bodies' tiles, then the (q4, sb) table they share
template <typename C>
struct ColMultiLds {
    template <int N>
    static constexpr int need() {
        return (ColMultiT<C>::value / ColR<N, C>::NT) * ColR<N, C>::ELEMS + N * 16 / (int)sizeof(C);
    }
    static constexpr int a = need<64>() > need<128>() ? need<64>() : need<128>();
    static constexpr int b = need<256>() > need<512>() ? need<256>() : need<512>();
    static constexpr int c = need<1024>() > need<2048>() ? need<1024>() : need<2048>();
    static constexpr int ab = a > b ? a : b;
    static constexpr int value = ab > c ? ab : c;
    static_assert(value * sizeof(C) <= 160 * 1024, "LDS of a column launch");
};

// the row (x), trajectory (z) and thread of a row body in block b of its group
template <int N, int T>
__device__ __forceinline__ BlockIx row_slot(int b) {
    constexpr int NT = RowE<N>::NT, RPB = T / NT, NRB = N / RPB;
    const int s = threadIdx.x / NT;
    return BlockIx{(b % NRB) * RPB + s, 0, b / NRB, (int)threadIdx.x % NT};
}
template <int N, int T>
__device__ __forceinline__ int row_sub() { return threadIdx.x / RowE<N>::NT; }

// noise: T / (threads of a row) rows of one plane pair in a block; plane pairs, then trajectories
template <int N> struct RowNoiseNT { static constexpr int value = RegFft<N>::T; };
template <typename C, int T>
__global__ __launch_bounds__(T, RowWaves<C>::value) void k_row_noise_fwd_multi(MultiRun<C> m) {
    __shared__ C lds[RowMultiLds<T, 1, C>::value];
    dispatch_group<T, RowNoiseNT>(m, [&](auto n, const GroupRun<C>& g, int b) {
        constexpr int N = decltype(n)::value;
        constexpr int TR = RegFft<N>::T, RPB = T / TR, NRB = N / RPB;
        const int s = threadIdx.x / TR;
        const BlockIx bi{(b % NRB) * RPB + s, (b / NRB) % 4, b / (NRB * 4), (int)threadIdx.x % TR};
        row_noise_fwd_body<N, 0, C>(lds + s * RowT<N, C>::PL, bi, g.Xi, g.V, g.ns, g.sa_pos, g.tw);
    });
}
template <typename C, int T>
__global__ __launch_bounds__(T, RowWaves<C>::value) void k_row_uxiu_fwd_multi(MultiRun<C> m) {
    __shared__ C lds[RowMultiLds<T, 4, C>::value];
    dispatch_group<T, RowNT>(m, [&](auto n, const GroupRun<C>& g, int b) {
        constexpr int N = decltype(n)::value;
        row_uxiu_fwd_body<N, 0, C>(lds + row_sub<N, T>() * 4 * RowT<N, C>::PL, row_slot<N, T>(b), g.Vv, g.U, g.V,
                                   g.ns, g.sa_pos, g.tw);
    });
}
template <typename C, int T>
__global__ __launch_bounds__(T, RowWaves<C>::value) void k_row_uxiu_corr_multi(MultiRun<C> m) {
    __shared__ C lds[RowMultiLds<T, 4, C>::value];
    dispatch_group<T, RowNT>(m, [&](auto n, const GroupRun<C>& g, int b) {
        constexpr int N = decltype(n)::value;
        row_uxiu_corr_body<N, 0, C>(lds + row_sub<N, T>() * 4 * RowT<N, C>::PL, row_slot<N, T>(b), g.Vv, g.U, g.Xi,
                                    g.V, g.tw);
    });
}
template <typename C, int T>
__global__ __launch_bounds__(T, RowWaves<C>::value) void k_row_update_multi(MultiRun<C> m, double ss, int reunit) {
    __shared__ C lds[RowMultiLds<T, 4, C>::value];
    dispatch_group<T, RowNT>(m, [&](auto n, const GroupRun<C>& g, int b) {
        constexpr int N = decltype(n)::value;
        row_update_body<N, 0, C>(lds + row_sub<N, T>() * 4 * RowT<N, C>::PL, row_slot<N, T>(b), g.U, g.ZA, g.ZB,
                                 g.V, ss, reunit, 0, g.tw, 0, g.Xi, g.ns, g.sa_pos);
    });
}
// column passes: the strips of a group in the order strip, plane pair, trajectory
// (the order of the grouped launch's grid), T / NT of one trajectory in a block
template <typename C, int CORR, int GEN, int MODE>
__global__ __launch_bounds__((ColMultiT<C>::value), (ColR<2048, C>::WAVES)) void k_col_reg_multi(MultiRun<C> m, int use_v) {
    __shared__ __align__(16) C lds[ColMultiLds<C>::value];
    constexpr int T = ColMultiT<C>::value;
    dispatch_group<T, ColNT<C>::template of>(m, [&](auto n, const GroupRun<C>& g, int b) {
        constexpr int N = decltype(n)::value;
        typedef ColR<N, C> CR;
        constexpr int SPB = T / CR::NT, NS = N / CR::W, NB = 4 * NS / SPB;      // blocks of a trajectory
        const int s = threadIdx.x / CR::NT, u = (b % NB) * SPB + s;
        const BlockIx bi{u % NS, u / NS, b / NB, (int)threadIdx.x % CR::NT};
        C* X = use_v ? g.Vv : g.Xi;
        col_reg_body<N, CORR, GEN, MODE, 0, C>(lds + s * CR::ELEMS, reinterpret_cast<double2*>(lds + SPB * CR::ELEMS), bi,
                                            use_v ? g.ZB : g.ZA, X, X + 4 * g.V, g.V, g.q4, g.sb, g.sa_k, g.tw, g.ns);
    });
}

// f(int_c<N>) for a batch size
template <typename F>
inline int for_size(int N, F&& f) {
    switch (N) {
        case 64: return f(int_c<64>{});
        case 128: return f(int_c<128>{});
        case 256: return f(int_c<256>{});
        case 512: return f(int_c<512>{});
        case 1024: return f(int_c<1024>{});
        default: return f(int_c<2048>{});
    }
}
// blocks of group g in a row launch of T threads, in the noise launch and in a
// column launch
inline int row_blocks(int N, int count, int T) {
    return for_size(N, [&](auto n) { constexpr int M = decltype(n)::value; return count * M / (T / RowE<M>::NT); });
}
inline int noise_blocks(int N, int count, int T) {
    return for_size(N, [&](auto n) { constexpr int M = decltype(n)::value; return count * 4 * (M / (T / RegFft<M>::T)); });
}
template <typename C>
inline int col_blocks(int N, int count) {
    return for_size(N, [&](auto n) {
        constexpr int M = decltype(n)::value;
        constexpr int SPB = ColMultiT<C>::value / ColR<M, C>::NT;
        constexpr int units = 4 * (M / ColR<M, C>::W);      // strips of the four plane pairs
        static_assert(SPB >= 1 && units % SPB == 0, "strips of a block");
        return count * (units / SPB);
    });
}

// one step of every group of a batch, one launch per kernel class (row-major
// planes; the noise pass separate from the update).  counts[g]: trajectories.
template <typename C>
static hipError_t step_multi_t(hipStream_t st, MultiRun<C> m, const int* counts, int maxN, const StepArgs& a) {
    if (m.ng < 1 || m.ng > JW_MAX_GROUPS) return hipErrorInvalidValue;
    const int T = maxN > 1024 ? 512 : 256;
    int nrow = 0, ncol = 0, nnoise = 0;
    for (int g = 0; g < m.ng; g++) {
        if (m.g[g].N < 64 || m.g[g].N > 2048) return hipErrorInvalidValue;
        nrow += row_blocks(m.g[g].N, counts[g], T);
        nnoise += noise_blocks(m.g[g].N, counts[g], T);
        ncol += col_blocks<C>(m.g[g].N, counts[g]);
    }
    auto set_blocks = [&](bool col) {
        for (int g = 0; g < m.ng; g++)
            m.g[g].nblk = col ? col_blocks<C>(m.g[g].N, counts[g]) : row_blocks(m.g[g].N, counts[g], T);
    };
    const int wb = a.corr || a.kspace;
    hipError_t e;
    if (!a.kspace) {
        for (int g = 0; g < m.ng; g++) m.g[g].nblk = noise_blocks(m.g[g].N, counts[g], T);
        if (T == 256) hipLaunchKernelGGL((k_row_noise_fwd_multi<C, 256>), dim3(nnoise), dim3(256), 0, st, m);
        else hipLaunchKernelGGL((k_row_noise_fwd_multi<C, 512>), dim3(nnoise), dim3(512), 0, st, m);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    set_blocks(true);
    constexpr int TC = ColMultiT<C>::value;
#define JW_COL_MULTI(corr, gen, mode, use_v) \
    hipLaunchKernelGGL((k_col_reg_multi<C, corr, gen, mode>), dim3(ncol), dim3(TC), 0, st, m, use_v)
    if (a.kspace) {
        if (a.corr) JW_COL_MULTI(1, 1, 2, 0);
        else if (a.sqrt_coupling) JW_COL_MULTI(1, 1, 1, 0);
        else JW_COL_MULTI(1, 1, 0, 0);
    } else if (a.corr) {
        JW_COL_MULTI(1, 0, 2, 0);
    } else if (a.sqrt_coupling) {
        JW_COL_MULTI(0, 0, 1, 0);
    } else {
        JW_COL_MULTI(0, 0, 0, 0);
    }
    if ((e = hipGetLastError()) != hipSuccess) return e;
    set_blocks(false);
    if (wb) {
        if (T == 256) hipLaunchKernelGGL((k_row_uxiu_corr_multi<C, 256>), dim3(nrow), dim3(256), 0, st, m);
        else hipLaunchKernelGGL((k_row_uxiu_corr_multi<C, 512>), dim3(nrow), dim3(512), 0, st, m);
    } else {
        if (T == 256) hipLaunchKernelGGL((k_row_uxiu_fwd_multi<C, 256>), dim3(nrow), dim3(256), 0, st, m);
        else hipLaunchKernelGGL((k_row_uxiu_fwd_multi<C, 512>), dim3(nrow), dim3(512), 0, st, m);
    }
    if ((e = hipGetLastError()) != hipSuccess) return e;
    set_blocks(true);
    if (a.sqrt_coupling) JW_COL_MULTI(0, 0, 1, 1);
    else JW_COL_MULTI(0, 0, 0, 1);
#undef JW_COL_MULTI
    if ((e = hipGetLastError()) != hipSuccess) return e;
    set_blocks(false);
    if (T == 256)
        hipLaunchKernelGGL((k_row_update_multi<C, 256>), dim3(nrow), dim3(256), 0, st, m, a.sqrt_step, a.reunit);
    else
        hipLaunchKernelGGL((k_row_update_multi<C, 512>), dim3(nrow), dim3(512), 0, st, m, a.sqrt_step, a.reunit);
    return hipGetLastError();
}

// the batch's groups as one MultiRun (at most JW_MAX_GROUPS)
template <typename C>
static hipError_t step_multi_from(hipStream_t st, const GroupArgs* ga, int ng, const StepArgs& a) {
    if (ng < 1 || ng > JW_MAX_GROUPS) return hipErrorInvalidValue;
    MultiRun<C> m{};
    int counts[JW_MAX_GROUPS], maxN = 0;
    m.ng = ng;
    for (int g = 0; g < ng; g++) {
        const GroupArgs& s = ga[g];
        m.g[g] = GroupRun<C>{s.N, 0, (C*)s.U, (C*)s.Xi, (C*)s.Vv, (C*)s.ZA, (C*)s.ZB, s.V, s.ns,
                             s.sa_pos, s.sa_k, s.q4, s.sb, (const C*)s.tw};
        counts[g] = s.count;
        maxN = s.N > maxN ? s.N : maxN;
    }
    return step_multi_t<C>(st, m, counts, maxN, a);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
template <typename C>
static const C* twiddles(const jw_ctx* c) {
    if constexpr (sizeof(C) == sizeof(cplx)) return c->tw;
    else return c->twf;
}

// corr: the correlated-noise variant (xi~ written back); gen: the xi spectra
// drawn per mode from ns (implies the write-back); noise_scale: the drawn or
// transformed spectra are multiplied by sa (correlated coupling)
template <int N, int BF, typename C>
static hipError_t col_pass(jw_ctx* c, C* Z, C* X, C* Y, const double* sa_k, int sqrt_coupling, int corr,
                           int nbatch, const NoiseSrc& ns, int gen, int noise_scale) {
    const size_t V = c->V;
    const C* tw = twiddles<C>(c);
#define JW_COL_ARGS Z, X, Y, V, sqrt_coupling, c->q4, c->sb, sa_k, tw, ns, noise_scale
    if constexpr (BF == 5) {
        // split-BF16 matrix-core radix-16 stages (FP32 storage)
        const dim3 grid(N / ColE<N, C>::W, 4, nbatch);
        if (gen)
            hipLaunchKernelGGL((k_col_kmult<N, 1, C, 0, 1, 1>), grid, dim3(ColE<N, C, 1>::NT), 0, c->stream, JW_COL_ARGS);
        else if (corr)
            hipLaunchKernelGGL((k_col_kmult<N, 1, C, 0, 1>), grid, dim3(ColE<N, C, 1>::NT), 0, c->stream, JW_COL_ARGS);
        else
            hipLaunchKernelGGL((k_col_kmult<N, 0, C, 0, 1>), grid, dim3(ColE<N, C, 0>::NT), 0, c->stream, JW_COL_ARGS);
    } else if constexpr (BF == 0 || BF == 3) {
        typedef ColR<N, C> CR;
        const dim3 grid(N / CR::W, 4, nbatch);
#define JW_COL_REG(corr_, gen_, mode_)                                                                               \
    hipLaunchKernelGGL((k_col_reg<N, corr_, gen_, mode_, BF, C>), grid, dim3(CR::NT), 0, c->stream, Z, X, Y, V, c->q4, \
                       c->sb, sa_k, tw, ns)
        if (gen) {
            if (noise_scale) JW_COL_REG(1, 1, 2);
            else if (sqrt_coupling) JW_COL_REG(1, 1, 1);
            else JW_COL_REG(1, 1, 0);
        } else if (corr) {
            JW_COL_REG(1, 0, 2);
        } else if (sqrt_coupling) {
            JW_COL_REG(0, 0, 1);
        } else {
            JW_COL_REG(0, 0, 0);
        }
#undef JW_COL_REG
    } else if constexpr (BF == 2) {
        const dim3 grid(N / ColE<N, C>::W, 4, nbatch);
        if (gen)
            hipLaunchKernelGGL((k_col_kmult<N, 1, C, 1, 0, 1>), grid, dim3(ColE<N, C, 1>::NT), 0, c->stream, JW_COL_ARGS);
        else if (corr)
            hipLaunchKernelGGL((k_col_kmult<N, 1, C, 1>), grid, dim3(ColE<N, C, 1>::NT), 0, c->stream, JW_COL_ARGS);
        else
            hipLaunchKernelGGL((k_col_kmult<N, 0, C, 1>), grid, dim3(ColE<N, C, 0>::NT), 0, c->stream, JW_COL_ARGS);
    } else {
        constexpr int CPB = ColB<N, BF, C>::CPB, NT = ColB<N, BF, C>::NT;
        const dim3 grid(N / CPB, 4, nbatch);
        // the matrix-core stages in the 16-byte strips of the large lattices
        if constexpr (sizeof(C) == sizeof(float2) && BF == 32) {
            if (c->fft_mfma) {
                if (gen)
                    hipLaunchKernelGGL((k_col_kmult_blk<N, BF, 1, C, 1, 1>), grid, dim3(NT), 0, c->stream, JW_COL_ARGS);
                else if (corr)
                    hipLaunchKernelGGL((k_col_kmult_blk<N, BF, 1, C, 0, 1>), grid, dim3(NT), 0, c->stream, JW_COL_ARGS);
                else
                    hipLaunchKernelGGL((k_col_kmult_blk<N, BF, 0, C, 0, 1>), grid, dim3(NT), 0, c->stream, JW_COL_ARGS);
                return hipGetLastError();
            }
        }
        if (gen)
            hipLaunchKernelGGL((k_col_kmult_blk<N, BF, 1, C, 1>), grid, dim3(NT), 0, c->stream, JW_COL_ARGS);
        else if (corr)
            hipLaunchKernelGGL((k_col_kmult_blk<N, BF, 1, C>), grid, dim3(NT), 0, c->stream, JW_COL_ARGS);
        else
            hipLaunchKernelGGL((k_col_kmult_blk<N, BF, 0, C>), grid, dim3(NT), 0, c->stream, JW_COL_ARGS);
    }
#undef JW_COL_ARGS
    return hipGetLastError();
}

template <int N, int BF, typename C>
static hipError_t step_fused_n(jw_ctx* c, C* U, C* Xi, C* Vv, C* ZA, C* ZB, const StepArgs& a, const int* kcls) {
    const size_t V = c->V;
    const C* tw = twiddles<C>(c);
    hipError_t e;
    // The next step's noise rides on the update pass up to N = 1024, where that is
    // faster: its instructions hide under the update's memory time, and a launch goes (us a
    // step, fixed coupling, separate -> fused, FP64 / FP32: N = 64 26.8 -> 23.8 / 24.7 ->
    // 22.3; 256 57.0 -> 53.9 / 42.1 -> 40.3; 512 95.9 -> 91.3 / 64.2 -> 61.2; 1024 365 ->
    // 353 / 187 -> 182).  At 2048 it is slower in FP64 (1449 -> 1507), whose update then
    // runs with one workgroup a CU, and the same in FP32 (766 -> 763, correlated 894 -> 897).
    // Momentum-space noise (a.kspace): no noise pass; the first column pass
    // draws the spectra and writes the position-space noise's row spectra back
    // for the correlated row pass.
    constexpr bool fuse_noise = N <= 1024;
    const int first_noise = a.kspace ? 0 : fuse_noise ? a.first_noise : 1;
    const int next_noise = a.kspace ? 0 : fuse_noise ? a.next_noise : 0;
    if (first_noise) {
        KTimer t(c, kcls[0]);
        hipLaunchKernelGGL((k_row_noise_fwd<N, BF, C>), dim3(N / RowN<N>::RPW, 4, a.nbatch), dim3(RowN<N>::NT), 0, c->stream, Xi, V, a.ns,
                           a.sa_pos, tw);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    {
        KTimer t(c, kcls[1]);
        if ((e = col_pass<N, BF>(c, ZA, Xi, Xi + 4 * V, a.sa_k, a.sqrt_coupling, a.corr, a.nbatch, a.ns, a.kspace,
                                 a.corr)) != hipSuccess)
            return e;
    }
    {
        KTimer t(c, kcls[2]);
        if (a.corr || a.kspace)
            hipLaunchKernelGGL((k_row_uxiu_corr<N, BF, C>), dim3(N, 1, a.nbatch), dim3(RowE<N>::NT), 0, c->stream, Vv, U, Xi, V,
                               tw);
        else
            hipLaunchKernelGGL((k_row_uxiu_fwd<N, BF, C>), dim3(N, 1, a.nbatch), dim3(RowE<N>::NT), 0, c->stream, Vv, U, V, a.ns,
                               a.sa_pos, tw);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    {
        KTimer t(c, kcls[1]);
        if ((e = col_pass<N, BF>(c, ZB, Vv, Vv + 4 * V, a.sa_k, a.sqrt_coupling, 0, a.nbatch, a.ns, 0, 0)) != hipSuccess)
            return e;
    }
    {
        KTimer t(c, kcls[3]);
        hipLaunchKernelGGL((k_row_update<N, BF, C>), dim3(N, 1, a.nbatch), dim3(RowE<N>::NT), 0, c->stream, U, ZA, ZB, V,
                           a.sqrt_step, a.reunit, a.whole != nullptr, tw, next_noise, Xi, a.ns, a.sa_pos);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    return hipSuccess;
}

// instantiated once per size and type (jw_step_n.hip)
template <int N, typename C>
hipError_t step_fused_layout(jw_ctx* c, C* U, C* Xi, C* Vv, C* ZA, C* ZB, const StepArgs& a,
                                    const int* kcls) {
    switch (c->layout) {
        case 0:
            if constexpr (sizeof(C) == sizeof(float2))
                if (c->fft_mfma) return step_fused_n<N, 5>(c, U, Xi, Vv, ZA, ZB, a, kcls);
            return step_fused_n<N, 0>(c, U, Xi, Vv, ZA, ZB, a, kcls);
        case 1: return step_fused_n<N, 1>(c, U, Xi, Vv, ZA, ZB, a, kcls);
        case 2: return step_fused_n<N, 2>(c, U, Xi, Vv, ZA, ZB, a, kcls);
        case 4: return step_fused_n<N, 4>(c, U, Xi, Vv, ZA, ZB, a, kcls);
        case 8: return step_fused_n<N, 8>(c, U, Xi, Vv, ZA, ZB, a, kcls);
        case 16: return step_fused_n<N, 16>(c, U, Xi, Vv, ZA, ZB, a, kcls);
        default: return hipErrorInvalidValue;
    }
}

#define JW_FUSED_SIZES(M, C) M(64, C) M(128, C) M(256, C) M(512, C) M(1024, C) M(2048, C)
#define JW_FUSED_EXTERN(n, C) \
    extern template hipError_t step_fused_layout<n, C>(jw_ctx*, C*, C*, C*, C*, C*, const StepArgs&, const int*);
#ifndef JW_STEP_N
JW_FUSED_SIZES(JW_FUSED_EXTERN, cplx)
JW_FUSED_SIZES(JW_FUSED_EXTERN, cplxf)
#endif

template <typename C>
static hipError_t step_fused_t(jw_ctx* c, C* U, C* Xi, C* Vv, C* ZA, C* ZB, const StepArgs& a) {
    static const int kcls[4] = {K_ROW_NOISE, K_COL_KMULT, K_ROW_UXIU, K_ROW_UPDATE};
#define JW_FUSED_CASE(n) \
    case n: return step_fused_layout<n>(c, U, Xi, Vv, ZA, ZB, a, kcls);
    switch (c->N) {
        JW_FUSED_CASE(64)
        JW_FUSED_CASE(128)
        JW_FUSED_CASE(256)
        JW_FUSED_CASE(512)
        JW_FUSED_CASE(1024)
        JW_FUSED_CASE(2048)
        default: return hipErrorInvalidValue;
    }
#undef JW_FUSED_CASE
}

}  // namespace jw
