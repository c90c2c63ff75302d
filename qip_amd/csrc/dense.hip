// dense.hip -- dense operators on 4..12 target qubits, and any kronselect_dot descriptor component
// (qip/ext/kronprod.pyx:41-235) that no specialised sweep covers.
//
// Terms: a dense operator U (D x D, D = 2^K, row-major, first target = MSB of the row index) acts
// on the state's "bases": a base is a state index with every target bit 0 and every control bit 1;
// the D amplitudes base + off[j] form one closed group, and out[base + off[i]] =
// sum_j U[i][j] * in[base + off[j]]. That is the matrix product Y = U X with X[j][b] the amplitudes
// of base b. FP64 arithmetic for both state precisions, rounded once on store.
//
//   k_dense_mfma<R, K>   K = 4..6, in place. Each wave forms Y = U X for 1024 amplitudes at a time with
//                        three real products on FP64 MFMA (v_mfma_f64_16x16x4f64), U's fragments in
//                        LDS. It holds every amplitude of its bases before any is written, so in place
//                        is safe. Small states take k_dense_split, a tile by four waves.
//   k_dense_low<R>       the same on the four lowest state bits, a tile loaded and stored in address order.
//   k_dense_wide<R, K>   K = 7 and 8 on states of enough tiles, in place: a workgroup holds all rows of its bases
//                        in 128 KB of LDS and forms Y on FP64 MFMA, U's fragments from the caches.
//   k_dense_gemm<R>      other K = 7..12, out of place: a 64 x 64 output tile per workgroup over 16-column
//                        steps of j through LDS, into a compact [D][nbase] buffer; k_dense_scatter
//                        writes it back to the bases' positions.
//   k_kron_general<R>    the reference's own formula, out of place: for every output row r, the sum
//                        over the 2^u columns c that agree with r outside the union of the groups'
//                        qubits, in increasing order, of prod_g entry_g(r|_g, c|_g) * in[c] (the
//                        product stops at a zero factor), with entry_g following C_MAT levels and a
//                        NUMPY or SWAP_MAT inner matrix (calc_mat_entry, kronprod.pyx:203-235).
#include "engine.h"

#include <algorithm>
#include <complex>
#include <cstring>
#include <vector>

using namespace qipgpu;

namespace {

template <typename R>
__device__ __forceinline__ cx<double> to_d(cx<R> v) {
    cx<double> o;
    o.re = (double)v.re;
    o.im = (double)v.im;
    return o;
}

template <typename R>
__device__ __forceinline__ cx<R> from_d(cx<double> v) {
    cx<R> o;
    o.re = (R)v.re;
    o.im = (R)v.im;
    return o;
}

__device__ __forceinline__ void mac(cx<double> &acc, const cx<double> a, const cx<double> b) {
    acc.re = fma(a.re, b.re, acc.re);
    acc.re = fma(-a.im, b.im, acc.re);
    acc.im = fma(a.re, b.im, acc.im);
    acc.im = fma(a.im, b.re, acc.im);
}

__device__ __forceinline__ uint64_t base_of(uint64_t g, const PosList &pl, uint64_t ctrl_mask) {
    return insert_zeros(g, pl) | ctrl_mask;
}

// ---- K = 4..6: tiles in place on FP64 MFMA -------------------------------------------------------
//
// Y = U X with U = A + i Bm and X = P + i Q takes three real D x D products (the 3M method, Higham,
// "Stability of a method for multiplying complex matrices with three real matrix multiplications",
// SIAM J. Matrix Anal. Appl. 13 (1992)): T1 = A P, T2 = Bm Q, T3 = (A + Bm)(P + Q), then
// Re Y = T1 - T2 and Im Y = T3 - T1 - T2. That is 6 D^2 real FMAs per base instead of the 8 of the
// real 2D x 2D form. Re Y rounds as the usual form does; the rounding error of Im Y is bounded in
// terms of (|A| + |Bm|)(|P| + |Q|) instead of |A||Q| + |Bm||P|, at most a small constant factor more
// in FP64 (the paper's bound).
// v_mfma_f64_16x16x4f64 computes D[16 x 16] += A[16 x 4] B[4 x 16]; lane l holds A[l % 16][l / 16]
// and B[l / 16][l % 16], and D[4 i + l / 16][l % 16] for its items i = 0..3.
//
// A wave works by itself on tiles of 1024 amplitudes: all D rows of 16 CB bases, 16 CB D = 1024. The rows
// are numbered with their bits in state-bit order, so that item i of output row block rb (row 16 rb + 4 i
// + l / 16) is the row the lane loaded for k-step 4 rb + i: amplitudes go from memory to the lanes
// that multiply them and back from the same addresses, with no LDS in between. Sixteen lanes run along
// the bases and the other four ways along the two lowest targets, so a load instruction reads runs of
// 16 bases when the targets are high bits and of the four rows (64 B of complex128) when they are low.
// U's fragments (64 KB at K = 6) are in LDS, where all waves read them; nothing else is, so the
// tile loop has no barrier: while one wave of a SIMD loads or stores, the other's MFMAs run, and the
// next tile's loads are in flight during this one's.
// Bound: HBM, and at K = 6 on complex64 states the MFMAs (1.41 ms on 2^28 amplitudes at the 73 TFLOP/s
// that a large FP64 product reaches). Per call on 2^28 amplitudes, targets low / high / scattered,
// with the tile in LDS (four barriers a tile) before, and now; a copy takes 1.63 (complex128) and
// 0.81 ms (complex64):
//   complex128 K = 4 1.76 / 1.87 / 1.69 -> 1.90 / 1.66 / 1.61 ms; K = 5 1.94 / 1.76 / 1.66 -> 1.88 / 1.67 /
//   1.72; K = 6 2.94 / 2.46 / 2.40 -> 1.74 / 1.79 / 1.82
//   complex64 K = 4 1.39 / 1.04 / 1.04 -> 1.11 / 0.84 / 0.86; K = 5 1.95 / 1.51 / 1.51 -> 1.10 / 0.95 / 0.90;
//   K = 6 2.95 / 2.39 / 2.39 -> 1.62 / 1.61 / 1.60
// (K = 4 on the four lowest bits is k_dense_low's.)
// Workgroups take tiles a grid apart: 1.66 against 1.74 ms (K = 4, high targets) with contiguous ranges.
template <int K>
struct MfmaShape {
    static constexpr int D = 1 << K;
    static constexpr int KS = D / 4;             // 4-row k-steps
    static constexpr int RB = D / 16;            // 16-row output blocks
    static constexpr int CB = 64 / D;            // 16-base column blocks of a wave's tile
    static constexpr int NR = K == 4 ? 1 : 2;    // output blocks formed at a time: NR rows of NC columns
    static constexpr int NC = K == 4 ? 2 : 1;
    static constexpr int BASES = 16 * CB;
    static_assert(K >= 4 && K <= 6, "MFMA tiles for 4 to 6 targets");
};

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

constexpr int kTileThreads = 256;
constexpr int kTileWaves = kTileThreads / 64;

template <typename R, int K>
struct DenseTileArgs {
    cx<R> *amps;
    uint64_t nbase;
    uint64_t ntiles;                        // tiles of 16 CB bases
    PosList pl;                             // target and control bits
    uint64_t row_k[4];                      // offset of the two lowest targets' values, and the controls
    uint64_t row_s[MfmaShape<K>::KS];       // offset of the other targets' values
};

template <typename R, int K>
__global__ __launch_bounds__(kTileThreads, 2) void k_dense_mfma(const DenseTileArgs<R, K> a,
                                                                const f64x2 *__restrict__ frag) {
    using M = MfmaShape<K>;
    constexpr int NF = M::KS * M::RB * 64;
    __shared__ f64x2 sU[NF];                // [k-step][row block][lane]: Re and Im of U
    for (int e = threadIdx.x; e < NF; e += kTileThreads) sU[e] = frag[e];
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // this lane's part of its bases' positions (every tile is full: there are more than kSplitTiles)
    uint64_t at[M::CB];
    const int kap = lane >> 4;
    const uint64_t row = kap & 2 ? (kap & 1 ? a.row_k[3] : a.row_k[2]) : (kap & 1 ? a.row_k[1] : a.row_k[0]);
#pragma unroll
    for (int c = 0; c < M::CB; ++c) at[c] = insert_zeros((uint64_t)(16 * c + (lane & 15)), a.pl) + row;
    const uint64_t step = (uint64_t)gridDim.x * kTileWaves, end = a.ntiles;
    uint64_t t = (uint64_t)blockIdx.x * kTileWaves + wave;
    if (t >= end) return;
    auto tile_at = [&](uint64_t tile) { return a.amps + insert_zeros(tile * M::BASES, a.pl); };
    auto load = [&](cx<R> (&x)[16], uint64_t tile) {
        const cx<R> *p = tile_at(tile);
        // a base's rows one after the other: low targets' rows share cache lines
#pragma unroll
        for (int c = 0; c < M::CB; ++c)
#pragma unroll
            for (int s = 0; s < M::KS; ++s) x[s * M::CB + c] = p[at[c] + a.row_s[s]];
    };
    auto process = [&](const cx<R> (&x)[16], uint64_t tile) {
        cx<R> *p = tile_at(tile);
#pragma unroll
        for (int r0 = 0; r0 < M::RB; r0 += M::NR)
#pragma unroll
            for (int c0 = 0; c0 < M::CB; c0 += M::NC) {
                // U's fragments are read again for every tile: kept in registers over the loop they would spill
                asm volatile("" ::: "memory");
                f64x4 acc[3][M::NR][M::NC];
#pragma unroll
                for (int m = 0; m < 3; ++m)
#pragma unroll
                    for (int r = 0; r < M::NR; ++r)
#pragma unroll
                        for (int c = 0; c < M::NC; ++c) acc[m][r][c] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int s = 0; s < M::KS; ++s) {
                    f64x2 u[M::NR];
#pragma unroll
                    for (int r = 0; r < M::NR; ++r) u[r] = sU[(s * M::RB + r0 + r) * 64 + lane];
#pragma unroll
                    for (int c = 0; c < M::NC; ++c) {
                        const cx<double> v = to_d(x[s * M::CB + c0 + c]);
                        const double sum = v.re + v.im;
#pragma unroll
                        for (int r = 0; r < M::NR; ++r) {
                            acc[0][r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(u[r][0], v.re, acc[0][r][c], 0, 0, 0);
                            acc[1][r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(u[r][1], v.im, acc[1][r][c], 0, 0, 0);
                            acc[2][r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(u[r][0] + u[r][1], sum, acc[2][r][c], 0, 0, 0);
                        }
                    }
                }
#pragma unroll
                for (int r = 0; r < M::NR; ++r)
#pragma unroll
                    for (int c = 0; c < M::NC; ++c)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const double t1 = acc[0][r][c][i], t2 = acc[1][r][c][i];
                            cx<double> y;
                            y.re = t1 - t2;
                            y.im = acc[2][r][c][i] - t1 - t2;
                            __builtin_amdgcn_sched_barrier(0);   // kept apart: K = 6, complex64, 1.620 ms scheduled freely, 1.602 so
                            p[at[c0 + c] + a.row_s[4 * (r0 + r) + i]] = from_d<R>(y);
                        }
            }
    };
    // two register buffers alternate (the last prefetch re-reads an in-range tile and is not used)
    cx<R> xa[16], xb[16];
    load(xa, t);
    for (;;) {
        const uint64_t t1 = t + step, t2 = t1 + step;
        load(xb, min(t1, end - 1));
        process(xa, t);
        if (t1 >= end) return;
        load(xa, min(t2, end - 1));
        process(xb, t1);
        if (t2 >= end) return;
        t = t2;
    }
}

// Four targets on the four lowest state bits: a base is 16 amplitudes in a row, and k_dense_mfma's lanes, 16 along the
// bases, would touch 16 B of a line each. Here a wave loads and stores its tile in address order and turns it
// through LDS of its own (slots of 16 amplitudes padded by one), so there is still no barrier in the loop.
// Bound: HBM. A call, by k_dense_mfma and here: 2^28 amplitudes complex128 1908 -> 1690 us, complex64 1110 -> 863; 2^26 481
// -> 430 and 286 -> 218; 2^24 77 -> 78 and 66 -> 52; 2^22 30 -> 31 and 27 -> 24. One bit higher k_dense_mfma takes 1690
// and 836 at 2^28; on 5 of the lowest bits its runs are 128 B and more in complex128 (1877).
template <typename R>
__global__ __launch_bounds__(kTileThreads, 2) void k_dense_low(const DenseTileArgs<R, 4> a, const f64x2 *__restrict__ frag) {
    using M = MfmaShape<4>;
    // an amplitude as a vector: structs copied from memory to LDS went through scratch memory
    typedef R Amp __attribute__((ext_vector_type(2)));
    __shared__ f64x2 sU[M::KS * 64];
    __shared__ Amp turn[kTileWaves][1024 + 64];
    for (int e = threadIdx.x; e < M::KS * 64; e += kTileThreads) sU[e] = frag[e];
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // amplitude 64 j + lane of the tile is row lane % 16 of base 4 j + lane / 16
    Amp *const line = &turn[wave][17 * (lane >> 4) + (lane & 15)];             // + 68 j
    Amp *const cell = &turn[wave][17 * (lane & 15) + (lane >> 4)];             // base 16 c + lane % 16, row 4 s + lane / 16: + 272 c + 4 s
    const uint64_t at = insert_zeros((uint64_t)(lane >> 4), a.pl) + a.row_k[0] + (lane & 15);
    uint64_t base[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) base[j] = insert_zeros(4ull * j, a.pl);
    f64x2 u[M::KS];
#pragma unroll
    for (int s = 0; s < M::KS; ++s) u[s] = sU[s * 64 + lane];
    const uint64_t step = (uint64_t)gridDim.x * kTileWaves, end = a.ntiles;
    uint64_t t = (uint64_t)blockIdx.x * kTileWaves + wave;
    if (t >= end) return;
    // the wave's LDS accesses are carried out in order: only the compiler has to keep theirs
    auto in_order = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    Amp *const amps = reinterpret_cast<Amp *>(a.amps) + at;
    auto tile_at = [&](uint64_t tile) { return amps + insert_zeros(tile * M::BASES, a.pl); };
    auto load = [&](Amp (&x)[16], uint64_t tile) {
        const Amp *p = tile_at(tile);
#pragma unroll
        for (int j = 0; j < 16; ++j) x[j] = p[base[j]];
    };
    auto process = [&](const Amp (&x)[16], uint64_t tile) {
        Amp *p = tile_at(tile);
#pragma unroll
        for (int j = 0; j < 16; ++j) line[68 * j] = x[j];
        in_order();
#pragma unroll
        for (int c = 0; c < M::CB; ++c) {
            f64x4 acc[3];
#pragma unroll
            for (int m = 0; m < 3; ++m) acc[m] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int s = 0; s < M::KS; ++s) {
                const Amp v = cell[272 * c + 4 * s];
                const double re = v.x, im = v.y;
                acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(u[s][0], re, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(u[s][1], im, acc[1], 0, 0, 0);
                acc[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(u[s][0] + u[s][1], re + im, acc[2], 0, 0, 0);
            }
            // row 4 i + lane / 16: the cells this lane read
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                cell[272 * c + 4 * i] = Amp{(R)(acc[0][i] - acc[1][i]), (R)(acc[2][i] - acc[0][i] - acc[1][i])};
            }
        }
        in_order();
#pragma unroll
        for (int j = 0; j < 16; ++j) p[base[j]] = line[68 * j];
        in_order();
    };
    Amp xa[16], xb[16];
    load(xa, t);
    for (;;) {
        const uint64_t t1 = t + step, t2 = t1 + step;
        load(xb, min(t1, end - 1));
        process(xa, t);
        if (t1 >= end) return;
        load(xa, min(t2, end - 1));
        process(xb, t1);
        if (t2 >= end) return;
        t = t2;
    }
}

// The same tile by the four waves of a workgroup, one 16 x 16 block of outputs each, for states with at most
// kSplitTiles tiles: a wave that works a tile alone has a chain of up to 192 MFMAs (5 us), and fewer
// tiles than the GPU has places for waves leave most of it idle. A wave's fragments come straight from
// memory, all its loads at once; a barrier keeps the columns' loads ahead of the stores. 6 targets on
// 2^17 amplitudes: 24.4 us a call with the kernel above, 20.2 so (most of both is staging U); at 2^20 they meet.
constexpr uint64_t kSplitTiles = 512;

template <typename R, int K>
__global__ __launch_bounds__(kTileThreads) void k_dense_split(const DenseTileArgs<R, K> a,
                                                              const f64x2 *__restrict__ frag) {
    using M = MfmaShape<K>;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rb = wave % M::RB, col = wave / M::RB;
    const int kap = lane >> 4;
    f64x2 u[M::KS];
#pragma unroll
    for (int s = 0; s < M::KS; ++s) u[s] = frag[(s * M::RB + rb) * 64 + lane];
    const uint64_t g = (uint64_t)blockIdx.x * M::BASES + 16 * col + (lane & 15);
    cx<R> *p = a.amps + insert_zeros(g & (a.nbase - 1), a.pl) +
               (kap & 2 ? (kap & 1 ? a.row_k[3] : a.row_k[2]) : (kap & 1 ? a.row_k[1] : a.row_k[0]));
    cx<R> x[M::KS];
#pragma unroll
    for (int s = 0; s < M::KS; ++s) x[s] = p[a.row_s[s]];
    f64x4 acc[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) acc[m] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < M::KS; ++s) {
        const cx<double> v = to_d(x[s]);
        acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(u[s][0], v.re, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(u[s][1], v.im, acc[1], 0, 0, 0);
        acc[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(u[s][0] + u[s][1], v.re + v.im, acc[2], 0, 0, 0);
    }
    __syncthreads();   // every wave of the tile holds its columns' amplitudes
    if (g >= a.nbase) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        cx<double> y;
        y.re = acc[0][i] - acc[1][i];
        y.im = acc[2][i] - acc[0][i] - acc[1][i];
        // row 16 rb + 4 i + kap: k-step 4 rb + i
        uint64_t off = 0;
#pragma unroll
        for (int r = 0; r < M::RB; ++r) off = rb == r ? a.row_s[4 * r + i] : off;
        p[off] = from_d<R>(y);
    }
}

// ---- K = 7, 8: tiles in place in LDS --------------------------------------------------------------
//
// A tile is all D rows of 8192 / D bases, 128 KB of LDS as FP64 pairs, for one workgroup of 8 waves a CU. It
// is read once: each wave forms D / 8 output rows for every base from it, with the rows numbered and the
// fragments laid out as in k_dense_mfma, and writes them over the amplitudes read. The next tile is on
// its way to registers meanwhile. A k-step takes 1 KB of U a row block from the L2 and CB KB of X from LDS
// for 12 MFMAs of 64 cycles, so the matrix cores are the bound: 0.70 ms for 7 targets on 2^26 amplitudes at
// the 73 TFLOP/s that a large FP64 product reaches. The GEMM below gathers its rows 16 B at a time when the
// targets are low bits and writes its results back from a temporary as large as the state. A call on 2^26
// amplitudes, targets low / high / scattered, by the GEMM and here:
//   complex128 K = 7 4.19 / 1.51 / 2.05 -> 1.07 / 1.06 / 1.05 ms; K = 8 4.62 / 2.42 / 2.39 -> 1.81 / 1.80 / 1.78
//   complex64 K = 7 4.07 / 1.33 / 1.45 -> 0.99 / 0.98 / 0.95 ms; K = 8 3.74 / 2.21 / 2.43 -> 1.73 / 1.74 / 1.71
template <int K>
struct WideShape {
    static constexpr int D = 1 << K;
    static constexpr int KS = D / 4;
    static constexpr int RB = D / 16;
    static constexpr int BASES = 8192 / D;
    static constexpr int CB = BASES / 16;
    static constexpr int WAVES = 8;
    static constexpr int NR = RB / WAVES;        // row blocks of a wave
    static_assert(K == 7 || K == 8, "tiles of 7 and 8 targets");
};

template <typename R, int K>
struct DenseWideArgs {
    cx<R> *amps;
    uint64_t nbase, ntiles;
    PosList pl;                             // target and control bits
    uint64_t row_k[4];                      // offset of the two lowest targets' values, and the controls
    uint64_t row_s[WideShape<K>::KS];       // offset of the other targets' values
};

template <typename R, int K>
__global__ __launch_bounds__(512) void k_dense_wide(const DenseWideArgs<R, K> a, const f64x2 *__restrict__ frag) {
    using M = WideShape<K>;
    __shared__ f64x2 sX[M::D * M::BASES];   // [row][base]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kap = lane >> 4, rho = lane & 15;
    const uint64_t row = kap & 2 ? (kap & 1 ? a.row_k[3] : a.row_k[2]) : (kap & 1 ? a.row_k[1] : a.row_k[0]);
    auto base_at = [&](int c) { return insert_zeros((uint64_t)(16 * c + rho), a.pl) + row; };
    // this wave loads 16 k-steps' rows of one column block
    constexpr int kPerBlock = M::WAVES / M::CB;
    const int lc = wave / kPerBlock, ls = wave % kPerBlock * 16;
    const uint64_t load_at = base_at(lc);
    auto tile_at = [&](uint64_t tile) { return a.amps + insert_zeros(tile * M::BASES, a.pl); };
    cx<R> x[16];
    uint64_t tile = blockIdx.x;
    auto load = [&](uint64_t t) {
        const cx<R> *p = tile_at(t) + load_at;
#pragma unroll
        for (int e = 0; e < 16; ++e) x[e] = p[a.row_s[ls + e]];
    };
    const f64x2 *f = frag + (size_t)wave * M::NR * 64 + lane;
    load(tile);
    for (;;) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const cx<double> v = to_d(x[e]);
            sX[(4 * (ls + e) + kap) * M::BASES + 16 * lc + rho] = f64x2{v.re, v.im};
        }
        const uint64_t next = tile + gridDim.x;
        __syncthreads();
        load(next < a.ntiles ? next : tile);
        f64x4 acc[3][M::NR][M::CB];
#pragma unroll
        for (int m = 0; m < 3; ++m)
#pragma unroll
            for (int r = 0; r < M::NR; ++r)
#pragma unroll
                for (int c = 0; c < M::CB; ++c) acc[m][r][c] = f64x4{0.0, 0.0, 0.0, 0.0};
        // U's fragments four k-steps ahead (1.06 ms; two: 1.09). The loop is not unrolled further: 252 B of spills
        // at K = 7.
        constexpr int kAhead = 4;
        f64x2 u[kAhead][M::NR];
#pragma unroll
        for (int s = 0; s < kAhead; ++s)
#pragma unroll
            for (int r = 0; r < M::NR; ++r) u[s][r] = f[(s * M::RB + r) * 64];
#pragma unroll 1
        for (int s0 = 0; s0 < M::KS; s0 += kAhead) {
            const int sn = s0 + kAhead < M::KS ? s0 + kAhead : 0;
#pragma unroll
            for (int s = 0; s < kAhead; ++s) {
                f64x2 now[M::NR];
#pragma unroll
                for (int r = 0; r < M::NR; ++r) {
                    now[r] = u[s][r];
                    u[s][r] = f[((sn + s) * M::RB + r) * 64];
                }
#pragma unroll
                for (int c = 0; c < M::CB; ++c) {
                    const f64x2 v = sX[(4 * (s0 + s) + kap) * M::BASES + 16 * c + rho];
                    const double sum = v[0] + v[1];
#pragma unroll
                    for (int r = 0; r < M::NR; ++r) {
                        acc[0][r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(now[r][0], v[0], acc[0][r][c], 0, 0, 0);
                        acc[1][r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(now[r][1], v[1], acc[1][r][c], 0, 0, 0);
                        acc[2][r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(now[r][0] + now[r][1], sum, acc[2][r][c], 0, 0, 0);
                    }
                }
            }
        }
        cx<R> *p = tile_at(tile);
#pragma unroll
        for (int c = 0; c < M::CB; ++c) {
            cx<R> *pc = p + base_at(c);
#pragma unroll
            for (int r = 0; r < M::NR; ++r)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const double t1 = acc[0][r][c][i], t2 = acc[1][r][c][i];
                    cx<double> y;
                    y.re = t1 - t2;
                    y.im = acc[2][r][c][i] - t1 - t2;
                    pc[a.row_s[4 * (wave * M::NR + r) + i]] = from_d<R>(y);
                }
        }
        if (next >= a.ntiles) return;      // the same for every wave of the workgroup
        tile = next;
        __syncthreads();                   // every wave is done with this tile's rows
    }
}

// ---- K = 7..12: tiled GEMM out of place ---------------------------------------------------------
//
// A workgroup computes a 64-row x 64-base block of Y = U X into a compact [D][nbase] buffer, over
// the D input rows in steps of 16 through LDS (Re / Im planes of the U block and of the X block,
// padded by one slot per row). On FP64 MFMA with the same three real products per complex one as
// the tiles above: wave w owns output rows 16 w .. 16 w + 15 and all four 16-base column blocks,
// 12 accumulators; per step it reads its A fragments (Re U, Im U; Re U + Im U formed in registers)
// and the B fragments of X from LDS. Bases past nbase read the last base and are not stored.

constexpr int kGemmTile = 64;
constexpr int kGemmStep = 16;

template <typename R>
__global__ __launch_bounds__(256, 2) void k_dense_gemm(const cx<R> *__restrict__ amps, cx<R> *__restrict__ out,
                                                       uint64_t nbase, int D, uint64_t ctrl_mask, PosList pl,
                                                       const uint64_t *__restrict__ off,
                                                       const cx<double> *__restrict__ U) {
    constexpr int US = kGemmStep + 1;          // padded U row (doubles)
    constexpr int XS = kGemmTile + 1;          // padded X row
    __shared__ double sU[2][kGemmTile * US];
    __shared__ double sX[2][kGemmStep * XS];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int rho = lane & 15, kap = lane >> 4;
    const uint64_t b0 = (uint64_t)blockIdx.x * kGemmTile;   // first base of the block
    const int i0 = blockIdx.y * kGemmTile;                    // first output row of the block
    // loader roles: X row jj0 + 4 s of base b_ld; U row u_row, columns u_col + 4 s
    const int b_ld = tid % kGemmTile;
    const int jj0 = tid / kGemmTile;
    const uint64_t gb = b0 + b_ld;
    const uint64_t base = base_of(gb < nbase ? gb : nbase - 1, pl, ctrl_mask);
    const int u_row = tid / 4, u_col = tid % 4;
    f64x4 acc[3][4];
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[m][c] = f64x4{0.0, 0.0, 0.0, 0.0};
    for (int jc = 0; jc < D; jc += kGemmStep) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int jj = jj0 + 4 * s;
            const cx<double> v = to_d(amps[base + off[jc + jj]]);
            sX[0][jj * XS + b_ld] = v.re;
            sX[1][jj * XS + b_ld] = v.im;
            const cx<double> u = U[(size_t)(i0 + u_row) * D + jc + u_col + 4 * s];
            sU[0][u_row * US + u_col + 4 * s] = u.re;
            sU[1][u_row * US + u_col + 4 * s] = u.im;
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < kGemmStep / 4; ++s) {
            const int ua = (16 * wave + rho) * US + 4 * s + kap;
            const double a0 = sU[0][ua], a1 = sU[1][ua];
            const double a2 = a0 + a1;
            const int xa = (4 * s + kap) * XS + rho;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const double p = sX[0][xa + 16 * c], q = sX[1][xa + 16 * c];
                acc[0][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, p, acc[0][c], 0, 0, 0);
                acc[1][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, q, acc[1][c], 0, 0, 0);
                acc[2][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a2, p + q, acc[2][c], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    // item i of column block c: output row i0 + 16 wave + 4 i + kap, base b0 + 16 c + rho
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const uint64_t b = b0 + 16 * c + rho;
        if (b < nbase) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const double t1 = acc[0][c][i], t2 = acc[1][c][i];
                cx<double> y;
                y.re = t1 - t2;
                y.im = acc[2][c][i] - t1 - t2;
                out[(size_t)(i0 + 16 * wave + 4 * i + kap) * nbase + b] = from_d<R>(y);
            }
        }
    }
}

// out[i][b] (compact) -> amps[base(b) + off[i]]
template <typename R>
__global__ __launch_bounds__(256) void k_dense_scatter(cx<R> *amps, const cx<R> *__restrict__ out, uint64_t nbase,
                                                       int D, uint64_t ctrl_mask, PosList pl,
                                                       const uint64_t *__restrict__ off) {
    const uint64_t total = nbase * (uint64_t)D;
    for (uint64_t e = (uint64_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (uint64_t)gridDim.x * 256) {
        const uint64_t i = e / nbase, b = e % nbase;
        amps[base_of(b, pl, ctrl_mask) + off[i]] = out[e];
    }
}

// ---- any descriptor component: the reference's column sum ---------------------------------------

struct KronGroupDev {
    int32_t len;        // indices in the group
    int32_t levels;     // C_MAT levels: the first `levels` indices are controls
    int32_t kind;       // inner matrix: 1 NUMPY (dense), 3 SWAP_MAT
    int32_t param;      // SWAP_MAT block width
    int32_t pos_at;     // first entry in the positions array (state bits, first = MSB of the index)
    int32_t pad_;
    uint64_t mat_at;    // first complex entry of a NUMPY inner matrix
};

struct KronArgs {
    int32_t n_groups;
    int32_t u;                  // union size
    uint8_t upos[QIPGPU_MAX_QUBITS];   // union state bits, enumeration bit u-1-j -> upos[j]
    uint64_t umask;
};

__device__ __forceinline__ cx<double> group_entry(const KronGroupDev &g, const int32_t *__restrict__ pos,
                                                 const cx<double> *__restrict__ mats, uint64_t row, uint64_t col) {
    uint64_t ri = 0, ci = 0;
    for (int m = 0; m < g.len; ++m) {
        const int p = pos[g.pos_at + m];
        ri = (ri << 1) | ((row >> p) & 1ull);
        ci = (ci << 1) | ((col >> p) & 1ull);
    }
    cx<double> one, zero;
    one.re = 1.0;
    one.im = 0.0;
    zero.re = zero.im = 0.0;
    int len = g.len;
    for (int lv = 0; lv < g.levels; ++lv) {
        const uint64_t top = 1ull << (len - 1);
        const bool rb = (ri & top) != 0, cb = (ci & top) != 0;
        if (rb != cb) return zero;
        ri &= top - 1;
        ci &= top - 1;
        --len;
        if (!rb) return ri == ci ? one : zero;
    }
    if (g.kind == 3) {
        const uint64_t half = 1ull << g.param;
        const uint64_t partner = (ri % half) * half + ri / half;
        return partner == ci ? one : zero;
    }
    return mats[g.mat_at + (ri << len) + ci];
}

template <typename R>
__global__ __launch_bounds__(256) void k_kron_general(const cx<R> *__restrict__ in, cx<R> *__restrict__ out,
                                                      uint64_t len, KronArgs a,
                                                      const KronGroupDev *__restrict__ groups,
                                                      const int32_t *__restrict__ pos,
                                                      const cx<double> *__restrict__ mats) {
    const uint64_t cols = 1ull << a.u;
    for (uint64_t row = (uint64_t)blockIdx.x * 256 + threadIdx.x; row < len; row += (uint64_t)gridDim.x * 256) {
        cx<double> s;
        s.re = s.im = 0.0;
        const uint64_t keep = row & ~a.umask;
        for (uint64_t e = 0; e < cols; ++e) {
            uint64_t col = keep;
            for (int j = 0; j < a.u; ++j) col |= ((e >> (a.u - 1 - j)) & 1ull) << a.upos[j];
            cx<double> p;
            p.re = 1.0;
            p.im = 0.0;
            for (int gi = 0; gi < a.n_groups; ++gi) {
                const cx<double> m = group_entry(groups[gi], pos, mats, row, col);
                cx<double> np;
                np.re = p.re * m.re - p.im * m.im;
                np.im = p.re * m.im + p.im * m.re;
                p = np;
                if (p.re == 0.0 && p.im == 0.0) break;
            }
            const cx<double> v = to_d(in[col]);
            s.re += p.re * v.re - p.im * v.im;
            s.im += p.re * v.im + p.im * v.re;
        }
        out[row] = from_d<R>(s);
    }
}

// Diagonal on up to QIPGPU_MAX_DENSE targets, entries in device memory; one item per amplitude of the
// controlled subspace.
template <typename R>
__global__ __launch_bounds__(256) void k_diag_table(cx<R> *amps, uint64_t count, uint64_t ctrl_mask, PosList pl,
                                                    int K, const uint8_t *__restrict__ tpos_g,
                                                    const cx<double> *__restrict__ d) {
    __shared__ uint8_t tpos[QIPGPU_MAX_DENSE];
    if (threadIdx.x < K) tpos[threadIdx.x] = tpos_g[threadIdx.x];
    __syncthreads();
    for (uint64_t g = (uint64_t)blockIdx.x * 256 + threadIdx.x; g < count; g += (uint64_t)gridDim.x * 256) {
        const uint64_t i = base_of(g, pl, ctrl_mask);
        uint32_t j = 0;
        for (int b = 0; b < K; ++b) j = (j << 1) | (uint32_t)((i >> tpos[b]) & 1ull);
        const cx<double> v = to_d(amps[i]), f = d[j];
        cx<double> o;
        o.re = f.re * v.re - f.im * v.im;
        o.im = f.re * v.im + f.im * v.re;
        amps[i] = from_d<R>(o);
    }
}

template <typename R>
__global__ __launch_bounds__(256) void k_copy_amps(cx<R> *dst, const cx<R> *__restrict__ src, uint64_t len) {
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < len; i += (uint64_t)gridDim.x * 256) dst[i] = src[i];
}

// ---- host side -----------------------------------------------------------------------------------

using StreamBuffer = TempBuffer;

std::vector<uint64_t> offsets(const std::vector<int> &tbits) {
    const int K = (int)tbits.size();
    std::vector<uint64_t> off((size_t)1 << K);
    for (size_t j = 0; j < off.size(); ++j) {
        uint64_t o = 0;
        for (int t = 0; t < K; ++t)
            if ((j >> (K - 1 - t)) & 1) o |= 1ull << tbits[t];
        off[j] = o;
    }
    return off;
}

PosList poslist(std::vector<int> pos) {
    std::sort(pos.begin(), pos.end());
    PosList pl;
    pl.count = (int32_t)pos.size();
    for (size_t i = 0; i < pos.size(); ++i) pl.set((int)i, (uint32_t)pos[i]);
    return pl;
}

// The arguments (DenseTileArgs, DenseWideArgs) of a kernel that numbers the rows in state-bit order: bit b of a
// row is the b-th lowest target bit. caller[j]: row j's place in the caller's index.
template <typename M, typename A>
void tile_arguments(A &a, int (&caller)[M::D], qipgpu_state *s, const std::vector<int> &tbits, uint64_t ctrl_mask,
                    const std::vector<int> &allpos) {
    const int K = (int)tbits.size();
    std::vector<int> sorted(tbits);
    std::sort(sorted.begin(), sorted.end());
    for (int j = 0; j < M::D; ++j) {
        caller[j] = 0;
        for (int t = 0; t < K; ++t) {
            const int b = (int)(std::find(sorted.begin(), sorted.end(), tbits[t]) - sorted.begin());
            caller[j] |= (j >> b & 1) << (K - 1 - t);
        }
    }
    std::memset(&a, 0, sizeof(a));
    a.amps = (decltype(a.amps))s->amps;
    a.nbase = s->len >> allpos.size();
    a.ntiles = (a.nbase + M::BASES - 1) / M::BASES;
    a.pl = poslist(allpos);
    for (int j = 0; j < 4; ++j)
        a.row_k[j] = ctrl_mask + ((uint64_t)(j & 1) << sorted[0]) + ((uint64_t)(j >> 1) << sorted[1]);
    for (int j = 0; j < M::KS; ++j)
        for (int b = 2; b < K; ++b) a.row_s[j] += (uint64_t)(j >> (b - 2) & 1) << sorted[b];
}

// U's fragments for such a kernel, D x D entries: [k-step][row block][lane].
template <typename M>
void fragments(std::complex<double> *out, const int (&caller)[M::D], const std::complex<double> *U) {
    for (int st = 0; st < M::KS; ++st)
        for (int rb = 0; rb < M::RB; ++rb)
            for (int l = 0; l < 64; ++l)
                out[(size_t)(st * M::RB + rb) * 64 + l] = U[(size_t)caller[16 * rb + l % 16] * M::D + caller[4 * st + l / 16]];
}

template <typename R, int K>
int launch_tile(qipgpu_state *s, const std::vector<int> &tbits, uint64_t ctrl_mask, const std::vector<int> &allpos,
                const std::complex<double> *U) {
    DenseTileArgs<R, K> a;
    int caller[1 << K];
    tile_arguments<MfmaShape<K>>(a, caller, s, tbits, ctrl_mask, allpos);
    std::vector<std::complex<double>> frag((size_t)1 << 2 * K);
    fragments<MfmaShape<K>>(frag.data(), caller, U);
    void *d = nullptr;
    int rc = ring_upload(s, frag.data(), frag.size() * sizeof(frag[0]), &d);
    if (rc) return rc;
    if (a.ntiles <= kSplitTiles) {
        hipLaunchKernelGGL((k_dense_split<R, K>), dim3((uint32_t)a.ntiles), dim3(kTileThreads), 0, s->stream, a,
                           (const f64x2 *)d);
        QIP_LAUNCHED();
        return QIPGPU_OK;
    }
    const uint64_t grid = std::min<uint64_t>((a.ntiles + kTileWaves - 1) / kTileWaves, (uint64_t)device_cus() * 2);
    if constexpr (K == 4) {
        if (*std::max_element(tbits.begin(), tbits.end()) == 3) {      // the lowest four: figures at the kernel
            hipLaunchKernelGGL(k_dense_low<R>, dim3((uint32_t)grid), dim3(kTileThreads), 0, s->stream, a, (const f64x2 *)d);
            QIP_LAUNCHED();
            return QIPGPU_OK;
        }
    }
    hipLaunchKernelGGL((k_dense_mfma<R, K>), dim3((uint32_t)grid), dim3(kTileThreads), 0, s->stream, a,
                       (const f64x2 *)d);
    QIP_LAUNCHED();
    return QIPGPU_OK;
}

// Temporaries of wide dense operators up to this size stay with the state for the next call.
constexpr size_t kKeepGemmTmpBytes = size_t(1) << 30;

// `need` bytes of a wide dense operator into the state's operator buffer, on its queue: `fill` writes them to
// pinned memory, so the copy is asynchronous and the queue is not drained first. The pinned buffer is
// rewritten only once the previous copy out of it has run; the device buffer is rewritten in queue
// order, after the kernels that read it. (Fragments go straight to the pinned buffer: by an array of their own, 1 MiB
// of fresh pages, a waited-for call of K = 8 on 22 qubits took 290 us, 244 so; the GEMM 239.)
template <typename F>
int stage_gemm_operator(qipgpu_state *s, size_t need, F fill, void **dev) {
    if (!s->gemm_ev) QIP_HIP(hipEventCreateWithFlags(&s->gemm_ev, hipEventDisableTiming));
    else QIP_HIP(hipEventSynchronize(s->gemm_ev));
    if (s->h_gemm_op_bytes < need) {
        if (s->h_gemm_op) QIP_HIP(hipHostFree(s->h_gemm_op));
        s->h_gemm_op = nullptr;
        s->h_gemm_op_bytes = 0;
        QIP_HIP(hipHostMalloc(&s->h_gemm_op, need, hipHostMallocDefault));
        s->h_gemm_op_bytes = need;
    }
    if (s->d_gemm_op_bytes < need) {
        QIP_HIP(hipStreamSynchronize(s->stream));   // queued kernels may still read the old buffer
        if (s->d_gemm_op) QIP_HIP(hipFree(s->d_gemm_op));
        s->d_gemm_op = nullptr;
        s->d_gemm_op_bytes = 0;
        QIP_HIP(hipMalloc(&s->d_gemm_op, need));
        s->d_gemm_op_bytes = need;
    }
    fill(static_cast<char *>(s->h_gemm_op));
    QIP_HIP(hipMemcpyAsync(s->d_gemm_op, s->h_gemm_op, need, hipMemcpyHostToDevice, s->stream));
    QIP_HIP(hipEventRecord(s->gemm_ev, s->stream));
    *dev = s->d_gemm_op;
    return QIPGPU_OK;
}

// From this many tiles on k_dense_wide is used: a workgroup's waves have D / 4 k-steps of a whole tile before
// them, where the GEMM spreads a small state's rows over workgroups, and its fragments cost the host more than
// a copy of U. GEMM / k_dense_wide, complex128, targets low, us a call among others and a call waited for: K = 7
// 128 tiles (20 qubits) 63 / 62 and 77 / 82, 256 77 / 65 and 91 / 84; K = 8 256 tiles (21 qubits) 119 / 134,
// 512 187 / 160 and 239 / 244. complex64: 62 / 61 and 76 / 80, 77 / 61 and 90 / 80; 512 tiles 196 / 154 and 248 / 241.
constexpr uint64_t kWideTiles7 = 256, kWideTiles8 = 512;

template <typename R, int K>
int launch_wide(qipgpu_state *s, const std::vector<int> &tbits, uint64_t ctrl_mask, const std::vector<int> &allpos,
                const std::complex<double> *U) {
    DenseWideArgs<R, K> a;
    int caller[1 << K];
    tile_arguments<WideShape<K>>(a, caller, s, tbits, ctrl_mask, allpos);
    void *d = nullptr;
    const int rc = stage_gemm_operator(s, sizeof(std::complex<double>) << 2 * K, [&](char *to) {
        fragments<WideShape<K>>(reinterpret_cast<std::complex<double> *>(to), caller, U);
    }, &d);
    if (rc) return rc;
    const uint32_t grid = (uint32_t)std::min<uint64_t>(a.ntiles, (uint64_t)device_cus());
    hipLaunchKernelGGL((k_dense_wide<R, K>), dim3(grid), dim3(512), 0, s->stream, a, (const f64x2 *)d);
    QIP_LAUNCHED();
    return QIPGPU_OK;
}

template <typename R>
int launch_gemm(qipgpu_state *s, const std::vector<int> &tbits, uint64_t ctrl_mask, const std::vector<int> &allpos,
                const std::complex<double> *U) {
    const int K = (int)tbits.size();
    const int D = 1 << K;
    const std::vector<uint64_t> off = offsets(tbits);
    void *op = nullptr;
    const size_t ob = off.size() * sizeof(uint64_t), ub = (size_t)D * D * sizeof(cx<double>);
    int rc = stage_gemm_operator(s, ob + ub, [&](char *to) {
        std::memcpy(to, off.data(), ob);
        std::memcpy(to + ob, U, ub);
    }, &op);
    if (rc) return rc;
    const uint64_t nbase = s->len >> allpos.size();
    // the compact temporary: the state's kept one when small, else one for this call
    const size_t tb = nbase * (size_t)D * sizeof(cx<R>);
    StreamBuffer big(s->stream);
    void *tmp = nullptr;
    if (tb <= kKeepGemmTmpBytes) {
        if (s->gemm_tmp_bytes < tb) {
            QIP_HIP(hipStreamSynchronize(s->stream));   // queued kernels may still use the old one
            if (s->gemm_tmp) QIP_HIP(hipFree(s->gemm_tmp));
            s->gemm_tmp = nullptr;
            s->gemm_tmp_bytes = 0;
            QIP_HIP(hipMalloc(&s->gemm_tmp, tb));
            s->gemm_tmp_bytes = tb;
        }
        tmp = s->gemm_tmp;
    } else {
        QIP_HIP(big.alloc(tb));
        tmp = big.p;
    }
    const PosList pl = poslist(allpos);
    const uint64_t *doff = (const uint64_t *)op;
    const cx<double> *dU = (const cx<double> *)((char *)op + off.size() * sizeof(uint64_t));
    const dim3 grid((uint32_t)((nbase + kGemmTile - 1) / kGemmTile), (uint32_t)(D / kGemmTile));
    hipLaunchKernelGGL((k_dense_gemm<R>), grid, dim3(256), 0, s->stream, (const cx<R> *)s->amps, (cx<R> *)tmp,
                       nbase, D, ctrl_mask, pl, doff, dU);
    QIP_LAUNCHED();
    const uint64_t total = nbase * (uint64_t)D;
    const uint32_t sb = (uint32_t)std::min<uint64_t>((total + 255) / 256, (uint64_t)device_cus() * 64);
    hipLaunchKernelGGL((k_dense_scatter<R>), dim3(sb), dim3(256), 0, s->stream, (cx<R> *)s->amps,
                       (const cx<R> *)tmp, nbase, D, ctrl_mask, pl, doff);
    QIP_LAUNCHED();
    return QIPGPU_OK;
}

template <typename R>
int kron_general(qipgpu_state *s, int32_t n_groups, const int32_t *group_len, const int32_t *group_idx,
                 const int32_t *levels, const int32_t *kinds, const int32_t *params, const double *mats) {
    const int n = s->n;
    std::vector<KronGroupDev> groups((size_t)n_groups);
    std::vector<int32_t> pos;
    std::vector<int32_t> uq;
    size_t mat_entries = 0;
    int32_t at = 0;
    for (int g = 0; g < n_groups; ++g) {
        KronGroupDev &G = groups[g];
        G.len = group_len[g];
        G.levels = levels[g];
        G.kind = kinds[g];
        G.param = params[g];
        G.pos_at = (int32_t)pos.size();
        G.pad_ = 0;
        G.mat_at = mat_entries;
        for (int m = 0; m < G.len; ++m) {
            const int32_t q = group_idx[at + m];
            pos.push_back(n - 1 - q);
            if (std::find(uq.begin(), uq.end(), q) == uq.end()) uq.push_back(q);
        }
        at += G.len;
        if (G.kind == 1) {
            const int inner = G.len - G.levels;
            mat_entries += (size_t)1 << (2 * inner);
        }
    }
    std::sort(uq.begin(), uq.end());    // ascending qubits: the enumeration's MSB is the smallest qubit
    KronArgs a;
    a.n_groups = n_groups;
    a.u = (int32_t)uq.size();
    a.umask = 0;
    for (size_t j = 0; j < uq.size(); ++j) {
        a.upos[j] = (uint8_t)(n - 1 - uq[j]);
        a.umask |= 1ull << (n - 1 - uq[j]);
    }
    const size_t gb = groups.size() * sizeof(KronGroupDev), pb = std::max<size_t>(pos.size(), 1) * sizeof(int32_t);
    const size_t mb = std::max<size_t>(mat_entries, 1) * sizeof(cx<double>);
    StreamBuffer desc(s->stream), tmp(s->stream);
    QIP_HIP(desc.alloc(gb + pb + mb));
    char *d = (char *)desc.p;
    QIP_HIP(hipMemcpyAsync(d, groups.data(), gb, hipMemcpyHostToDevice, s->stream));
    if (!pos.empty()) QIP_HIP(hipMemcpyAsync(d + gb, pos.data(), pos.size() * sizeof(int32_t), hipMemcpyHostToDevice, s->stream));
    if (mat_entries) QIP_HIP(hipMemcpyAsync(d + gb + pb, mats, mat_entries * sizeof(cx<double>), hipMemcpyHostToDevice, s->stream));
    QIP_HIP(tmp.alloc(s->len * sizeof(cx<R>)));
    const uint32_t nb = (uint32_t)std::min<uint64_t>((s->len + 255) / 256, (uint64_t)device_cus() * 16);
    hipLaunchKernelGGL((k_kron_general<R>), dim3(nb), dim3(256), 0, s->stream, (const cx<R> *)s->amps,
                       (cx<R> *)tmp.p, s->len, a, (const KronGroupDev *)d, (const int32_t *)(d + gb),
                       (const cx<double> *)(d + gb + pb));
    QIP_LAUNCHED();
    const uint32_t cb = (uint32_t)std::min<uint64_t>((s->len + 255) / 256, (uint64_t)device_cus() * 64);
    hipLaunchKernelGGL((k_copy_amps<R>), dim3(cb), dim3(256), 0, s->stream, (cx<R> *)s->amps, (const cx<R> *)tmp.p, s->len);
    QIP_LAUNCHED();
    QIP_HIP(hipStreamSynchronize(s->stream));   // the host descriptor arrays may be pageable
    return QIPGPU_OK;
}

template <typename R>
int launch_diag_table(qipgpu_state *s, const std::vector<int> &tbits, uint64_t ctrl_mask, const std::vector<int> &cpos,
                      const std::complex<double> *d) {
    const int K = (int)tbits.size();
    const size_t D = (size_t)1 << K;
    std::vector<char> host(D * sizeof(cx<double>) + 64);
    std::memcpy(host.data(), d, D * sizeof(cx<double>));
    uint8_t *tp = (uint8_t *)(host.data() + D * sizeof(cx<double>));
    for (int b = 0; b < K; ++b) tp[b] = (uint8_t)tbits[b];
    StreamBuffer buf(s->stream);
    QIP_HIP(buf.alloc(host.size()));
    QIP_HIP(hipMemcpyAsync(buf.p, host.data(), host.size(), hipMemcpyHostToDevice, s->stream));
    const uint64_t count = s->len >> cpos.size();
    const uint32_t nb = (uint32_t)std::min<uint64_t>((count + 255) / 256, (uint64_t)device_cus() * 64);
    hipLaunchKernelGGL((k_diag_table<R>), dim3(nb), dim3(256), 0, s->stream, (cx<R> *)s->amps, count, ctrl_mask,
                       poslist(cpos), K, (const uint8_t *)buf.p + D * sizeof(cx<double>), (const cx<double> *)buf.p);
    QIP_LAUNCHED();
    QIP_HIP(hipStreamSynchronize(s->stream));   // the host copy may be pageable
    return QIPGPU_OK;
}

}  // namespace

namespace qipgpu {

int diag_large(qipgpu_state *s, const std::vector<int> &tbits, uint64_t ctrl_mask, const std::vector<int> &cpos,
               const std::complex<double> *d) {
    QIP_NOT_CAPTURING(s, "a diagonal on more than 6 targets");
    if ((int)tbits.size() > QIPGPU_MAX_DENSE)
        return set_error(QIPGPU_EUNSUP, "diagonal operator on %d qubits exceeds %d", (int)tbits.size(), QIPGPU_MAX_DENSE);
    return s->dtype == QIPGPU_C128 ? launch_diag_table<double>(s, tbits, ctrl_mask, cpos, d)
                                   : launch_diag_table<float>(s, tbits, ctrl_mask, cpos, d);
}

int dense_large(qipgpu_state *s, const std::vector<int> &tbits, uint64_t ctrl_mask, const std::vector<int> &allpos,
                const std::complex<double> *U) {
    QIP_NOT_CAPTURING(s, "a dense operator on more than 3 targets");
    const int K = (int)tbits.size();
    const bool c128 = s->dtype == QIPGPU_C128;
    switch (K) {
        case 4: return c128 ? launch_tile<double, 4>(s, tbits, ctrl_mask, allpos, U) : launch_tile<float, 4>(s, tbits, ctrl_mask, allpos, U);
        case 5: return c128 ? launch_tile<double, 5>(s, tbits, ctrl_mask, allpos, U) : launch_tile<float, 5>(s, tbits, ctrl_mask, allpos, U);
        case 6: return c128 ? launch_tile<double, 6>(s, tbits, ctrl_mask, allpos, U) : launch_tile<float, 6>(s, tbits, ctrl_mask, allpos, U);
        case 7:
            if ((s->len >> allpos.size()) / WideShape<7>::BASES < kWideTiles7) break;
            return c128 ? launch_wide<double, 7>(s, tbits, ctrl_mask, allpos, U) : launch_wide<float, 7>(s, tbits, ctrl_mask, allpos, U);
        case 8:
            if ((s->len >> allpos.size()) / WideShape<8>::BASES < kWideTiles8) break;
            return c128 ? launch_wide<double, 8>(s, tbits, ctrl_mask, allpos, U) : launch_wide<float, 8>(s, tbits, ctrl_mask, allpos, U);
        default: break;
    }
    if (K >= 7 && K <= QIPGPU_MAX_DENSE)
        return c128 ? launch_gemm<double>(s, tbits, ctrl_mask, allpos, U) : launch_gemm<float>(s, tbits, ctrl_mask, allpos, U);
    return set_error(QIPGPU_EUNSUP, "dense operator on %d target qubits exceeds %d", K, QIPGPU_MAX_DENSE);
}

}  // namespace qipgpu

extern "C" {

int qipgpu_apply_kron(qipgpu_state *s, int32_t n_groups, const int32_t *group_len, const int32_t *group_idx,
                      const int32_t *levels, const int32_t *kinds, const int32_t *params, const double *mats) {
    if (!s) return set_error(QIPGPU_EINVAL, "null state");
    QIP_NOT_CAPTURING(s, "a descriptor by the column sum");
    if (n_groups < 1) return set_error(QIPGPU_EINVAL, "a descriptor needs at least one group");
    std::vector<int32_t> all;
    int32_t at = 0;
    for (int g = 0; g < n_groups; ++g) {
        const int32_t L = group_len[g];
        if (L < 1 || L > s->n) return set_error(QIPGPU_EINVAL, "group %d has %d indices", g, L);
        if (levels[g] < 0 || levels[g] > L) return set_error(QIPGPU_EINVAL, "group %d: %d control levels", g, levels[g]);
        const int inner = L - levels[g];
        if (kinds[g] == 1) {
            if (inner > 14) return set_error(QIPGPU_EUNSUP, "group %d: a %d-qubit dense matrix", g, inner);
        } else if (kinds[g] == 3) {
            if (params[g] < 0 || 2 * params[g] != inner)
                return set_error(QIPGPU_EINVAL, "group %d: SwapMat(%d) on %d indices", g, params[g], inner);
        } else {
            return set_error(QIPGPU_EINVAL, "group %d: matrix kind %d", g, kinds[g]);
        }
        // indices within one group must differ; groups may share indices (kronprod.pyx:140-141)
        int rc = check_qubits(s, L, group_idx + at, "group indices");
        if (rc) return rc;
        for (int m = 0; m < L; ++m)
            if (std::find(all.begin(), all.end(), group_idx[at + m]) == all.end()) all.push_back(group_idx[at + m]);
        at += L;
    }
    if ((int)all.size() > 30) return set_error(QIPGPU_EUNSUP, "descriptor spans %d qubits", (int)all.size());
    int rc = flush_recorded(s);
    if (rc) return rc;
    return s->dtype == QIPGPU_C128 ? kron_general<double>(s, n_groups, group_len, group_idx, levels, kinds, params, mats)
                                   : kron_general<float>(s, n_groups, group_len, group_idx, levels, kinds, params, mats);
}

}  // extern "C"
