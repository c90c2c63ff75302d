// runs.hip -- small gates held back on a state and applied in runs, one pass over the state per run.
//
// Held gates are single-qubit operators (any 2x2 under any controls), two-qubit swaps and diagonals on
// at most two targets. A pass cuts the state into tiles: of 4096 amplitudes on large states (12 tile bits,
// state bits 0..3 among them for runs of 256 B of complex128, so up to 8 others), of 1024 on small ones
// (10 tile bits with bits 0 and 1 among them, again 8 others). Only a bit that a gate changes
// has to be a tile bit: a diagonal multiplies an amplitude by a factor that its index decides, and a
// control only decides whether an amplitude takes part, so their bits may lie anywhere. A tile is read
// once, every gate of the run is applied to it in order, and it is written once.
//
// Results. Each gate is applied by itself, with the expression its own sweep uses: a pair by k_dense's
// FP64 sums from zero, a factor by k_diag's product, each rounded to the state's precision. Gates
// change places only where that changes no amplitude's value (plan_pass). So the state is what one
// launch per gate gives, bit for bit but for the sign of a zero, as long as every amplitude is finite: X, swaps
// and factors of 1 and -1 form no products here, and a real matrix none with its zero imaginary parts, where a
// gate's own sweep multiplies by those zeros (an infinity or a NaN would make a NaN of them).
#include <algorithm>
#include <cstring>
#include <type_traits>
#include <utility>
#include <vector>

#include "engine.h"

using qipgpu::cx;
using namespace qipgpu;

namespace {

constexpr int kMaxTileBits = 12;

// How a kernel cuts the state: its tiles, the lowest state bits that are in every one, and the register
// bits of a thread's amplitudes. In layout l the registers hold tile bits
// [tile_bits - reg_bits (l + 1), tile_bits - reg_bits l).
struct Shape {
    int tile_bits, low_bits, reg_bits;
    int high_bits() const { return tile_bits - low_bits; }
    int layouts() const { return tile_bits / reg_bits; }
    int first_reg(int layout) const { return tile_bits - reg_bits * (layout + 1); }
    int layout_of(int u) const { return layouts() - 1 - u / reg_bits; }
};
constexpr Shape kWide = {12, 4, 4};      // k_tile_run
constexpr Shape kThin = {10, 2, 2};      // k_tile_thin

// What one operation of a pass does to the amplitudes whose index matches its masks.
enum OpKind : uint32_t {
    kGeneral,    // 2x2: 8 coefficients
    kReal,       // 2x2 with a real matrix: 4 coefficients (its imaginary products are all zero)
    kFlip,       // exactly X: the two amplitudes change places
    kPhase,      // a factor: 2 coefficients
    kNegate,     // the factor -1 (some lanes or all)
    kSomeGeneral, kSomeFlip, kSomePhase,   // the same for some lanes of a wave
};

// 32-bit words, read with one scalar load (narrower fields would need vector loads, whose waits also
// drain the prefetched tile).
struct __attribute__((aligned(32))) RunOp {
    uint32_t omask, oval;   // tile-index bits that have to read oval
    uint32_t tmask, tval;   // tile position bits of the thread that have to read tval
    uint32_t live;          // the registers (amplitudes, or pairs by their lower one) that take part
    uint32_t action;        // bit 4 kind + the target's register bit
    uint32_t layout;        // layout the operation is applied in
    uint32_t coef;          // first coefficient
};

// One launch's operations fit 4 KB of kernel arguments. The kernels read up to two operations and eight
// coefficients past the last.
constexpr uint32_t kAnyLayout = ~0u;    // (host) an operation without a target fits every layout
constexpr int kOpsMax = 72;
constexpr int kCoefsMax = 200;

template <typename R>
struct TileRunArgs {
    cx<R> *amps;
    uint32_t ntiles;
    uint32_t nops;
    uint32_t dead;           // tile position bits that the state does not have
    uint8_t pbits[kMaxTileBits];   // u bit i <-> state bit pbits[i]
    uint8_t zbits[kMaxTileBits];   // the same state bits, ascending (tile bases)
    RunOp op[kOpsMax + 2];
    double coef[kCoefsMax + 8];
};
static_assert(sizeof(TileRunArgs<double>) <= 4096, "kernel arguments");

template <int T, typename R>
__device__ __forceinline__ uint64_t tile_base(uint64_t t, const TileRunArgs<R> &a) {
#pragma unroll
    for (int i = 0; i < T; ++i) {
        const uint32_t p = a.zbits[i];
        const uint64_t lo = t & ((1ull << p) - 1ull);
        t = ((t ^ lo) << 1) | lo;
    }
    return t;
}

template <int LO, int HI, typename R>
__device__ __forceinline__ uint64_t u_offset(uint32_t u, const TileRunArgs<R> &a) {
    uint64_t o = 0;
#pragma unroll
    for (int i = LO; i < HI; ++i) o |= (uint64_t)((u >> i) & 1u) << a.pbits[i];
    return o;
}

// A thread's 16 amplitudes as separate real and imaginary parts. They are only ever indexed by constants
// (each16 below instead of loops), so that they are registers from the start.
template <typename R>
struct Regs {
    R re[16], im[16];
};

template <typename F, size_t... E>
__device__ __forceinline__ void each_of(F f, std::index_sequence<E...>) {
    (f(std::integral_constant<int, (int)E>()), ...);
}

// f(0) .. f(15), the argument a constant
template <typename F>
__device__ __forceinline__ void each16(F f) {
    each_of(f, std::make_index_sequence<16>());
}

// One operation's coefficients, in scalar registers.
typedef double Coefs __attribute__((ext_vector_type(8)));

// A pair (a, b) under a 2x2, in place: FP64 sums from zero in k_dense's order (a's real part is
// c0 ar - c1 ai + c2 br - c3 bi, one rounding per term). Written as instructions because the operations
// of a run meet in one loop: from plain expressions the compiler evaluated both sides of its branches
// and kept a second copy of the 16 amplitudes, which cost more than the arithmetic (8 gates on 2^24
// complex128 amplitudes: 132 us, 104 us so).
__device__ __forceinline__ void pair_general(double &ar, double &ai, double &br, double &bi, const Coefs &c) {
    double t0, t1, t2, t3;
    asm("v_mul_f64 %[t0], %[c0], %[ar]\n\t"
        "v_mul_f64 %[t1], %[c0], %[ai]\n\t"
        "v_mul_f64 %[t2], %[c4], %[ar]\n\t"
        "v_mul_f64 %[t3], %[c4], %[ai]\n\t"
        "v_fma_f64 %[t0], -%[c1], %[ai], %[t0]\n\t"
        "v_fma_f64 %[t1], %[c1], %[ar], %[t1]\n\t"
        "v_fma_f64 %[t2], -%[c5], %[ai], %[t2]\n\t"
        "v_fma_f64 %[t3], %[c5], %[ar], %[t3]\n\t"
        "v_fma_f64 %[t0], %[c2], %[br], %[t0]\n\t"
        "v_fma_f64 %[t1], %[c2], %[bi], %[t1]\n\t"
        "v_fma_f64 %[t2], %[c6], %[br], %[t2]\n\t"
        "v_fma_f64 %[t3], %[c6], %[bi], %[t3]\n\t"
        "v_fma_f64 %[ar], -%[c3], %[bi], %[t0]\n\t"
        "v_fma_f64 %[ai], %[c3], %[br], %[t1]\n\t"
        "v_fma_f64 %[t3], %[c7], %[br], %[t3]\n\t"
        "v_fma_f64 %[br], -%[c7], %[bi], %[t2]\n\t"
        "v_mov_b64 %[bi], %[t3]"
        : [ar] "+v"(ar), [ai] "+v"(ai), [br] "+v"(br), [bi] "+v"(bi), [t0] "=&v"(t0), [t1] "=&v"(t1),
          [t2] "=&v"(t2), [t3] "=&v"(t3)
        : [c0] "s"(c[0]), [c1] "s"(c[1]), [c2] "s"(c[2]), [c3] "s"(c[3]), [c4] "s"(c[4]), [c5] "s"(c[5]),
          [c6] "s"(c[6]), [c7] "s"(c[7]));
}

// The same for a real matrix, whose imaginary products are zero.
__device__ __forceinline__ void pair_real(double &ar, double &ai, double &br, double &bi, const Coefs &c) {
    double t0, t1, t2, t3;
    asm("v_mul_f64 %[t0], %[c0], %[ar]\n\t"
        "v_mul_f64 %[t1], %[c0], %[ai]\n\t"
        "v_mul_f64 %[t2], %[c2], %[ar]\n\t"
        "v_mul_f64 %[t3], %[c2], %[ai]\n\t"
        "v_fma_f64 %[ar], %[c1], %[br], %[t0]\n\t"
        "v_fma_f64 %[ai], %[c1], %[bi], %[t1]\n\t"
        "v_fma_f64 %[br], %[c3], %[br], %[t2]\n\t"
        "v_fma_f64 %[bi], %[c3], %[bi], %[t3]"
        : [ar] "+v"(ar), [ai] "+v"(ai), [br] "+v"(br), [bi] "+v"(bi), [t0] "=&v"(t0), [t1] "=&v"(t1),
          [t2] "=&v"(t2), [t3] "=&v"(t3)
        : [c0] "s"(c[0]), [c1] "s"(c[1]), [c2] "s"(c[2]), [c3] "s"(c[3]));
}

// An amplitude times a factor, in k_diag's order.
__device__ __forceinline__ void factor(double &re, double &im, const Coefs &c) {
    double t0, t1;
    asm("v_mul_f64 %[t0], %[c1], %[im]\n\t"
        "v_mul_f64 %[t1], %[c1], %[re]\n\t"
        "v_fma_f64 %[re], %[c0], %[re], -%[t0]\n\t"
        "v_fma_f64 %[im], %[c0], %[im], %[t1]"
        : [re] "+v"(re), [im] "+v"(im), [t0] "=&v"(t0), [t1] "=&v"(t1)
        : [c0] "s"(c[0]), [c1] "s"(c[1]));
}

__device__ __forceinline__ void exchange(double &a, double &b) {
    double t;
    asm("v_mov_b64 %[t], %[a]\n\tv_mov_b64 %[a], %[b]\n\tv_mov_b64 %[b], %[t]"
        : [a] "+v"(a), [b] "+v"(b), [t] "=&v"(t));
}

__device__ __forceinline__ void exchange(float &a, float &b) {
    asm("v_swap_b32 %[a], %[b]" : [a] "+v"(a), [b] "+v"(b));
}

// A sign turned on the lanes where `sign` is 0x80000000 (0 elsewhere).
__device__ __forceinline__ void turn(double &a, uint32_t sign) {
    a = __hiloint2double(__double2hiint(a) ^ (int)sign, __double2loint(a));
}

__device__ __forceinline__ void turn(float &a, uint32_t sign) {
    a = __uint_as_float(__float_as_uint(a) ^ sign);
}

// One operation on register bit J. `live` is uniform, so a pair that takes no part costs a scalar
// branch. SOME: on the lanes where `on` holds; the others compute too and keep what they had, which
// leaves every branch of the kernel uniform.
template <typename R, int KIND, bool SOME, int J>
__device__ __forceinline__ void pairs(Regs<R> &x, const Coefs &c, uint32_t live, bool on) {
    each16([&](auto E) {
        constexpr int e = E, f = e | (1 << J);
        if constexpr (e != f) {
            if (!(live >> e & 1u)) return;
            if constexpr (KIND == kFlip && !SOME) {
                exchange(x.re[e], x.re[f]);
                exchange(x.im[e], x.im[f]);
            } else if constexpr (KIND == kFlip) {
                const R ar = x.re[e], ai = x.im[e], br = x.re[f], bi = x.im[f];
                x.re[e] = on ? br : ar;
                x.im[e] = on ? bi : ai;
                x.re[f] = on ? ar : br;
                x.im[f] = on ? ai : bi;
            } else {
                double ar = x.re[e], ai = x.im[e], br = x.re[f], bi = x.im[f];
                if constexpr (KIND == kReal) pair_real(ar, ai, br, bi, c);
                else pair_general(ar, ai, br, bi, c);
                x.re[e] = !SOME || on ? (R)ar : x.re[e];
                x.im[e] = !SOME || on ? (R)ai : x.im[e];
                x.re[f] = !SOME || on ? (R)br : x.re[f];
                x.im[f] = !SOME || on ? (R)bi : x.im[f];
            }
        }
    });
}

template <typename R, bool SOME>
__device__ __forceinline__ void factors(Regs<R> &x, const Coefs &c, uint32_t live, bool on) {
    each16([&](auto E) {
        constexpr int e = E;
        if (!(live >> e & 1u)) return;
        double re = x.re[e], im = x.im[e];
        factor(re, im, c);
        x.re[e] = !SOME || on ? (R)re : x.re[e];
        x.im[e] = !SOME || on ? (R)im : x.im[e];
    });
}

template <typename R>
__device__ __forceinline__ void negate(Regs<R> &x, uint32_t live, bool on) {
    const uint32_t sign = on ? 0x80000000u : 0u;
    each16([&](auto E) {
        constexpr int e = E;
        if (!(live >> e & 1u)) return;
        turn(x.re[e], sign);
        turn(x.im[e], sign);
    });
}

template <typename R, int KIND, bool SOME>
__device__ __forceinline__ void pairs_on(Regs<R> &x, uint32_t regs, const RunOp &op, const Coefs &c, bool on) {
    if (regs & 1u) pairs<R, KIND, SOME, 0>(x, c, op.live, on);
    if (regs & 2u) pairs<R, KIND, SOME, 1>(x, c, op.live, on);
    if (regs & 4u) pairs<R, KIND, SOME, 2>(x, c, op.live, on);
    if (regs & 8u) pairs<R, KIND, SOME, 3>(x, c, op.live, on);
}

// The action is one bit of 32, tested bit by bit: to the compiler the branches are then independent,
// each leaving the amplitudes where they are, while the branches of a switch meet in one place with a
// copy of all 16 from each. In two groups, so that an operation jumps over few others (order finding on 27 qubits,
// 170 phases: 11.75 -> 11.3 ms).
template <typename R>
__device__ __forceinline__ void apply_op(Regs<R> &x, const RunOp &op, const Coefs &c, bool on) {
    const uint32_t act = op.action;
    constexpr uint32_t kFactors = 1u << 4 * kPhase | 1u << 4 * kNegate | 1u << 4 * kSomePhase;
    if (act & kFactors) {
        if (act & 1u << 4 * kPhase) factors<R, false>(x, c, op.live, on);
        if (act & 1u << 4 * kNegate) negate<R>(x, op.live, on);
        if (act & 1u << 4 * kSomePhase) factors<R, true>(x, c, op.live, on);
    }
    if (act & ~kFactors) {
        if (act & 0xfu << 4 * kGeneral) pairs_on<R, kGeneral, false>(x, act >> 4 * kGeneral, op, c, on);
        if (act & 0xfu << 4 * kReal) pairs_on<R, kReal, false>(x, act >> 4 * kReal, op, c, on);
        if (act & 0xfu << 4 * kFlip) pairs_on<R, kFlip, false>(x, act >> 4 * kFlip, op, c, on);
        if (act & 0xfu << 4 * kSomeGeneral) pairs_on<R, kGeneral, true>(x, act >> 4 * kSomeGeneral, op, c, on);
        if (act & 0xfu << 4 * kSomeFlip) pairs_on<R, kFlip, true>(x, act >> 4 * kSomeFlip, op, c, on);
    }
}

// Tile position u of register e in each layout: A: tid + 256 e;  B: (tid & 15) | e << 4 | (tid >> 4) << 8;
// C: tid << 4 | e. Position u sits in LDS slot u + u / 16, so a layout's slots are a per-thread base
// plus a constant per register (A 272 e, B 17 e, C e).
template <int STRIDE, typename R>
__device__ __forceinline__ void put16(cx<R> *p, const Regs<R> &x) {
    each16([&](auto E) {
        constexpr int e = E;
        cx<R> v;
        v.re = x.re[e];
        v.im = x.im[e];
        p[STRIDE * e] = v;
    });
}

template <int STRIDE, typename R>
__device__ __forceinline__ void get16(const cx<R> *p, Regs<R> &x) {
    each16([&](auto E) {
        constexpr int e = E;
        const cx<R> v = p[STRIDE * e];
        x.re[e] = v.re;
        x.im[e] = v.im;
    });
}

template <typename R>
__device__ __forceinline__ void lds_put(cx<R> *t, const Regs<R> &x, uint32_t layout, uint32_t tid) {
    if (layout == 0) put16<272>(t + tid + (tid >> 4), x);
    else if (layout == 1) put16<17>(t + (tid & 15u) + 272u * (tid >> 4), x);
    else put16<1>(t + 17u * tid, x);
}

// The (empty) instructions at the ends of the branches differ, or the compiler sinks the loads into the place
// where they meet, in halves and with a second set of registers (250 VGPRs for 164).
template <typename R>
__device__ __forceinline__ void lds_get(const cx<R> *t, Regs<R> &x, uint32_t layout, uint32_t tid) {
    if (layout == 0) {
        get16<272>(t + tid + (tid >> 4), x);
        asm volatile("; layout A");
    } else if (layout == 1) {
        get16<17>(t + (tid & 15u) + 272u * (tid >> 4), x);
        asm volatile("; layout B");
    } else {
        get16<1>(t + 17u * tid, x);
        asm volatile("; layout C");
    }
}

template <typename R>
__device__ __forceinline__ void tile_load(Regs<R> &x, uint64_t base, const TileRunArgs<R> &a) {
    each16([&](auto E) {
        constexpr int e = E;
        const cx<R> v = a.amps[base + u_offset<8, 12>(256u * e, a)];
        x.re[e] = v.re;
        x.im[e] = v.im;
    });
}

template <typename R>
__device__ __forceinline__ Coefs coefs_at(const TileRunArgs<R> &a, uint32_t at) {
    typedef Coefs Unaligned __attribute__((aligned(8)));
    return *reinterpret_cast<const Unaligned *>(a.coef + at);
}

// Bound: HBM for complex128, the FP64 arithmetic and the roundings between gates for complex64. Per pass
// at 28 qubits, 8 Haar gates and 4 CNOTs: complex128 2220 us before, 1860 us now (4.6 TB/s; a copy of
// that size takes 1627); complex64 1704 and 1397 (813). 12 Haar gates on the lowest bits: 2297 and 2093,
// 1729 and 1790. A 28-qubit depth-20 layered circuit, 20 passes of CNOTs and CZs fewer as well: 200 ms
// before, 117 ms now.
//
// 256 threads, 16 amplitudes each. The four tile bits that vary across a thread's registers are u bits
// 8..11 as loaded (layout A), 4..7 (B) or 0..3 (C); an operation is applied in the layout that has its
// target among them, and the tile moves between layouts through LDS. The host puts the first four
// targets above bit 3 on u bits 8..11 and the other four on 4..7, so the usual run of gates on 8 high
// bits takes one move (A, then B, stored from B) where a pass that keeps the tile in LDS takes a read
// and a write for every gate or two. The next tile's loads are in flight while one is worked on.
template <typename R>
__global__ __launch_bounds__(256, sizeof(R) == 8 ? 2 : 4) void k_tile_run(const TileRunArgs<R> a) {
    __shared__ cx<R> t[4096 + 256];
    const uint32_t tid = threadIdx.x;
    const uint64_t off_a = u_offset<0, 8>(tid, a);
    const uint64_t off_b = u_offset<0, 12>((tid & 15u) | (tid >> 4) << 8, a);
    const uint32_t per = (a.ntiles + gridDim.x - 1) / gridDim.x;
    uint32_t tile = blockIdx.x * per;
    const uint32_t end = min(tile + per, a.ntiles);
    if (tile >= end) return;   // the same for every thread of the workgroup
    Regs<R> nx;
    tile_load<R>(nx, tile_base<12>(tile, a) + off_a, a);
    for (bool first = true;; first = false) {
        Regs<R> x = nx;
        const uint64_t base = tile_base<12>(tile, a);
        tile_load<R>(nx, tile_base<12>(min(tile + 1, end - 1), a) + off_a, a);
        // a tile's first move writes slots that others may still read from the tile before
        bool fresh = !first;
        uint32_t layout = 0, ut = tid;
        // each operation and its coefficients are read while the one before it is applied
        RunOp op = a.op[0];
        Coefs c = coefs_at(a, op.coef);
        for (uint32_t q = 0; q < a.nops; ++q) {
            const RunOp nop = a.op[q + 1];
            if (op.layout != layout) {
                if (fresh) __syncthreads();
                fresh = false;
                lds_put(t, x, layout, tid);
                __syncthreads();
                layout = op.layout;
                lds_get(t, x, layout, tid);
                ut = layout == 0 ? tid : layout == 1 ? ((tid & 15u) | (tid >> 4) << 8) : tid << 4;
            }
            const Coefs nc = coefs_at(a, nop.coef);
            if (((tile ^ op.oval) & op.omask) == 0) {
                const bool on = ((ut ^ op.tval) & op.tmask) == 0;
                if (__ballot(on) != 0) apply_op<R>(x, op, c, on);
            }
            op = nop;
            c = nc;
        }
        if (layout == 2) {   // lanes of C run 16 amplitudes apart: back to the layout the tile came in
            if (fresh) __syncthreads();
            lds_put(t, x, layout, tid);
            __syncthreads();
            lds_get(t, x, 0, tid);
            layout = 0;
        }
        if (layout == 0) {
            each16([&](auto E) {
                constexpr int e = E;
                cx<R> v;
                v.re = x.re[e];
                v.im = x.im[e];
                a.amps[base + off_a + u_offset<8, 12>(256u * e, a)] = v;
            });
        } else {
            each16([&](auto E) {
                constexpr int e = E;
                cx<R> v;
                v.re = x.re[e];
                v.im = x.im[e];
                a.amps[base + off_b + u_offset<4, 8>(16u * e, a)] = v;
            });
        }
        if (++tile >= end) return;
    }
}

// One operation on four amplitudes, register bit J its target; the registers of `live` and the lanes of `on`
// keep the result.
template <typename R, int KIND, int J>
__device__ __forceinline__ void thin_pairs(R (&re)[4], R (&im)[4], const Coefs &c, uint32_t live, bool on) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        constexpr int f = 1 << J;
        const int e = J == 0 ? 2 * i : i;
        const bool keep = on && (live >> e & 1u);
        double ar = re[e], ai = im[e], br = re[e + f], bi = im[e + f];
        if constexpr (KIND == kFlip) {
            const double tr = ar, ti = ai;
            ar = br;
            ai = bi;
            br = tr;
            bi = ti;
        } else if constexpr (KIND == kReal) {
            pair_real(ar, ai, br, bi, c);
        } else {
            pair_general(ar, ai, br, bi, c);
        }
        re[e] = keep ? (R)ar : re[e];
        im[e] = keep ? (R)ai : im[e];
        re[e + f] = keep ? (R)br : re[e + f];
        im[e + f] = keep ? (R)bi : im[e + f];
    }
}

// The same passes on small states, whose few tiles leave a kernel waiting on itself: k_tile_run's 16 amplitudes
// a thread take an operation's pairs one after the other on 16 CUs of a 16-qubit state, through 42 KB
// of code that each pass fetches anew. Here a tile has 1024 amplitudes, four to a thread, and an operation is
// the same few instructions for each. Two tile bits vary across a thread's registers, so a tile moves
// through LDS for every other target; a thread writes the slots it read, and a state that lives in the
// caches may be stored from any layout.
template <typename R>
__global__ __launch_bounds__(256) void k_tile_thin(const TileRunArgs<R> a) {
    constexpr int T = kThin.tile_bits;
    __shared__ cx<R> t[(1 << T) + (1 << (T - 4))];
    const uint32_t tid = threadIdx.x, tile = blockIdx.x;
    const uint64_t base = tile_base<T>(tile, a);
    // the first tile position of this thread's registers with their bits from `lo` on
    auto first = [&](uint32_t lo) { return (tid & ((1u << lo) - 1u)) | (tid >> lo) << (lo + 2); };
    uint32_t layout = 0, lo = T - 2, u = first(lo);
    R re[4], im[4];
#pragma unroll
    for (uint32_t e = 0; e < 4; ++e) {
        re[e] = 0;
        im[e] = 0;
        if ((u | e << lo) & a.dead) continue;
        const cx<R> v = a.amps[base + u_offset<0, T>(u | e << lo, a)];
        re[e] = v.re;
        im[e] = v.im;
    }
    // an operation's coefficients are read while the one before it is applied, its other words while the one
    // before that is
    RunOp op = a.op[0], nop = a.op[1];
    Coefs c = coefs_at(a, op.coef);
    for (uint32_t q = 0; q < a.nops; ++q) {
        const Coefs nc = coefs_at(a, nop.coef);
        const RunOp nnop = a.op[q + 2];
        if (op.layout != layout) {
#pragma unroll
            for (uint32_t e = 0; e < 4; ++e) {
                const uint32_t p = u | e << lo;
                cx<R> v;
                v.re = re[e];
                v.im = im[e];
                t[p + (p >> 4)] = v;
            }
            __syncthreads();
            layout = op.layout;
            lo = T - 2 - 2 * layout;
            u = first(lo);
#pragma unroll
            for (uint32_t e = 0; e < 4; ++e) {
                const uint32_t p = u | e << lo;
                const cx<R> v = t[p + (p >> 4)];
                re[e] = v.re;
                im[e] = v.im;
            }
        }
        if (((tile ^ op.oval) & op.omask) == 0) {
            const bool on = ((u ^ op.tval) & op.tmask) == 0;
            const uint32_t act = op.action;
            // nested, so that an operation jumps over few others
            if (act & 1u << 4 * kPhase) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const bool keep = on && (op.live >> e & 1u);
                    double vr = re[e], vi = im[e];
                    factor(vr, vi, c);
                    re[e] = keep ? (R)vr : re[e];
                    im[e] = keep ? (R)vi : im[e];
                }
            } else if (act & 1u << 4 * kNegate) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t sign = on && (op.live >> e & 1u) ? 0x80000000u : 0u;
                    turn(re[e], sign);
                    turn(im[e], sign);
                }
            } else if (act & (1u << 4 * kGeneral | 1u << 4 * kReal | 1u << 4 * kFlip)) {
                if (act & 1u << 4 * kGeneral) thin_pairs<R, kGeneral, 0>(re, im, c, op.live, on);
                else if (act & 1u << 4 * kReal) thin_pairs<R, kReal, 0>(re, im, c, op.live, on);
                else thin_pairs<R, kFlip, 0>(re, im, c, op.live, on);
            } else {
                if (act & 2u << 4 * kGeneral) thin_pairs<R, kGeneral, 1>(re, im, c, op.live, on);
                else if (act & 2u << 4 * kReal) thin_pairs<R, kReal, 1>(re, im, c, op.live, on);
                else thin_pairs<R, kFlip, 1>(re, im, c, op.live, on);
            }
        }
        op = nop;
        nop = nnop;
        c = nc;
    }
#pragma unroll
    for (uint32_t e = 0; e < 4; ++e) {
        if ((u | e << lo) & a.dead) continue;
        cx<R> v;
        v.re = re[e];
        v.im = im[e];
        a.amps[base + u_offset<0, T>(u | e << lo, a)] = v;
    }
}

// States of up to 19 qubits take the thin kernel, but for one kind of pass on 19. Graphs of a Fourier transform / of 8 layers of a random circuit, us a
// launch, wide -> thin: complex128 10 qubits 56 / 107 -> 37 / 64, 13 80 / 149 -> 53 / 95, 16 110 / 184 -> 71 / 122, 18 127 / 226
// -> 86 / 176, 19 154 / 275 -> 127 / 265, 20 177 / 311 -> 203 / 356 (its 1024 tiles fill the GPU, and a pass's instructions
// for four amplitudes count again); complex64 10 52 / 108 -> 36 / 61, 13 75 / 154 -> 48 / 99, 16 104 / 191 -> 63 / 124, 18 121 /
// 222 -> 75 / 163, 19 142 / 251 -> 110 / 232, 20 157 / 289 -> 176 / 367. On 19 qubits passes of nothing but single-qubit
// operators, a move through LDS for every other one, are the wide kernel's: a layer of them 47 / 43 us thin and 38 to 41 /
// 35 to 38 wide (complex128 / complex64), while swaps, phases and controlled gates are the thin one's (19 phases 20 / 19 and
// 25 / 25).
constexpr int kThinQubits = 19;

Shape shape_of(const qipgpu_state *s) {
    if (s->n != kThinQubits) return s->n > kThinQubits ? kWide : kThin;
    for (const HeldGate &g : s->held)
        if (g.kind != HeldGate::kSingle || g.ctrl_mask) return kThin;
    return kWide;
}

// Exchanges of state bits, all at once: amplitude i and amplitude P(i) change places, P the permutation of
// the index bits that exchanges bit a.at(j) with b.at(j) for every j (all different). One pass over the amplitudes
// that move, where tiles take the exchanges four to a pass. P acts on each index bit by itself, so a
// workgroup's part of P(i) is formed once, in scalar registers, and a thread's part once per launch.
// Bound: HBM, in runs of 2^(lowest exchanged bit) amplitudes.
constexpr int kExchangesMax = 17;      // disjoint pairs of 34 state bits
constexpr int kExchangeItems = 4;

template <typename R>
struct ExchangeArgs {
    cx<R> *amps;
    uint64_t nblocks;       // of 256 kExchangeItems amplitudes
    uint64_t of_item[kExchangeItems];   // P(256 it)
    PosList a, b;
    PosList order;          // the state bit of each bit of the block number
};

template <typename R>
__host__ __device__ __forceinline__ uint64_t exchanged(uint64_t i, const ExchangeArgs<R> &x) {
    for (int j = 0; j < x.a.count; ++j) {
        const uint32_t p = x.a.at(j), q = x.b.at(j);
        const uint64_t d = (i >> p ^ i >> q) & 1ull;
        i ^= d << p | d << q;
    }
    return i;
}

template <typename R>
__global__ __launch_bounds__(256) void k_exchange(const ExchangeArgs<R> x) {
    const uint64_t of_thread = exchanged<R>(threadIdx.x, x);
    for (uint64_t blk = blockIdx.x; blk < x.nblocks; blk += gridDim.x) {
        uint64_t base = 0;
        for (int b = 0; b < x.order.count; ++b) base |= (blk >> b & 1ull) << x.order.at(b);
        const uint64_t to = exchanged<R>(base, x);
        uint64_t i[kExchangeItems], j[kExchangeItems];
        bool any = false;
#pragma unroll
        for (int it = 0; it < kExchangeItems; ++it) {
            i[it] = base + 256 * it + threadIdx.x;
            j[it] = to | x.of_item[it] | of_thread;
            any = any || i[it] < j[it];
        }
        if (__ballot(any) == 0) continue;      // the other side's waves move these
        // a lane whose amplitude stays, or is another lane's to move, reads it and writes nothing: loads
        // without a branch are all in flight at once
        R vr[kExchangeItems], vi[kExchangeItems], wr[kExchangeItems], wi[kExchangeItems];
#pragma unroll
        for (int it = 0; it < kExchangeItems; ++it) {
            const cx<R> v = x.amps[i[it]], w = x.amps[i[it] < j[it] ? j[it] : i[it]];
            vr[it] = v.re;
            vi[it] = v.im;
            wr[it] = w.re;
            wi[it] = w.im;
        }
#pragma unroll
        for (int it = 0; it < kExchangeItems; ++it)
            if (i[it] < j[it]) {
                cx<R> v, w;
                v.re = vr[it];
                v.im = vi[it];
                w.re = wr[it];
                w.im = wi[it];
                x.amps[i[it]] = w;
                x.amps[j[it]] = v;
            }
    }
}

// ---- host side -------------------------------------------------------------------------------------

uint64_t changed_bits(const HeldGate &g) {
    if (g.kind == HeldGate::kDiagonal) return 0;
    uint64_t m = 0;
    for (int i = 0; i < g.k; ++i) m |= 1ull << g.tpos[i];
    return m;
}

uint64_t all_bits(const HeldGate &g) {
    uint64_t m = g.ctrl_mask;
    for (int i = 0; i < g.k; ++i) m |= 1ull << g.tpos[i];
    return m;
}

bool is_x(const HeldGate &g) {
    return g.m[0].re == 0.0 && g.m[0].im == 0.0 && g.m[1].re == 1.0 && g.m[1].im == 0.0 && g.m[2].re == 1.0 &&
           g.m[2].im == 0.0 && g.m[3].re == 0.0 && g.m[3].im == 0.0;
}

// Gates that round nothing: X and swaps move amplitudes, a factor -1 (CZ) turns their signs.
bool rounds_nothing(const HeldGate &g) {
    if (g.kind == HeldGate::kSwap) return true;
    if (g.kind == HeldGate::kSingle) return is_x(g);
    return g.k == 0 && g.m[0].re == -1.0 && g.m[0].im == 0.0;
}

// Whether a gate may go before gates that come earlier, given what those change and read: gates that
// act on disjoint bits (apart from bits that both only read) commute as operators, and when one of the
// two only moves amplitudes or turns signs, the other does the same arithmetic on the same values in
// either order. Two gates that both round never change places.
struct Passed {
    uint64_t changed = 0, bits = 0;
    bool any = false, rounds = false;

    bool lets(const HeldGate &g) const {
        if (!any) return true;
        if (rounds && !rounds_nothing(g)) return false;
        return !(changed_bits(g) & bits) && !(all_bits(g) & changed);
    }
    void add(const HeldGate &g) {
        any = true;
        rounds = rounds || !rounds_nothing(g);
        changed |= changed_bits(g);
        bits |= all_bits(g);
    }
};

bool is_real(const HeldGate &g) {
    return g.m[0].im == 0.0 && g.m[1].im == 0.0 && g.m[2].im == 0.0 && g.m[3].im == 0.0;
}

// Operations and coefficients of a gate in a pass.
void op_counts(const HeldGate &g, int *ops, int *coefs) {
    *ops = 1;
    *coefs = 0;
    if (g.kind == HeldGate::kSwap) {
        *ops = 3;
    } else if (g.kind == HeldGate::kSingle) {
        *coefs = is_x(g) ? 0 : is_real(g) && !g.ctrl_mask ? 4 : 8;
    } else {
        *ops = 1 << g.k;
        *coefs = 2 * *ops;
    }
}

// A swap that k_exchange may take: no controls, and neither bit among those that every tile holds (its runs
// would be shorter than a tile's).
bool exchanges(const Shape &sh, int n, const HeldGate &g) {
    return n > sh.tile_bits && g.kind == HeldGate::kSwap && !g.ctrl_mask && g.tpos[0] >= sh.low_bits &&
           g.tpos[1] >= sh.low_bits;
}

// The swaps that the next k_exchange takes: the first held gate, and every later one on other bits that
// may go before the gates left behind.
void plan_exchange(const Shape &sh, int n, const std::vector<HeldGate> &held, std::vector<char> &taken) {
    taken.assign(held.size(), 0);
    uint64_t bits = 0;
    Passed left;
    for (size_t i = 0; i < held.size(); ++i) {
        const HeldGate &g = held[i];
        if (!exchanges(sh, n, g) || (changed_bits(g) & bits) || !left.lets(g)) {
            left.add(g);
            continue;
        }
        bits |= changed_bits(g);
        taken[i] = 1;
    }
}

// The held gates that the next pass takes, in order: the first, and every later one whose changed bits
// fit the tile beside those taken and that may go before the gates left behind. On a layered circuit
// the CNOTs and CZs of a layer so join the passes of its single-qubit gates. A swap that would bring two
// bits of its own is left for k_exchange.
void plan_pass(const Shape &sh, int n, const std::vector<HeldGate> &held, std::vector<char> &taken) {
    taken.assign(held.size(), 0);
    uint64_t high = 0;
    int ops = 0, coefs = 0;
    Passed left;
    for (size_t i = 0; i < held.size(); ++i) {
        const HeldGate &g = held[i];
        const uint64_t h = (high | changed_bits(g)) & ~((1ull << sh.low_bits) - 1ull);
        int no, nc;
        op_counts(g, &no, &nc);
        const bool apart = exchanges(sh, n, g) && __builtin_popcountll(h & ~high) > 1;
        if (apart || !left.lets(g) || __builtin_popcountll(h) > sh.high_bits() || ops + no > kOpsMax || coefs + nc > kCoefsMax) {
            left.add(g);
            continue;
        }
        high = h;
        ops += no;
        coefs += nc;
        taken[i] = 1;
    }
}

template <typename R>
int launch_pass(qipgpu_state *s, const Shape &shape, const std::vector<HeldGate> &gates) {
    const int n = s->n;
    TileRunArgs<R> a;
    std::memset(&a, 0, sizeof(a));
    a.amps = (cx<R> *)s->amps;
    a.ntiles = n > shape.tile_bits ? 1u << (n - shape.tile_bits) : 1u;
    // tile position of each state bit: the low bits on the lowest, changed bits by first use on the registers
    // of layout 0, then of 1 and so on, the lowest other bits on what is left (position bits a small
    // state has no bit for are dead)
    int upos[64], state_bit[kMaxTileBits];
    std::fill(upos, upos + 64, -1);
    std::fill(state_bit, state_bit + kMaxTileBits, -1);
    auto place = [&](int p, int u) {
        upos[p] = u;
        state_bit[u] = p;
    };
    for (int p = 0; p < shape.low_bits && p < n; ++p) place(p, p);
    int order[kMaxTileBits], next = 0;
    for (int l = 0; l < shape.layouts(); ++l)
        for (int j = 0; j < shape.reg_bits; ++j) order[l * shape.reg_bits + j] = shape.first_reg(l) + j;
    for (const HeldGate &g : gates)
        for (int i = 0; i < g.k && g.kind != HeldGate::kDiagonal; ++i)
            if (upos[g.tpos[i]] < 0) place(g.tpos[i], order[next++]);
    // free positions: the lowest first (longer runs together), from the free bits in the order 0..5, 12..17,
    // 6..11, 18..: the memory pattern measured fastest for tiles
    std::vector<int> fill;
    for (int p = 0; p < 6; ++p) fill.push_back(p);
    for (int p = 12; p < 18; ++p) fill.push_back(p);
    for (int p = 6; p < 12; ++p) fill.push_back(p);
    for (int p = 18; p < 64; ++p) fill.push_back(p);
    size_t f = 0;
    for (int u = 0; u < shape.tile_bits; ++u) {
        if (state_bit[u] >= 0) continue;
        while (f < fill.size() && (fill[f] >= n || upos[fill[f]] >= 0)) ++f;
        if (f < fill.size()) place(fill[f], u);
    }
    std::vector<int> sorted;
    for (int u = 0; u < shape.tile_bits; ++u) {
        if (state_bit[u] < 0) {
            a.dead |= 1u << u;
            continue;
        }
        a.pbits[u] = (uint8_t)state_bit[u];
        sorted.push_back(state_bit[u]);
    }
    std::sort(sorted.begin(), sorted.end());
    for (size_t i = 0; i < sorted.size(); ++i) a.zbits[i] = (uint8_t)sorted[i];
    // bits outside the tile, ascending, are the tile index's bits
    int tpos[64], nt = 0;
    for (int p = 0; p < n; ++p) tpos[p] = upos[p] < 0 ? nt++ : -1;

    // the operations in the order the gates come, then sorted into stays in one layout: from the layout
    // at hand every operation that can be applied there and may go before those left, then on to
    // the layout of the first one left
    struct Part {
        RunOp op;
        HeldGate gate;      // the elementary gate, for what may change places
        bool done;
    };
    std::vector<Part> parts;
    int ncoef = 0;
    // tmask / tval hold every tile position bit until the operation's layout is known
    auto masks = [&](RunOp &op, uint64_t mask, uint64_t val) {
        for (int p = 0; p < n; ++p) {
            if (!(mask >> p & 1)) continue;
            if (upos[p] >= 0) {
                op.tmask |= 1u << upos[p];
                if (val >> p & 1) op.tval |= 1u << upos[p];
            } else {
                op.omask |= 1u << tpos[p];
                if (val >> p & 1) op.oval |= 1u << tpos[p];
            }
        }
    };
    auto target = [&](RunOp &op, int p) {
        op.layout = (uint32_t)shape.layout_of(upos[p]);
        op.action <<= upos[p] % shape.reg_bits;
    };
    auto push = [&](const RunOp &op, const HeldGate &g) { parts.push_back(Part{op, g, false}); };
    for (const HeldGate &g : gates) {
        if (g.kind == HeldGate::kSingle) {
            RunOp op;
            std::memset(&op, 0, sizeof(op));
            // a real matrix under controls takes the general form, which also serves some lanes only
            const OpKind kind = is_x(g) ? kFlip : is_real(g) && !g.ctrl_mask ? kReal : kGeneral;
            op.action = 1u << 4 * kind;
            op.coef = (uint32_t)ncoef;
            for (int i = 0; i < 4 && kind != kFlip; ++i) {
                a.coef[ncoef++] = g.m[i].re;
                if (kind == kGeneral) a.coef[ncoef++] = g.m[i].im;
            }
            masks(op, g.ctrl_mask, g.ctrl_mask);
            target(op, g.tpos[0]);
            push(op, g);
        } else if (g.kind == HeldGate::kSwap) {
            // b ^= a, a ^= b, b ^= a
            for (int i = 0; i < 3; ++i) {
                const int t = g.tpos[i == 1 ? 0 : 1], c = g.tpos[i == 1 ? 1 : 0];
                HeldGate x = g;
                x.kind = HeldGate::kSingle;
                x.k = 1;
                x.tpos[0] = (uint8_t)t;
                x.ctrl_mask = g.ctrl_mask | (1ull << c);
                std::memset(x.m, 0, sizeof(x.m));
                x.m[1].re = x.m[2].re = 1.0;
                RunOp op;
                std::memset(&op, 0, sizeof(op));
                op.action = 1u << 4 * kFlip;
                masks(op, x.ctrl_mask, x.ctrl_mask);
                target(op, t);
                push(op, x);
            }
        } else {
            // one operation per value of the targets; a factor of exactly 1 changes nothing
            for (int j = 0; j < (1 << g.k); ++j) {
                if (g.m[j].re == 1.0 && g.m[j].im == 0.0) continue;
                uint64_t mask = g.ctrl_mask, val = g.ctrl_mask;
                for (int b = 0; b < g.k; ++b) {
                    mask |= 1ull << g.tpos[b];
                    if (j >> (g.k - 1 - b) & 1) val |= 1ull << g.tpos[b];
                }
                RunOp op;
                std::memset(&op, 0, sizeof(op));
                const OpKind kind = g.m[j].re == -1.0 && g.m[j].im == 0.0 ? kNegate : kPhase;
                op.action = 1u << 4 * kind;
                op.layout = kAnyLayout;
                op.coef = (uint32_t)ncoef;
                if (kind == kPhase) {
                    a.coef[ncoef++] = g.m[j].re;
                    a.coef[ncoef++] = g.m[j].im;
                }
                masks(op, mask, val);
                push(op, g);
            }
        }
    }
    uint32_t layout = 0;
    for (size_t done = 0; done < parts.size();) {
        Passed left;
        int goal = -1;
        for (Part &p : parts) {
            if (p.done) continue;
            if ((p.op.layout == layout || p.op.layout == kAnyLayout) && left.lets(p.gate)) {
                RunOp &op = a.op[a.nops++] = p.op;
                const uint32_t regs = 1u << shape.reg_bits, sh = (uint32_t)shape.first_reg((int)layout);
                const uint32_t rm = op.tmask >> sh & (regs - 1u), rv = op.tval >> sh & (regs - 1u);
                op.layout = layout;
                op.tmask &= ~((regs - 1u) << sh);
                op.tval &= ~((regs - 1u) << sh);
                for (uint32_t e = 0; e < regs; ++e)
                    if ((e & rm) == rv) op.live |= 1u << e;
                if (op.tmask && shape.reg_bits == kWide.reg_bits) {     // some lanes of a wave
                    if (op.action & 0xfu << 4 * kGeneral) op.action <<= 4 * (kSomeGeneral - kGeneral);
                    else if (op.action & 0xfu << 4 * kFlip) op.action <<= 4 * (kSomeFlip - kFlip);
                    else if (op.action & 1u << 4 * kPhase) op.action <<= 4 * (kSomePhase - kPhase);
                }
                p.done = true;
                ++done;
            } else {
                if (goal < 0) goal = p.op.layout;
                left.add(p.gate);
            }
        }
        if (done < parts.size()) layout = (uint32_t)goal;
    }
    if (!a.nops) return QIPGPU_OK;
    if (shape.reg_bits == kWide.reg_bits) {
        const uint32_t grid = std::min<uint32_t>(a.ntiles, (uint32_t)device_cus() * (sizeof(R) == 8 ? 2 : 4));
        return launch_gate(s, &k_tile_run<R>, dim3(grid), dim3(256), a);
    }
    return launch_gate(s, &k_tile_thin<R>, dim3(a.ntiles), dim3(256), a);
}

template <typename R>
int launch_exchange(qipgpu_state *s, const std::vector<HeldGate> &swaps) {
    ExchangeArgs<R> a;
    std::memset(&a, 0, sizeof(a));
    a.amps = (cx<R> *)s->amps;
    a.nblocks = s->len / (256 * kExchangeItems);
    if (swaps.size() > (size_t)kExchangesMax) return set_error(QIPGPU_EINVAL, "%zu disjoint swaps", swaps.size());
    for (const HeldGate &g : swaps) {
        a.a.set(a.a.count++, g.tpos[0]);
        a.b.set(a.b.count++, g.tpos[1]);
    }
    // block numbers count the lowest and the highest bits in turn: the workgroups in flight then differ in
    // both, so neither their amplitudes nor those these change places with lie all at one offset of the memory
    // channels (a register's reversal sends neighbours to places that differ in the highest bits only)
    for (int lo = 10, hi = s->n - 1; lo <= hi;) {
        a.order.set(a.order.count++, (uint32_t)lo++);
        if (lo <= hi) a.order.set(a.order.count++, (uint32_t)hi--);
    }
    for (int it = 0; it < kExchangeItems; ++it) a.of_item[it] = exchanged<R>(256u * it, a);
    const uint32_t grid = (uint32_t)std::min<uint64_t>(a.nblocks, 1u << 20);
    return launch_gate(s, &k_exchange<R>, dim3(grid), dim3(256), a);
}

// Amplitude-sized cost of one launch (about 4 us of HBM time) when choosing between one pass for a run
// and a launch per gate.
constexpr uint64_t kLaunchCostAmps = 1ull << 19;

// A swap alone moves half of the amplitudes by either kernel: on states that the caches (256 MiB) hold in good part
// k_exchange is the faster, beyond them the sweep of its own. High bits, us, sweep / k_exchange: complex128 256 MiB
// 87 / 68, 512 MiB 196 / 121, 1 GiB 422 / 441, 4 GiB 1540 / 1642; complex64 512 MiB 195 / 135, 1 GiB 373 / 438, 2 GiB 774 / 832.
constexpr uint64_t kLoneSwapBytes = 512ull << 20;

// Take the next pass's gates out of the held ones and apply them: as one exchange of bits, as one pass over
// the tiles, as one sweep over the amplitudes that share the controls every gate has (diagonals only), or gate by gate
// where that moves fewer amplitudes.
int apply_next(qipgpu_state *s) {
    std::vector<char> taken;
    const Shape shape = shape_of(s);
    const bool exchange = exchanges(shape, s->n, s->held[0]);
    if (exchange) plan_exchange(shape, s->n, s->held, taken);
    else plan_pass(shape, s->n, s->held, taken);
    std::vector<HeldGate> gates;
    size_t w = 0;
    for (size_t i = 0; i < s->held.size(); ++i) {
        if (taken[i]) gates.push_back(s->held[i]);
        else s->held[w++] = s->held[i];
    }
    s->held.resize(w);
    if (exchange && (gates.size() > 1 || s->len * s->amp_bytes <= kLoneSwapBytes))
        return s->dtype == QIPGPU_C128 ? launch_exchange<double>(s, gates) : launch_exchange<float>(s, gates);
    uint64_t common = ~0ull, separate = 0;
    bool diagonal = true;
    for (const HeldGate &g : gates) {
        common &= g.ctrl_mask;
        diagonal = diagonal && g.kind == HeldGate::kDiagonal;
        separate += (s->len >> __builtin_popcountll(g.ctrl_mask)) + kLaunchCostAmps;
    }
    const uint64_t pass = s->len + kLaunchCostAmps;
    const uint64_t chains = (gates.size() + kDiagChainMax - 1) / kDiagChainMax;
    const uint64_t swept = (s->len >> __builtin_popcountll(common)) * chains + chains * kLaunchCostAmps;
    if (gates.size() == 1 || separate < std::min(pass, diagonal ? swept : pass)) {
        for (const HeldGate &g : gates) {
            const int rc = launch_held_gate(s, g);
            if (rc) return rc;
        }
        return QIPGPU_OK;
    }
    if (diagonal && swept < pass) {
        for (size_t i = 0; i < gates.size(); i += kDiagChainMax) {
            const int rc = launch_diag_chain(s, &gates[i], (int)std::min<size_t>(kDiagChainMax, gates.size() - i));
            if (rc) return rc;
        }
        return QIPGPU_OK;
    }
    return s->dtype == QIPGPU_C128 ? launch_pass<double>(s, shape, gates) : launch_pass<float>(s, shape, gates);
}

}  // namespace

namespace qipgpu {

int hold_gate(qipgpu_state *s, const HeldGate &g) {
    // behind a held product only diagonals wait, for a second product that may share a pass with both
    if (s->before.bits &&
        (s->after.bits || g.kind != HeldGate::kDiagonal || s->held.size() == kBetweenMax)) {
        const int rc = apply_held_products(s);
        if (rc) return rc;
    }
    s->held.push_back(g);
    return s->held.size() < kHeldMax ? QIPGPU_OK : apply_next(s);
}

int apply_held_gates(qipgpu_state *s) {
    while (!s->held.empty()) {
        const int rc = apply_next(s);
        if (rc) return rc;
    }
    return QIPGPU_OK;
}

int flush_held(qipgpu_state *s) { return s->before.bits ? apply_held_products(s) : apply_held_gates(s); }

void drop_held(qipgpu_state *s) {
    s->before.bits = s->after.bits = 0;
    s->held.clear();
}

}  // namespace qipgpu
