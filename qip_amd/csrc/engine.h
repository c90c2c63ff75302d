// engine.h -- internal declarations shared by the translation units of libqipgpu.so.
#pragma once

#include <hip/hip_runtime.h>

#include <array>
#include <cstdarg>
#include <cstdint>
#include <complex>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "qipgpu.h"

namespace qipgpu {

// Interleaved complex amplitude, aligned so one amplitude is one vector load
// (16 B dwordx4 for complex128, 8 B dwordx2 for complex64).
template <typename R>
struct __attribute__((aligned(2 * sizeof(R)))) cx {
    R re, im;
};

// Ascending list of state-bit positions at which zero bits are inserted into a compressed
// index (the positions of target and control qubits). Lives in kernel arguments, four 8-bit
// positions per 32-bit word: a loop over them then reads the kernel arguments with scalar loads
// (byte elements would need vector loads, whose waits also drain every load and store the thread
// has in flight), and the arguments stay small (launch cost matters for small states).
struct PosList {
    int32_t count;
    uint32_t w[(QIPGPU_MAX_QUBITS + 3) / 4];

    __host__ __device__ __forceinline__ uint32_t at(int i) const { return (w[i >> 2] >> (8 * (i & 3))) & 0xffu; }
    void set(int i, uint32_t p) { w[i >> 2] = (w[i >> 2] & ~(0xffu << (8 * (i & 3)))) | (p << (8 * (i & 3))); }
};

// Insert a zero bit at each listed position (ascending), turning an enumeration index over
// the free bits into a state index with those bits clear.
__device__ __forceinline__ uint64_t insert_zeros(uint64_t g, const PosList &pl) {
    for (int i = 0; i < pl.count; ++i) {
        const uint32_t p = pl.at(i);
        const uint64_t lo = g & ((1ull << p) - 1ull);
        g = ((g ^ lo) << 1) | lo;
    }
    return g;
}

struct Recorder;   // recorder.hip: gates recorded for online fusion

// Product sweeps (product.hip): every pass keeps the kProductLowBits lowest state bits in its tile and
// takes at most kProductHighPerPass factors above them.
constexpr int kProductLowBits = 4;
constexpr int kProductHighPerPass = 8;

constexpr int kRingSlots = 8;
constexpr size_t kRingSlotBytes = 64 * 64 * 16 + 4096;  // a 64x64 complex128 matrix + offsets

// A small gate held back on the state (qipgpu_state::held) so that a run of them is applied in one pass
// (runs.hip), where the bits of ctrl_mask are all 1: a 2x2 on state bit tpos[0], the exchange of bits
// tpos[0] and tpos[1], or a diagonal on k <= 2 targets, its factor m[j] for j the value of state bits
// tpos[0] (MSB) .. tpos[k-1].
struct HeldGate {
    enum Kind : uint8_t { kSingle, kSwap, kDiagonal };
    uint64_t ctrl_mask;
    cx<double> m[4];
    Kind kind;
    uint8_t k;          // entries of tpos
    uint8_t tpos[2];
};
// Single-qubit operators on distinct state bits held back as one operator (product.hip): factor m[p] on
// state bit p, for every bit of `bits`.
struct HeldProduct {
    uint64_t bits = 0;
    std::vector<std::array<cx<double>, 4>> m;   // row-major 2x2 per state bit
};
// Diagonals that may stand between two held products (k_product_pair's arguments).
constexpr size_t kBetweenMax = 4;
// Gates held back at most: with this many, the next pass is applied. Enough for a pass to see the
// two-qubit gates that follow a layer of single-qubit gates on 30 qubits.
constexpr size_t kHeldMax = 64;
// Diagonals of one sweep over the amplitudes that share the controls all of them have (k_diag_chain).
constexpr int kDiagChainMax = 16;

}  // namespace qipgpu

struct qipgpu_state {
    int32_t n = 0;
    int32_t dtype = 0;
    int32_t device = 0;
    uint64_t len = 0;          // 2^n amplitudes
    size_t amp_bytes = 0;      // bytes per amplitude
    void *amps = nullptr;
    hipStream_t stream = nullptr;
    // growable device scratch (reduction partials, staging)
    void *scratch = nullptr;
    size_t scratch_cap = 0;
    // device staging ring for operators too large for kernel arguments
    void *d_ring = nullptr;
    void *h_ring = nullptr;      // pinned
    void *h_ring_dev = nullptr;  // the pinned ring as the device addresses it
    hipEvent_t ring_ev[qipgpu::kRingSlots] = {};
    bool ring_used[qipgpu::kRingSlots] = {};
    int ring_next = 0;
    // fused path: d_fused[0] = renormalisation factor and d_fused[1] = norm of the last block (written
    // when the state is settled or the norm asked for), then two arrays of `fused_partials` per-workgroup
    // norm partials used by consecutive blocks in turn. A block's output stays unnormalised until the
    // next block or a settle applies 1/sqrt(sum of its partials): fused_prev_count > 0 marks that
    // pending factor, with the partials in array fused_parity ^ 1.
    double *d_fused = nullptr;
    size_t fused_partials = 0;
    uint32_t fused_prev_count = 0;
    int fused_parity = 0;
    // fused path operator staging (split BF16 planes), device
    void *d_fmat = nullptr;
    size_t d_fmat_bytes = 0;
    // dense operators on 7..12 targets (dense.hip launch_gemm): the operator and its offsets pass
    // through pinned host memory to a device buffer on the state's queue (gemm_ev marks the last
    // copy out of the pinned buffer), and the compact temporary is kept while it is small
    void *h_gemm_op = nullptr;   // pinned
    size_t h_gemm_op_bytes = 0;
    void *d_gemm_op = nullptr;
    size_t d_gemm_op_bytes = 0;
    hipEvent_t gemm_ev = nullptr;
    void *gemm_tmp = nullptr;
    size_t gemm_tmp_bytes = 0;
    // a gate graph being recorded (qipgpu_capture_begin .. qipgpu_capture_end): gate kernels whose
    // operands are all kernel arguments become graph nodes, each after the previous one, instead of
    // launches (launch_gate); any other operation is refused and marks the recording refused
    bool capturing = false;
    bool capture_refused = false;
    hipGraph_t rec_graph = nullptr;
    hipGraphNode_t rec_last = nullptr;
    // gates recorded for online fusion and not launched yet (complex64 states)
    qipgpu::Recorder *recorder = nullptr;
    // held back, in program order: a product, gates, a product (flush_held applies them before anything
    // else touches the state). Gates held behind `before` are diagonals, at most kBetweenMax; `after` is
    // held only behind both.
    qipgpu::HeldProduct before;
    std::vector<qipgpu::HeldGate> held;
    qipgpu::HeldProduct after;
};

namespace qipgpu {

int set_error(int code, const char *fmt, ...);

#define QIP_HIP(expr)                                                                      \
    do {                                                                                   \
        hipError_t e_ = (expr);                                                            \
        if (e_ != hipSuccess)                                                              \
            return ::qipgpu::set_error(QIPGPU_EHIP, "%s failed: %s", #expr,                \
                                       hipGetErrorString(e_));                             \
    } while (0)

#define QIP_LAUNCHED()                                                                     \
    do {                                                                                   \
        hipError_t e_ = hipGetLastError();                                                 \
        if (e_ != hipSuccess)                                                              \
            return ::qipgpu::set_error(QIPGPU_EHIP, "kernel launch failed: %s",            \
                                       hipGetErrorString(e_));                             \
    } while (0)

// A device buffer for one call, freed on every exit path once the state's stream is done with it.
struct TempBuffer {
    hipStream_t stream;
    void *p = nullptr;
    explicit TempBuffer(hipStream_t st) : stream(st) {}
    TempBuffer(const TempBuffer &) = delete;
    TempBuffer &operator=(const TempBuffer &) = delete;
    hipError_t alloc(size_t bytes) { return hipMalloc(&p, bytes); }
    // hand the buffer over (it is not freed here any more)
    void *release() {
        void *q = p;
        p = nullptr;
        return q;
    }
    ~TempBuffer() {
        if (p) {
            (void)hipStreamSynchronize(stream);
            (void)hipFree(p);
        }
    }
};

// Make sure s->scratch holds at least `bytes`.
int ensure_scratch(qipgpu_state *s, size_t bytes);
// Copies between the caller's memory and that of `st`'s device through pinned staging memory (transfer.hip),
// in `st`'s order: to the host, complete on return; to the device, enqueued, the host memory free on
// return.
int copy_to_host(hipStream_t st, void *host, const void *dev, size_t bytes);
int copy_to_device(hipStream_t st, void *dev, const void *host, size_t bytes);
// Compute units of the current device, queried once per device (persistent grids are sized by it).
int device_cus();
// Validate a list of qubit indices against n (range, distinctness); returns QIPGPU_OK or EINVAL.
int check_qubits(const qipgpu_state *s, int32_t k, const int32_t *q, const char *what);
// Reserve a staging ring slot, copy `bytes` from `src` to the device, return device pointer.
int ring_upload(qipgpu_state *s, const void *src, size_t bytes, void **dev);
// Hold a small gate back on the state; with kHeldMax held, the next pass of them is applied (runs.hip).
int hold_gate(qipgpu_state *s, const HeldGate &g);
// Apply what is held back on the state (runs.hip): every entry point that touches the state does so
// first, through flush_recorded. drop_held forgets it (the state is overwritten).
int flush_held(qipgpu_state *s);
void drop_held(qipgpu_state *s);
// The gates of s->held alone, in passes (runs.hip).
int apply_held_gates(qipgpu_state *s);
// s->before, s->held and s->after, where a product is held (product.hip).
int apply_held_products(qipgpu_state *s);
// One held gate by a sweep of its own; up to kDiagChainMax diagonals, in order, by one sweep over the
// amplitudes that share the controls all of them have (engine.hip).
int launch_held_gate(qipgpu_state *s, const HeldGate &g);
int launch_diag_chain(qipgpu_state *s, const HeldGate *g, int count);
// Launch every recorded gate (recorder.hip), after what is held back; they may themselves be held back.
// Nothing while the recorder itself is launching.
int launch_recorded(qipgpu_state *s);
// launch_recorded, then apply what is held back.
int flush_recorded(qipgpu_state *s);
// While s is capturing: mark the capture refused and return QIPGPU_EUNSUP naming `what`.
int refuse_in_capture(qipgpu_state *s, const char *what);
#define QIP_NOT_CAPTURING(s, what)                                                        \
    do {                                                                                   \
        if ((s)->capturing) return ::qipgpu::refuse_in_capture((s), (what));               \
    } while (0)

// A gate kernel whose operands all travel as kernel arguments: launched on the state's queue, or,
// while a gate graph is recorded, added to it after the previously recorded kernel (the node copies
// the arguments).
template <typename... P>
int launch_gate(qipgpu_state *s, void (*kernel)(P...), dim3 grid, dim3 block, P... args) {
    if (!s->capturing) {
        hipLaunchKernelGGL(kernel, grid, block, 0, s->stream, args...);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return set_error(QIPGPU_EHIP, "kernel launch failed: %s", hipGetErrorString(e));
        return QIPGPU_OK;
    }
    void *params[] = {static_cast<void *>(&args)...};
    hipKernelNodeParams p;
    std::memset(&p, 0, sizeof(p));
    p.func = reinterpret_cast<void *>(kernel);
    p.gridDim = grid;
    p.blockDim = block;
    p.sharedMemBytes = 0;
    p.kernelParams = params;
    p.extra = nullptr;
    hipGraphNode_t node = nullptr;
    const hipGraphNode_t prev = s->rec_last;
    const hipError_t e = hipGraphAddKernelNode(&node, s->rec_graph, prev ? &prev : nullptr, prev ? 1 : 0, &p);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        s->capture_refused = true;
        return set_error(QIPGPU_EHIP, "hipGraphAddKernelNode failed: %s", hipGetErrorString(e));
    }
    s->rec_last = node;
    return QIPGPU_OK;
}
// Drop recorded gates (the state is about to be overwritten) / free the recorder.
void recorder_discard(qipgpu_state *s);
void recorder_free(qipgpu_state *s);
// Gates recorded and not launched yet.
int64_t recorder_pending(const qipgpu_state *s);
// Launch recorded gates, then apply a fused path's pending renormalisation factor: before the state
// is read or written from the host.
int settle(qipgpu_state *s);
// Sum of |psi|^2 in FP64, result left on the device at `dst` (enqueued on s->stream).
int norm_to_device(qipgpu_state *s, double *dst);
// Dense operator U (2^K x 2^K, row-major) on 4 <= K <= QIPGPU_MAX_DENSE targets at state bits `tbits`
// (first = MSB of U's index), where the bits of ctrl_mask are 1; `allpos` = control and target
// bits (dense.hip).
int dense_large(qipgpu_state *s, const std::vector<int> &tbits, uint64_t ctrl_mask, const std::vector<int> &allpos,
                const std::complex<double> *U);
// Diagonal d (2^K entries) on 7 <= K <= QIPGPU_MAX_DENSE targets, where the bits of ctrl_mask are 1;
// `cpos` = control bits (dense.hip).
int diag_large(qipgpu_state *s, const std::vector<int> &tbits, uint64_t ctrl_mask, const std::vector<int> &cpos,
               const std::complex<double> *d);

}  // namespace qipgpu
