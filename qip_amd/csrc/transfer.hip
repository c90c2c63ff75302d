// transfer.hip -- copies between the caller's arrays and device memory, through pinned staging memory.
//
// The runtime's own copies of pageable memory pass through its staging buffers a piece at a time, each
// piece waiting for the one before: 17 GB/s out of a 16 MiB state. Here a copy is
// cut into pieces of 1 MiB on four slots of pinned memory, so that the link works on some while the
// processor copies others, and a copy of 8 MiB and more is shared by up to four threads: what bounds
// a large result is the processor's first touch of the caller's fresh pages (64 MiB: 4.9 ms by one
// thread, 2.3 by four; the link takes 1.2; shares of 1 or 2 MiB and 8 threads measured the same).
// With real feeds crossing as real numbers: a search on a fed 24-qubit register 74.0 -> 23.3 ms, a
// 16-qubit Fourier transform with its 1 MiB input, state and probabilities 369 -> 333 us.
// A call, us, by the runtime's copies and here: reads of 64 KiB 13 / 13, 1 MiB 62 / 61, 16 MiB 920 / 475; uploads of
// 64 KiB 14 / 7 (18 until they are there), 1 MiB 56 / 33 (60), 16 MiB 464 / 227 (455).
#include <algorithm>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "engine.h"
#include "share.h"

namespace qipgpu {

// Words between a slot and device memory, the host's with system scope: no cache holds an older copy of a slot that
// is used again, and what is written there does not stay in one. In the state's own queue: a transfer by the copy
// engines waits for the queue's kernels and they for it, some 10 us a piece (uploads waited for, us, copy engine ->
// here: 64 KiB 20 -> 17, 1 MiB 64 -> 60, 4 MiB 170 -> 139, 16 MiB 600 -> 455), and of several pieces of a read from
// two threads each took 150 us in some processes (8 MiB 1330 us, 450 to 510 so; 16 MiB 600 -> 475). 16, 32
// and 64 workgroups upload 1 MiB in 80, 62 and 60 us.
constexpr uint32_t kMoveBlocks = 64;

template <bool OUT>
__global__ __launch_bounds__(256) void k_move(const uint64_t *__restrict__ src, uint64_t *__restrict__ dst, uint32_t words) {
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < words; i += gridDim.x * 256) {
        if constexpr (OUT) __hip_atomic_store(dst + i, src[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        else dst[i] = __hip_atomic_load(src + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// The words of a short upload as kernel arguments: no slot, and no event that holds up the kernel behind it
// (a small addition 22 -> 17 us with its wait).
constexpr uint32_t kPayloadWords = 480;
struct Payload {
    uint64_t w[kPayloadWords];
};

__global__ __launch_bounds__(256) void k_payload(uint64_t *dst, uint32_t words, const Payload p) {
    for (uint32_t i = threadIdx.x; i < words; i += 256) dst[i] = p.w[i];
}

namespace {

bool in_words(const void *p, size_t bytes) { return !((reinterpret_cast<uintptr_t>(p) | bytes) & 7u); }

constexpr int kSlots = 4;           // pieces that a thread has on their way
constexpr int kSlotsMade = 32;      // slots a device gets at most, 32 MiB, kept for later copies

// Pinned memory for one piece, one thread's from take() to give(). `busy`: the copy that `done` marks may
// still use it. A slot is given back while an upload reads it, so that the caller need not wait for the
// queue, and is taken again only once that is over: a copy never waits for another queue's work.
struct Slot {
    int device = 0;
    char *p = nullptr;
    hipEvent_t done = nullptr;
    bool busy = false;

    hipError_t wait() {
        if (!busy) return hipSuccess;
        const hipError_t e = hipEventSynchronize(done);
        if (e == hipSuccess) busy = false;
        return e;
    }
    hipError_t mark(hipStream_t st) {
        const hipError_t e = hipEventRecord(done, st);
        if (e == hipSuccess) busy = true;
        return e;
    }
    bool free() {
        if (busy && hipEventQuery(done) == hipSuccess) busy = false;
        if (busy) (void)hipGetLastError();      // "not ready" is no error of the next launch
        return !busy;
    }
};

struct Pool {
    std::mutex mutex;
    std::vector<Slot *> idle;       // the one given back longest ago first; room for every slot made
    std::vector<int> made;          // per device
};

Pool &pool() {
    static Pool *p = new Pool;      // alive as long as the process
    return *p;
}

// kSlots more slots for `device`, one of them returned, the others in the pool; null where it has its share or there is
// no memory.
Slot *make(int device) {
    Pool &pl = pool();
    try {
        std::lock_guard<std::mutex> lock(pl.mutex);
        if ((size_t)device >= pl.made.size()) pl.made.resize(device + 1, 0);
        if (pl.made[device] + kSlots > kSlotsMade) return nullptr;
        size_t all = kSlots;
        for (int m : pl.made) all += m;
        pl.idle.reserve(all);
        pl.made[device] += kSlots;
    } catch (const std::bad_alloc &) {
        return nullptr;
    }
    Slot *slot = new (std::nothrow) Slot[kSlots];       // never freed
    void *p = nullptr;
    bool ok = slot && hipHostMalloc(&p, kSlots * kPieceBytes, hipHostMallocDefault) == hipSuccess;
    for (int i = 0; i < kSlots && ok; ++i) {
        slot[i].device = device;
        slot[i].p = static_cast<char *>(p) + i * kPieceBytes;
        ok = hipEventCreateWithFlags(&slot[i].done, hipEventDisableTiming) == hipSuccess;
    }
    std::unique_lock<std::mutex> lock(pl.mutex);
    if (ok) {
        for (int i = 1; i < kSlots; ++i) pl.idle.push_back(&slot[i]);
        return slot;
    }
    pl.made[device] -= kSlots;
    lock.unlock();
    (void)hipGetLastError();
    for (int i = 0; slot && i < kSlots; ++i)
        if (slot[i].done) (void)hipEventDestroy(slot[i].done);
    if (p) (void)hipHostFree(p);
    delete[] slot;
    return nullptr;
}

// A slot that nothing uses, or null.
Slot *take(int device) {
    {
        Pool &pl = pool();
        std::lock_guard<std::mutex> lock(pl.mutex);
        for (size_t i = 0; i < pl.idle.size(); ++i) {
            Slot *slot = pl.idle[i];
            if (slot->device != device || !slot->free()) continue;
            pl.idle.erase(pl.idle.begin() + (long)i);
            return slot;
        }
    }
    return make(device);
}

void give(Slot *slot) {
    Pool &pl = pool();
    std::lock_guard<std::mutex> lock(pl.mutex);
    pl.idle.push_back(slot);
}

// The stream's device while a copy runs, the caller's afterwards: events are recorded on their own device's
// streams only.
struct OnDevice {
    int before = 0;
    bool changed = false;
    hipError_t rc;
    explicit OnDevice(int device) {
        rc = hipGetDevice(&before);
        if (rc == hipSuccess && before != device) {
            rc = hipSetDevice(device);
            changed = rc == hipSuccess;
        }
    }
    OnDevice(const OnDevice &) = delete;
    OnDevice &operator=(const OnDevice &) = delete;
    ~OnDevice() {
        if (changed) (void)hipSetDevice(before);
    }
};

struct Part {
    hipStream_t st;
    int device;
    char *host, *dev;
    size_t bytes;
    bool out;           // device to host
    hipError_t rc = hipSuccess;
    Slot *slot[kSlots] = {};
    int slots = 0;      // piece i goes through slot i % slots

    void run() {
        const size_t n = pieces();
        while (slots < kSlots && (size_t)slots < n && (slot[slots] = take(device))) ++slots;
        if (!slots) {
            // every slot is under an upload that waits for its queue: the runtime's own copy, and this queue's end
            rc = out ? hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st)
                     : hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, st);
            if (rc == hipSuccess) rc = hipStreamSynchronize(st);
            return;
        }
        rc = out ? copy_out(n) : copy_in(n);
        if (rc != hipSuccess) {
            // a copy that failed half way may have left slots in flight without an event
            (void)hipStreamSynchronize(st);
            for (int i = 0; i < slots; ++i) slot[i]->busy = false;
        }
        for (int i = 0; i < slots; ++i) give(slot[i]);
    }
    size_t pieces() const { return (bytes + kPieceBytes - 1) / kPieceBytes; }
    size_t piece(size_t i) const { return std::min(kPieceBytes, bytes - i * kPieceBytes); }
    hipError_t move(char *to, const char *from, size_t size) const {
        if (!in_words(to, size) || !in_words(from, 0))
            return hipMemcpyAsync(to, from, size, out ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice, st);
        const uint32_t words = (uint32_t)(size / 8);
        const dim3 grid(std::min((words + 255) / 256, kMoveBlocks));
        if (out) hipLaunchKernelGGL(k_move<true>, grid, dim3(256), 0, st, (const uint64_t *)from, (uint64_t *)to, words);
        else hipLaunchKernelGGL(k_move<false>, grid, dim3(256), 0, st, (const uint64_t *)from, (uint64_t *)to, words);
        return hipGetLastError();
    }
    hipError_t fetch(size_t i) {
        Slot *b = slot[i % slots];
        const hipError_t e = move(b->p, dev + i * kPieceBytes, piece(i));
        return e == hipSuccess ? b->mark(st) : e;
    }
    hipError_t copy_out(size_t n) {
        if (n == 1) {
            // an event would wait in the hardware queue, which other streams share; the stream's end is the copy's own
            // (128 KiB 22 us with an event, 16 so; a state whose queue is empty is read past a busy one)
            hipError_t e = hipMemcpyAsync(slot[0]->p, dev, bytes, hipMemcpyDeviceToHost, st);
            if (e == hipSuccess) e = hipStreamSynchronize(st);
            if (e == hipSuccess) std::memcpy(host, slot[0]->p, bytes);
            return e;
        }
        hipError_t e = hipSuccess;
        for (size_t i = 0; i < std::min<size_t>(n, slots) && e == hipSuccess; ++i) e = fetch(i);
        for (size_t i = 0; i < n && e == hipSuccess; ++i) {
            Slot *b = slot[i % slots];
            if ((e = b->wait()) != hipSuccess) break;
            std::memcpy(host + i * kPieceBytes, b->p, piece(i));
            if (i + slots < n) e = fetch(i + slots);
        }
        return e;
    }
    hipError_t copy_in(size_t n) {
        hipError_t e = hipSuccess;
        for (size_t i = 0; i < n && e == hipSuccess; ++i) {
            Slot *b = slot[i % slots];
            if ((e = b->wait()) != hipSuccess) break;
            std::memcpy(b->p, host + i * kPieceBytes, piece(i));
            e = move(dev + i * kPieceBytes, b->p, piece(i));
            if (e == hipSuccess) e = b->mark(st);
        }
        return e;
    }
};

// The copy, shared by threads that each take a stretch of it and enqueue on the same stream.
int copy(hipStream_t st, char *host, char *dev, size_t bytes, bool out) {
    if (!bytes) return QIPGPU_OK;
    hipDevice_t device = 0;
    QIP_HIP(hipStreamGetDevice(st, &device));
    const OnDevice on(device);
    QIP_HIP(on.rc);
    if (!out && bytes <= sizeof(Payload) && in_words(dev, bytes)) {
        Payload p;
        std::memcpy(p.w, host, bytes);
        hipLaunchKernelGGL(k_payload, dim3(1), dim3(256), 0, st, (uint64_t *)dev, (uint32_t)(bytes / 8), p);
        QIP_LAUNCHED();
        return QIPGPU_OK;
    }
    const Shares shares = shares_of(bytes);
    Part part[kCopyThreads];
    for (int i = 0; i < shares.count; ++i) {
        const size_t at = i * shares.each;
        Part &p = part[i];
        p.st = st;
        p.device = device;
        p.host = host + at;
        p.dev = dev + at;
        p.bytes = std::min(shares.each, bytes - at);
        p.out = out;
    }
    auto work = [&part](int i) {
        part[i].rc = hipSetDevice(part[i].device);
        if (part[i].rc == hipSuccess) part[i].run();
    };
    run_shares<std::thread>(shares.count, work);
    hipError_t e = hipSuccess;
    for (int i = 0; i < shares.count && e == hipSuccess; ++i) e = part[i].rc;
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return set_error(e == hipErrorOutOfMemory ? QIPGPU_ENOMEM : QIPGPU_EHIP, "a copy of %zu bytes %s failed: %s", bytes,
                         out ? "to the host" : "to the device", hipGetErrorString(e));
    }
    return QIPGPU_OK;
}

}  // namespace

int copy_to_host(hipStream_t st, void *host, const void *dev, size_t bytes) {
    return copy(st, static_cast<char *>(host), static_cast<char *>(const_cast<void *>(dev)), bytes, true);
}

int copy_to_device(hipStream_t st, void *dev, const void *host, size_t bytes) {
    return copy(st, static_cast<char *>(const_cast<void *>(host)), static_cast<char *>(dev), bytes, false);
}

}  // namespace qipgpu
