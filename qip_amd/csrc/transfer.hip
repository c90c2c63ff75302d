// transfer.hip -- copies between the caller's arrays and device memory, through pinned staging memory.
//
// The runtime's own copies of pageable memory pass through its staging buffers a piece at a time, each
// piece waiting for the one before: 17 GB/s out of a 16 MiB state, and 113 us for 256 KiB. Here a copy is
// cut into pieces of 1 MiB on four slots of pinned memory, so that the copy engine works on some while the
// processor copies others, and a copy of 8 MiB and more is shared by up to four threads: what bounds
// a large result is the processor's first touch of the caller's fresh pages (64 MiB: 4.9 ms by one
// thread, 2.3 by four; the link takes 1.2; shares of 1 or 2 MiB and 8 threads measured the same).
// With real feeds crossing as real numbers: a search on a fed 24-qubit register 74.0 -> 23.3 ms, a
// 16-qubit Fourier transform with its 1 MiB input, state and probabilities 369 -> 333 us.
#include <algorithm>
#include <cstring>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

#include "engine.h"
#include "share.h"

namespace qipgpu {

namespace {

constexpr int kSlots = 4;
constexpr size_t kSlotBytes = kPieceBytes;
constexpr size_t kKept = 8;                          // staging buffers kept for later copies (32 MiB)

// Pinned memory that one thread has to itself from take() to give(). A slot may still be read by a copy to
// the device then; whoever uses it next waits for its event.
struct Staging {
    int device = 0;
    char *p = nullptr;
    hipEvent_t ev[kSlots] = {};
    bool busy[kSlots] = {};

    hipError_t wait(int slot) {
        if (!busy[slot]) return hipSuccess;
        const hipError_t e = hipEventSynchronize(ev[slot]);
        if (e == hipSuccess) busy[slot] = false;
        return e;
    }
    hipError_t mark(int slot, hipStream_t st) {
        const hipError_t e = hipEventRecord(ev[slot], st);
        if (e == hipSuccess) busy[slot] = true;
        return e;
    }
};

void destroy(Staging *b) {
    for (int i = 0; i < kSlots; ++i) {
        (void)b->wait(i);
        if (b->ev[i]) (void)hipEventDestroy(b->ev[i]);
    }
    if (b->p) (void)hipHostFree(b->p);
    delete b;
}

std::mutex &pool_mutex() {
    static std::mutex *m = new std::mutex;    // alive as long as the process
    return *m;
}

std::vector<Staging *> &pool() {
    static std::vector<Staging *> *v = new std::vector<Staging *>;
    return *v;
}

hipError_t take(int device, Staging **out) {
    {
        std::lock_guard<std::mutex> lock(pool_mutex());
        std::vector<Staging *> &v = pool();
        for (size_t i = v.size(); i-- > 0;)
            if (v[i]->device == device) {
                *out = v[i];
                v.erase(v.begin() + (long)i);
                return hipSuccess;
            }
    }
    Staging *b = new (std::nothrow) Staging;
    if (!b) return hipErrorOutOfMemory;
    b->device = device;
    void *p = nullptr;
    hipError_t e = hipHostMalloc(&p, kSlots * kSlotBytes, hipHostMallocDefault);
    b->p = static_cast<char *>(p);
    for (int i = 0; i < kSlots && e == hipSuccess; ++i) e = hipEventCreateWithFlags(&b->ev[i], hipEventDisableTiming);
    if (e != hipSuccess) {
        destroy(b);
        return e;
    }
    *out = b;
    return hipSuccess;
}

void give(Staging *b) {
    {
        std::lock_guard<std::mutex> lock(pool_mutex());
        std::vector<Staging *> &v = pool();
        if (v.size() < kKept && v.capacity() >= kKept) {
            v.push_back(b);
            return;
        }
        if (v.capacity() < kKept) {
            try {
                v.reserve(kKept);
                v.push_back(b);
                return;
            } catch (...) {
            }
        }
    }
    destroy(b);
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

    void run() {
        Staging *b = nullptr;
        if ((rc = take(device, &b)) != hipSuccess) return;
        rc = out ? copy_out(b) : copy_in(b);
        // a copy that failed half way may have left slots in flight without an event
        if (rc != hipSuccess) (void)hipStreamSynchronize(st);
        give(b);
    }
    size_t piece(size_t i) const { return std::min(kSlotBytes, bytes - i * kSlotBytes); }
    hipError_t fetch(Staging *b, size_t i) {
        const int slot = (int)(i % kSlots);
        hipError_t e = b->wait(slot);
        if (e == hipSuccess)
            e = hipMemcpyAsync(b->p + slot * kSlotBytes, dev + i * kSlotBytes, piece(i), hipMemcpyDeviceToHost, st);
        return e == hipSuccess ? b->mark(slot, st) : e;
    }
    hipError_t copy_out(Staging *b) {
        const size_t n = (bytes + kSlotBytes - 1) / kSlotBytes;
        hipError_t e = hipSuccess;
        for (size_t i = 0; i < std::min<size_t>(n, kSlots) && e == hipSuccess; ++i) e = fetch(b, i);
        for (size_t i = 0; i < n && e == hipSuccess; ++i) {
            const int slot = (int)(i % kSlots);
            if ((e = b->wait(slot)) != hipSuccess) break;
            std::memcpy(host + i * kSlotBytes, b->p + slot * kSlotBytes, piece(i));
            if (i + kSlots < n) e = fetch(b, i + kSlots);
        }
        return e;
    }
    hipError_t copy_in(Staging *b) {
        const size_t n = (bytes + kSlotBytes - 1) / kSlotBytes;
        hipError_t e = hipSuccess;
        for (size_t i = 0; i < n && e == hipSuccess; ++i) {
            const int slot = (int)(i % kSlots);
            if ((e = b->wait(slot)) != hipSuccess) break;
            std::memcpy(b->p + slot * kSlotBytes, host + i * kSlotBytes, piece(i));
            e = hipMemcpyAsync(dev + i * kSlotBytes, b->p + slot * kSlotBytes, piece(i), hipMemcpyHostToDevice, st);
            if (e == hipSuccess) e = b->mark(slot, st);
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
    const Shares shares = shares_of(bytes);
    const int parts = shares.count;
    Part part[kCopyThreads];
    std::thread thread[kCopyThreads];
    for (int i = 0; i < parts; ++i) {
        const size_t at = i * shares.each;
        Part &p = part[i];
        p.st = st;
        p.device = device;
        p.host = host + at;
        p.dev = dev + at;
        p.bytes = std::min(shares.each, bytes - at);
        p.out = out;
    }
    for (int i = 1; i < parts; ++i) {
        Part *p = &part[i];
        try {
            thread[i] = std::thread([p] {
                p->rc = hipSetDevice(p->device);
                if (p->rc == hipSuccess) p->run();
            });
        } catch (const std::system_error &) {
            // no thread to be had: this one takes the stretch too, below
        }
    }
    part[0].run();
    hipError_t e = part[0].rc;
    for (int i = 1; i < parts; ++i) {
        if (thread[i].joinable()) thread[i].join();
        else part[i].run();
        if (e == hipSuccess) e = part[i].rc;
    }
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
