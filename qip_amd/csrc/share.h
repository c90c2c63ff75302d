// share.h -- how a copy between host and device memory is divided among threads (transfer.hip). Host only.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <memory>

namespace qipgpu {

constexpr size_t kPieceBytes = size_t(1) << 20;
constexpr size_t kThreadBytes = size_t(4) << 20;    // a thread for every 4 MiB
constexpr int kCopyThreads = 4;

// `bytes` as `count` shares of `each` bytes, the last one shorter: whole pieces, as many as there are threads
// at most.
struct Shares {
    int count;
    size_t each;
};

constexpr Shares shares_of(size_t bytes) {
    const size_t threads = std::max<size_t>(1, std::min<size_t>(kCopyThreads, bytes / kThreadBytes));
    const size_t each = std::max((bytes + threads * kPieceBytes - 1) / (threads * kPieceBytes), size_t(1)) * kPieceBytes;
    return Shares{(int)((bytes + each - 1) / each), each};
}

// work(0) .. work(count - 1), each once: the first on the caller, every other one on a helper thread, or on the caller
// too where that helper could not be started or has not begun by the time the caller is free. The caller
// waits for helpers that have begun only: where other threads keep the processors busy (a linear algebra
// library's workers spin for a while after each call) a new thread may wait for milliseconds. Reading 8 MiB
// right after a QR factorisation on 16 threads of 16 processors took 0.8 to 6.8 ms with a helper that was always
// waited for, 0.71 to 0.77 so. A helper that comes late finds its share taken and touches nothing else.
template <typename Thread, typename Work>
void run_shares(int count, Work &work) {
    struct Taken {
        std::atomic<bool> share[kCopyThreads] = {};
    };
    std::shared_ptr<Taken> taken;
    Thread helper[kCopyThreads];
    try {
        if (count > 1) taken = std::make_shared<Taken>();
        for (int i = 1; i < count; ++i)
            helper[i] = Thread([taken, &work, i] {
                if (!taken->share[i].exchange(true)) work(i);
            });
    } catch (...) {
        // no memory or no thread to be had: the caller takes what no helper does
    }
    work(0);
    for (int i = 1; i < count; ++i) {
        if (taken && taken->share[i].exchange(true)) continue;
        work(i);
        if (helper[i].joinable()) helper[i].detach();
    }
    for (int i = 1; i < count; ++i)
        if (helper[i].joinable()) helper[i].join();
}

}  // namespace qipgpu
