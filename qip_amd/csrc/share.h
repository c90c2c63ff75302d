// share.h -- how a copy between host and device memory is divided among threads (transfer.hip). Host only.
#pragma once

#include <algorithm>
#include <cstddef>

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

}  // namespace qipgpu
