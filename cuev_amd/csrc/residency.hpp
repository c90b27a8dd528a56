// residency.hpp — which solves' persistent kernels may be on a GPU at once (host code only).
#pragma once

#include <algorithm>
#include <condition_variable>
#include <cstdint>
#include <mutex>

namespace cuev {

// The panel QR and the bulge chase wait for workgroups of their own to become resident, and two of
// their workgroups may not fit on one CU (141 KB of LDS for a panel of 64 columns, 146 KB for a padded
// chase, of 160). Kernels of several solves that each got a part of the CUs and wait for the rest would
// block one another until their bounded waits expire. So a solve takes the CUs that its widest such
// grid needs, one per workgroup, before it queues the band reduction, and gives them back after the
// chase; what does not fit waits on the host, first come first served.
//
// CUs are counted in eighths of the GPU (32 of 256: four of each of the eight XCDs, one of each of an
// XCD's four shader engines), since workgroups are dealt out to these in turn, whether they have room
// or not: a grid of w workgroups puts up to ceil(w / 32) on any one of them.
constexpr int kCuShares = 8;

// shares of a solve of order n at bandwidth b: panels of up to 64 rows a workgroup, a hop of b rows
// each in the chase. One workgroup waits for nobody; a chase of more hops than CUs (two to a CU)
// takes the whole GPU.
inline int cu_shares(int64_t n, int b, int cus) {
    const int64_t rows = std::min(b, 64), wgs = (n + rows - 1) / rows, share = std::max(1, cus / kCuShares);
    if (wgs <= 1) return 0;
    return (int)std::min<int64_t>(kCuShares, (wgs + share - 1) / share);
}

class CuBudget { // of one GPU
  public:
    void take(int shares) {
        std::unique_lock<std::mutex> lk(mu_);
        const uint64_t ticket = next_++;
        cv_.wait(lk, [&] { return ticket == turn_ && used_ + shares <= kCuShares; });
        used_ += shares;
        ++turn_;
        cv_.notify_all();
    }
    void give(int shares) {
        std::lock_guard<std::mutex> lk(mu_);
        used_ -= shares;
        cv_.notify_all();
    }

  private:
    std::mutex mu_;
    std::condition_variable cv_;
    uint64_t next_ = 0, turn_ = 0;
    int used_ = 0;
};

} // namespace cuev
