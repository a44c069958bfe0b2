// The device memory, pinned read-back buffer and events of one PageRank or
// adjoint run, kept with the matrix between runs: allocating, clearing and
// freeing them took 0.2 ms of a call on 5,003 nodes and 9 ms of one on 2^24.
//
// A run leases a RunSpace for itself alone and gives it back once its stream
// has drained, so runs on other streams and threads never share one; a run
// that fails does not give it back (the memory is freed instead).  At most
// kIdleSpaces are kept per matrix and kIdleBytes over all matrices (the one
// given back longest ago goes first), and they go when the matrix's device data
// goes (destruction or a mutating call) or when an allocation of this library
// finds no memory (drop_idle_memory, common.hpp).
#pragma once

#include <cstddef>
#include <memory>
#include <vector>

#include "common.hpp"

namespace tbsla {
namespace hip {

constexpr std::size_t kIdleSpaces = 2;  // a forward's and a backward's
// 2^24 nodes of 8 edges take 0.8 GB a run, so graphs of up to 2^28 keep theirs;
// 6% of the card's memory
constexpr std::size_t kIdleBytes = std::size_t(16) << 30;
constexpr std::size_t kReadBackBytes = 1024;

struct RunSpace {
  DevBuf mem;                                // not cleared between runs
  void *pinned = nullptr;                    // kReadBackBytes of pinned host memory
  hipEvent_t timing[2] = {nullptr, nullptr}; // start and end of a run's loop
  hipEvent_t ready[2] = {nullptr, nullptr};  // read-backs in flight
  RunSpace() {
    try {
      TBSLA_HIP_CHECK(hipHostMalloc(&pinned, kReadBackBytes, hipHostMallocDefault));
      for (int k = 0; k < 2; k++) {
        TBSLA_HIP_CHECK(hipEventCreate(&timing[k]));
        TBSLA_HIP_CHECK(hipEventCreateWithFlags(&ready[k], hipEventDisableTiming));
      }
    } catch (...) {
      clear();
      throw;
    }
  }
  ~RunSpace() { clear(); }
  RunSpace(const RunSpace &) = delete;
  RunSpace &operator=(const RunSpace &) = delete;

 private:
  void clear() {
    if (pinned) (void)hipHostFree(pinned);
    for (int k = 0; k < 2; k++) {
      if (timing[k]) (void)hipEventDestroy(timing[k]);
      if (ready[k]) (void)hipEventDestroy(ready[k]);
    }
  }
};

// The run memory of one matrix.
class RunSpaces {
 public:
  RunSpaces() = default;
  ~RunSpaces();
  RunSpaces(const RunSpaces &) = delete;
  RunSpaces &operator=(const RunSpaces &) = delete;
  // the smallest idle space of at least `bytes`, or a new one
  std::unique_ptr<RunSpace> take(std::size_t bytes);
  void give(std::unique_ptr<RunSpace> s);
};

// One device buffer of a run: a slice of its memory.
struct WsBuf {
  std::size_t off = 0;
  void *p = nullptr;
  template <class T>
  T *as() const {
    return static_cast<T *>(p);
  }
};

// Lays a run's buffers out as consecutive 256-byte-aligned slices: alloc()
// for each, then place() at their memory.
class RunLayout {
 public:
  void alloc(WsBuf &b, std::size_t bytes) {
    b.off = used_;
    used_ += (std::max<std::size_t>(bytes, 1) + 255) & ~std::size_t(255);
    bufs_.push_back(&b);
  }
  std::size_t bytes() const { return used_; }
  void place(void *base) {
    for (WsBuf *b : bufs_) b->p = static_cast<unsigned char *>(base) + b->off;
  }

 private:
  std::vector<WsBuf *> bufs_;
  std::size_t used_ = 0;
};

}  // namespace hip
}  // namespace tbsla
