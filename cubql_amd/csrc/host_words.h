// host_words.h -- pinned host memory for the few words a build reads back.
//
// A copy to pageable memory waits by itself and goes through a staging buffer
// (three such copies a Morton build: 3000 points 227 us, 182 with one to pinned
// memory), and pinned memory costs more to allocate than a small build takes.  So
// blocks are lent from a list of the process: a build holds one from its first
// readback to its return, threads that build at the same time hold one each, and
// no more than kKept stay allocated when they are given back, however many threads
// there were.
#pragma once
#include <cstddef>
#include <cstdint>

namespace cubql {

class HostWords {
 public:
  static constexpr size_t kWords = 3072;  // of a block (12 KB)
  static constexpr size_t kKept = 16;     // blocks kept for later calls
  HostWords();
  ~HostWords();
  HostWords(const HostWords &) = delete;
  HostWords &operator=(const HostWords &) = delete;
  // nullptr if there was no memory (the error is set)
  uint32_t *get() const { return p_; }

 private:
  uint32_t *p_ = nullptr;
};

}  // namespace cubql
