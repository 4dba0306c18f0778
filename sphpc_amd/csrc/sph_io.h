// Chunks of a state transfer over a few host threads.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <thread>

namespace sph {

constexpr int kIoThreads = 4;

// Runs work(k) for every chunk k of `chunks`, on this thread and up to threads - 1
// (kIoThreads - 1, chunks - 1) more; without them where none can be started.
// `mine`, if given, is called on this thread between its own chunks.
template <class Work, class Mine>
static void io_chunks(size_t chunks, int threads, Work work, Mine mine) {
  std::atomic<size_t> next{0};
  auto take = [&]() {
    const size_t k = next.fetch_add(1);
    if (k < chunks) work(k);
    return k < chunks;
  };
  std::thread helpers[kIoThreads - 1];
  const size_t most = std::min<size_t>(std::min(threads, kIoThreads), chunks);
  for (size_t t = 0; t + 1 < most; ++t) {
    // no thread (std::system_error), or no memory for one (std::bad_alloc): nothing
    // may pass on to the C caller, or past helpers that already run
    try {
      helpers[t] = std::thread([&]() {
        while (take()) {
        }
      });
    } catch (...) {
      break;
    }
  }
  while (take()) mine();
  for (std::thread &h : helpers)
    if (h.joinable()) h.join();
  mine();
}

}  // namespace sph
