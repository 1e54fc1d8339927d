// A word of pinned host memory that a kernel writes and the calling thread waits for: no copy behind the
// kernel, and the thread looks at the word itself instead of waiting for the stream.  Words go round in a pool,
// one per call in progress at most; one whose kernel may still write stays out of it.
//
// The memory is coherent, whatever the environment says of pinned memory without that flag (HIP_HOST_COHERENT):
// the word is looked at while the kernel runs, and goes on to the next call as soon as it is there.  In memory
// that a kernel's caches may hold, the value would be seen only at the kernel's end, and its write-back could
// land in the next call's wait.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <mutex>
#include <thread>
#include <vector>

namespace cummhip {

constexpr uint32_t kNotYet = 0xFFFFFFFFu;

struct HostWord {
  uint32_t *at = nullptr;
  bool settled = false;

  static std::mutex &lock() {
    static std::mutex m;
    return m;
  }
  static std::vector<uint32_t *> &pool() {
    static std::vector<uint32_t *> words;
    return words;
  }

  hipError_t take() {
    {
      std::lock_guard<std::mutex> guard(lock());
      if (!pool().empty()) {
        at = pool().back();
        pool().pop_back();
      }
    }
    if (at == nullptr) {
      void *host = nullptr;
      const hipError_t e = hipHostMalloc(&host, 64, hipHostMallocPortable | hipHostMallocCoherent);
      if (e != hipSuccess) return e;
      at = reinterpret_cast<uint32_t *>(host);
    }
    __atomic_store_n(at, kNotYet, __ATOMIC_RELEASE);
    return hipSuccess;
  }
  // until the word is there; the stream is looked at now and then, for errors and for a launch that has ended
  hipError_t wait(hipStream_t s, uint32_t *value) {
    for (unsigned spin = 1;; ++spin) {
      uint32_t v = __atomic_load_n(at, __ATOMIC_ACQUIRE);
      if (v == kNotYet && spin % 512 == 0) {
        const hipError_t e = hipStreamQuery(s);
        if (e != hipSuccess && e != hipErrorNotReady) return e;
        (void)hipGetLastError();      // ("not ready" is no error of this call)
        if (e == hipErrorNotReady) {
          if (spin >= 1u << 16) std::this_thread::yield();
          continue;
        }
        v = __atomic_load_n(at, __ATOMIC_ACQUIRE);
      } else if (v == kNotYet) {
        __builtin_ia32_pause();
        continue;
      }
      settled = true;
      *value = v;
      return hipSuccess;
    }
  }
  ~HostWord() {
    if (!settled) return;
    std::lock_guard<std::mutex> guard(lock());
    pool().push_back(at);
  }
};

}  // namespace cummhip
