// Device memory and streams of destroyed trees, kept for the next ones.
//
// A build allocates its scratch and the tree's arrays, a destroyed tree gives them back.  The driver unmaps
// freed memory and clears it before it is used again: building 4 million keys, searching them and closing
// the tree took 3 to 10 ms, of which the kernels were 0.7 (the higher figure when the freed memory is still
// being cleared); with blocks and streams kept 0.66 ms.  Blocks are kept instead, at most kPoolKeep bytes per
// device and none above kPoolBlock, and handed out again: to requests of exactly their size, since what a tree
// holds is counted against its budget by the bytes it asked for, or for a call's own scratch to requests of at
// least half their size.  They go back to the driver when an allocation here finds no memory and at
// hm_device_synchronize.
//
// A block is given to the pool only when no work that may use it is in flight (dev_free's `idle`, after a wait
// that succeeded); others go to hipFree, which waits itself.  The wait for the whole device is hipFree's own:
// hipDeviceSynchronize fails while any stream of the process captures, another thread's too, and ends that
// capture.  The allocation and its hipFree take 1.3 us on an idle device.
#include <hip/hip_runtime.h>

#include <mutex>
#include <unordered_map>
#include <vector>

#include "hm_tree.h"

namespace hm {
namespace {

constexpr size_t kPoolKeep = (size_t)512 << 20;
constexpr size_t kPoolBlock = (size_t)256 << 20;
constexpr size_t kPoolStreams = 4;

struct Block {
  size_t bytes;
  int device;
};

struct Pool {
  std::mutex mu;
  std::unordered_map<void*, Block> live;  // blocks in use that may be kept later
  struct Free {
    void* p;
    size_t bytes;
    int device;
  };
  std::vector<Free> idle;  // oldest first; freed by their device's own calls
  struct IdleStream {
    hipStream_t s;
    int device;
  };
  std::vector<IdleStream> streams;
};
Pool& pool() {
  static Pool* p = new Pool();  // never destroyed: trees may outlive static destructors
  return *p;
}

}  // namespace

hipError_t dev_malloc_bytes(void** out, size_t bytes, bool scratch) {
  *out = nullptr;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  Pool& p = pool();
  {
    std::lock_guard<std::mutex> g(p.mu);
    size_t best = p.idle.size();
    for (size_t i = 0; i < p.idle.size(); ++i) {
      const auto& f = p.idle[i];
      if (f.device == dev && (scratch ? f.bytes >= bytes && f.bytes / 2 <= bytes : f.bytes == bytes) &&
          (best == p.idle.size() || f.bytes < p.idle[best].bytes))
        best = i;
    }
    if (best < p.idle.size()) {
      *out = p.idle[best].p;
      try {
        p.live[*out] = Block{p.idle[best].bytes, dev};
      } catch (...) {
      }
      p.idle.erase(p.idle.begin() + (long)best);
      return hipSuccess;
    }
  }
  e = hipMalloc(out, bytes);
  if (e == hipErrorOutOfMemory) {  // give back what is kept and try once more
    (void)hipGetLastError();
    dev_pool_trim();
    e = hipMalloc(out, bytes);
  }
  if (e != hipSuccess) {
    (void)hipGetLastError();  // reported here, not by the next launch
    return e;
  }
  if (bytes <= kPoolBlock) {
    try {
      std::lock_guard<std::mutex> g(p.mu);
      p.live[*out] = Block{bytes, dev};
    } catch (...) {  // no host memory to note it: the block will go back to the driver
    }
  }
  return hipSuccess;
}

hipError_t dev_free(void* ptr, bool idle) {
  if (!ptr) return hipSuccess;
  Pool& p = pool();
  Block b{0, 0};
  {
    std::lock_guard<std::mutex> g(p.mu);
    auto it = p.live.find(ptr);
    if (it != p.live.end()) {
      b = it->second;
      p.live.erase(it);
    }
  }
  int dev = -1;
  if (!idle || !b.bytes || hipGetDevice(&dev) != hipSuccess || dev != b.device) return hipFree(ptr);
  while (true) {  // the oldest blocks make room
    void* oldest = nullptr;
    {
      std::lock_guard<std::mutex> g(p.mu);
      size_t kept = b.bytes, first = p.idle.size();
      for (size_t i = p.idle.size(); i-- > 0;)
        if (p.idle[i].device == dev) {
          kept += p.idle[i].bytes;
          first = i;
        }
      if (kept <= kPoolKeep || first == p.idle.size()) {
        try {
          p.idle.push_back(Pool::Free{ptr, b.bytes, dev});
          ptr = nullptr;
        } catch (...) {
        }
        break;
      }
      oldest = p.idle[first].p;
      p.idle.erase(p.idle.begin() + (long)first);
    }
    (void)hipFree(oldest);
  }
  return ptr ? hipFree(ptr) : hipSuccess;
}

hipError_t dev_wait() {
  void* p = nullptr;
  hipError_t e = hipMalloc(&p, 256);
  if (e == hipSuccess) e = hipFree(p);
  if (e != hipSuccess) (void)hipGetLastError();  // the caller does without the pool
  return e;
}

void dev_pool_trim() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return;
  Pool& p = pool();
  while (true) {
    void* q = nullptr;
    {
      std::lock_guard<std::mutex> g(p.mu);
      for (size_t i = p.idle.size(); i-- > 0;)
        if (p.idle[i].device == dev) {
          q = p.idle[i].p;
          p.idle.erase(p.idle.begin() + (long)i);
          break;
        }
    }
    if (!q) return;
    (void)hipFree(q);
  }
}

hipError_t stream_take(hipStream_t* s) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  Pool& p = pool();
  {
    std::lock_guard<std::mutex> g(p.mu);
    for (size_t i = 0; i < p.streams.size(); ++i)
      if (p.streams[i].device == dev) {
        *s = p.streams[i].s;
        p.streams.erase(p.streams.begin() + (long)i);
        return hipSuccess;
      }
  }
  return hipStreamCreateWithFlags(s, hipStreamNonBlocking);
}

void stream_give(hipStream_t s, int device) {
  Pool& p = pool();
  {
    std::lock_guard<std::mutex> g(p.mu);
    if (p.streams.size() < kPoolStreams) {
      try {
        p.streams.push_back(Pool::IdleStream{s, device});
        return;
      } catch (...) {
      }
    }
  }
  (void)hipStreamDestroy(s);
}

}  // namespace hm
