// pool.cpp — device memory of the library: hipMalloc / hipFree behind a bounded per-device cache.
//
// A call that builds an octree, uploads queries or makes a mesh takes and gives back up to thirty
// buffers, and mapping and unmapping them costs more than the kernels between (an octree of 4M points
// with a first projection: 3.4 ms of kernels in 20 to 43 ms).  Freed blocks are therefore kept, up to
// 1/64 of the device's memory (4.5 GiB of 288), and handed out again to requests of the same size class
// (classes an eighth of an octave apart, so at most an eighth is unused); the oldest go back to the
// device when the bound is passed, all of them when an allocation of the library fails or the caller asks
// (mlod_memory_trim).  Larger blocks go straight to hipMalloc and hipFree.
//
// Safe from any thread.  dev_free waits for the device before a block can be handed out again, as
// hipFree does, so a block never passes to another stream or thread while work still uses it.  Nothing
// here throws: where the host has no memory for the books, a block is freed or the allocation fails.
#include <hip/hip_runtime.h>

#include <cstddef>
#include <list>
#include <mutex>
#include <new>
#include <unordered_map>
#include <vector>

#include "mlod_internal.h"

namespace mlod {
namespace {

struct Block {
  void* p;
  size_t bytes;
};
struct Device {
  size_t bound = 0, held = 0;
  std::list<Block> cached;  // oldest first
};
struct Pool {
  std::mutex mu;
  std::vector<Device> dev;
  struct Live {
    size_t bytes;
    int device;
  };
  std::unordered_map<void*, Live> live;
};

// Never destroyed: the runtime may be gone before a static destructor runs.
Pool& pool() {
  static Pool* p = new Pool;
  return *p;
}

size_t size_class(size_t n) {
  if (n < 4096) return 4096;
  int top = 63 - __builtin_clzll((unsigned long long)n);
  const size_t step = (size_t)1 << (top - 3);
  return (n + step - 1) / step * step;
}

void free_blocks(const std::list<Block>& back) {
  for (const Block& b : back) (void)hipFree(b.p);
}

// Gives every cached block of a device back to it (all devices: dev < 0).
void give_back(int dev) {
  std::list<Block> back;
  Pool& P = pool();
  {
    std::lock_guard<std::mutex> lk(P.mu);
    for (size_t k = 0; k < P.dev.size(); ++k) {
      if (dev >= 0 && (size_t)dev != k) continue;
      back.splice(back.end(), P.dev[k].cached);
      P.dev[k].held = 0;
    }
  }
  free_blocks(back);
}

// hipMalloc, and once more with the cache given back.
hipError_t raw_malloc(void** p, size_t bytes, size_t bytesRetry, size_t* got, int dev) {
  hipError_t e = hipMalloc(p, bytes);
  *got = bytes;
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    give_back(dev);
    e = hipMalloc(p, bytesRetry);
    *got = bytesRetry;
  }
  if (e != hipSuccess) {
    (void)hipGetLastError();  // (not left for the next launch's check)
    *p = nullptr;
  }
  return e;
}

hipError_t take(void** p, size_t bytes) {
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev)) return e;
  Pool& P = pool();
  size_t want = size_class(bytes);
  {
    std::lock_guard<std::mutex> lk(P.mu);
    if ((size_t)dev >= P.dev.size()) P.dev.resize(dev + 1);
    Device& d = P.dev[dev];
    if (!d.bound) {
      size_t freeB = 0, total = 0;
      if (hipError_t e = hipMemGetInfo(&freeB, &total)) return e;
      d.bound = total / 64;
    }
    if (want > d.bound / 2) {
      want = bytes;
    } else {
      for (auto it = d.cached.begin(); it != d.cached.end(); ++it) {
        if (it->bytes != want) continue;
        P.live[it->p] = Pool::Live{want, dev};
        *p = it->p;
        d.held -= it->bytes;
        d.cached.erase(it);
        return hipSuccess;
      }
    }
  }
  size_t got = 0;
  if (hipError_t e = raw_malloc(p, want, bytes, &got, dev)) return e;
  try {
    std::lock_guard<std::mutex> lk(P.mu);
    P.live[*p] = Pool::Live{got, dev};
  } catch (...) {
    (void)hipFree(*p);
    *p = nullptr;
    throw;
  }
  return hipSuccess;
}

}  // namespace

hipError_t dev_malloc_bytes(void** p, size_t bytes) {
  *p = nullptr;
  try {
    return take(p, bytes);
  } catch (const std::bad_alloc&) {
    return hipErrorOutOfMemory;
  }
}

hipError_t dev_malloc_raw(void** p, size_t bytes) {
  *p = nullptr;
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev)) return e;
  size_t got = 0;
  try {
    return raw_malloc(p, bytes, bytes, &got, dev);
  } catch (const std::bad_alloc&) {  // (the cache itself)
    return hipErrorOutOfMemory;
  }
}

size_t dev_block_bytes(void* p) {
  Pool& P = pool();
  std::lock_guard<std::mutex> lk(P.mu);
  auto it = P.live.find(p);
  return it == P.live.end() ? 0 : it->second.bytes;
}

void dev_trim() { give_back(-1); }

void dev_free(void* const* ps, size_t n) {
  int cur = 0;
  (void)hipGetDevice(&cur);
  int synced = -1;  // the device last waited for
  for (size_t i = 0; i < n; ++i) {
    void* p = ps[i];
    if (!p) continue;
    Pool& P = pool();
    Pool::Live lv{0, cur};
    bool known = false;
    {
      std::lock_guard<std::mutex> lk(P.mu);
      auto it = P.live.find(p);
      if (it != P.live.end()) {
        lv = it->second;
        known = true;
        P.live.erase(it);
      }
    }
    if (!known) {
      (void)hipFree(p);
      continue;
    }
    if (lv.device != synced) {
      if (lv.device != cur) (void)hipSetDevice(lv.device);
      const hipError_t e = hipDeviceSynchronize();
      if (lv.device != cur) (void)hipSetDevice(cur);
      if (e != hipSuccess) {  // the block may still be in use: it is not handed out again
        (void)hipFree(p);
        continue;
      }
      synced = lv.device;
    }
    std::list<Block> back;
    {
      std::lock_guard<std::mutex> lk(P.mu);
      Device& d = P.dev[lv.device];
      bool kept = false;
      if (lv.bytes <= d.bound / 2 && lv.bytes == size_class(lv.bytes)) {
        try {
          d.cached.push_back(Block{p, lv.bytes});
          kept = true;
        } catch (const std::bad_alloc&) {
        }
      }
      if (kept) {
        p = nullptr;
        d.held += lv.bytes;
        while (d.held > d.bound) {
          d.held -= d.cached.front().bytes;
          back.splice(back.end(), d.cached, d.cached.begin());
        }
      }
    }
    if (p) (void)hipFree(p);
    free_blocks(back);
  }
}

}  // namespace mlod

extern "C" int mlod_memory_trim(void) {
  mlod::dev_trim();
  return MLOD_OK;
}
