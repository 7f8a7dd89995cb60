// The device block cache (mlodsurfaces_amd/csrc/pool.cpp) over a counting stand-in for the HIP runtime: two devices of a
// settable size, allocations that fail when the device is full or when told to, host allocations that fail when told to.
#include <cassert>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <new>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include "hip/hip_runtime.h"

static std::mutex gMu;
static thread_local int gDev = 0;
static size_t gTotal[2] = {64ull << 20, 64ull << 20}, gUsed[2] = {0, 0};
static std::map<void*, std::pair<size_t, int>> gMem;
static int gMallocs = 0, gFrees = 0, gFailMallocs = 0;
static bool gSyncFails = false, gLastError = false;
static int gSyncs[2] = {0, 0};
static thread_local int gFailNew = -1;  // host allocations to go until one fails

void* operator new(size_t n) {
  if (gFailNew >= 0 && gFailNew-- == 0) throw std::bad_alloc();
  void* p = std::malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

struct NoFail {  // the stand-in's own books
  int keep = gFailNew;
  NoFail() { gFailNew = -1; }
  ~NoFail() { gFailNew = keep; }
};
hipError_t hipGetDevice(int* d) { return *d = gDev, hipSuccess; }
hipError_t hipSetDevice(int d) { return gDev = d, hipSuccess; }
hipError_t hipMemGetInfo(size_t* f, size_t* t) { return *f = gTotal[gDev] - gUsed[gDev], *t = gTotal[gDev], hipSuccess; }
hipError_t hipGetLastError() {
  const bool e = gLastError;
  gLastError = false;
  return e ? hipErrorOutOfMemory : hipSuccess;
}
hipError_t hipDeviceSynchronize() {
  std::lock_guard<std::mutex> lk(gMu);
  ++gSyncs[gDev];
  return gSyncFails ? hipErrorUnknown : hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
  NoFail nf;
  std::lock_guard<std::mutex> lk(gMu);
  if (gFailMallocs > 0 || gUsed[gDev] + n > gTotal[gDev]) {
    if (gFailMallocs > 0) --gFailMallocs;
    gLastError = true;
    return hipErrorOutOfMemory;
  }
  ++gMallocs;
  *p = std::malloc(1);
  gMem[*p] = {n, gDev};
  gUsed[gDev] += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  NoFail nf;
  std::lock_guard<std::mutex> lk(gMu);
  auto it = gMem.find(p);
  if (it == gMem.end()) std::printf("hipFree of an unknown block\n"), std::abort();
  ++gFrees;
  gUsed[it->second.second] -= it->second.first;
  gMem.erase(it);
  std::free(p);
  return hipSuccess;
}

#include "mlodsurfaces_amd/csrc/pool.cpp"

using namespace mlod;
#define CHECK(x) ((x) ? (void)0 : (std::printf("line %d: %s\n", __LINE__, #x), std::exit(1)))
static void* take1(size_t n) {
  void* p = nullptr;
  CHECK(dev_malloc_bytes(&p, n) == hipSuccess && p);
  return p;
}
constexpr size_t MB = 1 << 20;  // the bound is 1 MB a device

static void reuse() {
  void* a = take1(10000);
  CHECK(dev_block_bytes(a) == 10240 && gUsed[0] == 10240);
  dev_free(&a, 1);
  CHECK(gUsed[0] == 10240 && gSyncs[0] == 1 && gFrees == 0);  // kept, after a wait
  void* b = take1(9300);                                      // the same class
  CHECK(b == a && gMallocs == 1);
  void* c = take1(9100);  // another
  CHECK(gMallocs == 2 && dev_block_bytes(c) == 9216);
  void* two[3] = {b, nullptr, c};
  dev_free(two, 3);
  CHECK(gSyncs[0] == 2);  // one wait for both
  CHECK(dev_block_bytes(b) == 0);
  dev_trim();
  CHECK(gUsed[0] == 0 && gMem.empty());
}

static void bound_and_order() {
  std::vector<void*> p;
  std::vector<size_t> cls;
  for (int k = 0; k < 12; ++k) p.push_back(take1(cls.emplace_back((size_t)(8 + k % 8) << (14 + k / 8))));  // distinct classes
  size_t sum = 0;
  for (int k = 0; k < 12; ++k) CHECK(dev_block_bytes(p[k]) == cls[k]), sum += cls[k];
  CHECK(sum > 2 * MB);
  dev_free(p.data(), 12);
  CHECK(gUsed[0] <= MB);
  // what is left are the newest: the oldest went first
  size_t left = 0;
  int kept = 0;
  for (int k = 11; k >= 0 && left + cls[k] <= MB; --k) left += cls[k], ++kept;
  CHECK(gUsed[0] == left && gFrees == 12 - kept);
  const int m0 = gMallocs;
  for (int k = 12 - kept; k < 12; ++k) {
    void* q = take1(cls[k]);
    CHECK(q == p[k]);
  }
  CHECK(gMallocs == m0);
  void* old = take1(cls[0]);
  CHECK(gMallocs == m0 + 1);
  for (int k = 12 - kept; k < 12; ++k) dev_free(&p[k], 1);
  dev_free(&old, 1);
  dev_trim();
  CHECK(gMem.empty());
}

static void large_blocks() {
  void* a = take1(MB / 2 + 1);  // over half the bound: exact, and straight back
  CHECK(gUsed[0] == MB / 2 + 1);
  dev_free(&a, 1);
  CHECK(gMem.empty() && gSyncs[0] == 1);
  void* u = nullptr;
  CHECK(dev_malloc_raw(&u, 5000) == hipSuccess && gUsed[0] == 5000);
  CHECK(hipFree(u) == hipSuccess);
  CHECK(dev_malloc_raw(&u, 6000) == hipSuccess);
  dev_free(&u, 1);  // also by dev_free
  CHECK(gMem.empty());
}

static void out_of_memory() {
  void* a[8];
  for (int k = 0; k < 8; ++k) a[k] = take1(100000 + 8192 * k);
  dev_free(a, 8);
  const size_t cached = gUsed[0];
  CHECK(cached > 0);
  gTotal[0] = 4 * MB;  // (the bound stays)
  void* big = take1(4 * MB - 1000);  // does not fit beside the cache
  CHECK(gUsed[0] == 4 * MB - 1000 && !gLastError);
  void* more = (void*)1;
  CHECK(dev_malloc_bytes(&more, 8000) == hipErrorOutOfMemory && more == nullptr);
  CHECK(!gLastError);  // nothing left for the next launch's check
  dev_free(&big, 1);
  a[0] = take1(5000);
  dev_free(a, 1);
  void* raw = nullptr;
  CHECK(dev_malloc_raw(&raw, 4 * MB - 100) == hipSuccess);  // past the cache, at its cost
  CHECK(gUsed[0] == 4 * MB - 100);
  dev_free(&raw, 1);
  // one failure: the retry asks for the exact size
  gFailMallocs = 1;
  void* e = take1(4097);
  CHECK(dev_block_bytes(e) == 4097 && gUsed[0] == 4097);
  dev_free(&e, 1);  // of no class: not kept
  CHECK(gMem.empty());
}

static void failed_wait() {
  void* a = take1(20000);
  gSyncFails = true;
  dev_free(&a, 1);
  CHECK(gMem.empty());  // not handed out again
}

static void two_devices() {
  void* a = take1(20000);
  hipSetDevice(1);
  void* b = take1(20000);
  dev_free(&a, 1);  // of the other device
  CHECK(gDev == 1 && gSyncs[0] == 1 && gSyncs[1] == 0);
  void* c = take1(20000);
  CHECK(c != a && gMem[c].second == 1);
  hipSetDevice(0);
  CHECK(take1(20000) == a);
  void* all[3] = {a, b, c};
  dev_free(all, 3);
  dev_trim();
  CHECK(gMem.empty());
}

static void host_memory_fails() {
  for (int k = 0; k < 6; ++k) {
    void* p = nullptr;
    gFailNew = k;
    const hipError_t e = dev_malloc_bytes(&p, 30000 + 10000 * k);
    gFailNew = -1;
    CHECK((e == hipSuccess) == (p != nullptr) && (e == hipSuccess || e == hipErrorOutOfMemory));
    CHECK(gMem.size() == (p ? 1u : 0u));
    if (!p) continue;
    gFailNew = 0;
    dev_free(&p, 1);
    gFailNew = -1;
    dev_trim();
    CHECK(gMem.empty());
  }
}

static void threads() {
  std::mutex mu;
  std::set<void*> held;
  auto work = [&](int seed) {
    unsigned x = (unsigned)seed;
    std::vector<void*> mine;
    for (int i = 0; i < 4000; ++i) {
      x = x * 1664525u + 1013904223u;
      if (mine.size() < 6 && (x >> 16 & 1)) {
        void* p = take1(5000 + (x >> 20) * 20);
        std::lock_guard<std::mutex> lk(mu);
        CHECK(held.insert(p).second);  // nobody else has it
        mine.push_back(p);
      } else if (!mine.empty()) {
        void* p = mine.back();
        mine.pop_back();
        {
          std::lock_guard<std::mutex> lk(mu);
          held.erase(p);
        }
        dev_free(&p, 1);
        if ((x >> 8 & 63) == 0) dev_trim();
      }
    }
    {
      std::lock_guard<std::mutex> lk(mu);
      for (void* p : mine) held.erase(p);
    }
    dev_free(mine.data(), mine.size());
  };
  std::vector<std::thread> t;
  for (int k = 0; k < 8; ++k) t.emplace_back(work, k + 1);
  for (auto& x : t) x.join();
  CHECK(gUsed[0] <= MB);
  dev_trim();
  CHECK(gMem.empty() && gUsed[0] == 0);
}

int main(int argc, char** argv) {
  const std::string w = argc > 1 ? argv[1] : "";
  const std::map<std::string, void (*)()> all = {{"reuse", reuse}, {"bound_and_order", bound_and_order},
                                                 {"large_blocks", large_blocks}, {"out_of_memory", out_of_memory},
                                                 {"failed_wait", failed_wait}, {"two_devices", two_devices},
                                                 {"host_memory_fails", host_memory_fails}, {"threads", threads}};
  auto it = all.find(w);
  if (it == all.end()) return 2;
  it->second();
  std::printf("ok\n");
  return 0;
}
