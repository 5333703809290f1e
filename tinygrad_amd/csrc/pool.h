// Device allocations behind tga_malloc / tga_free (included by runtime.hip, and on the host by the test of its rules, which brings functions of its own under the names of the runtime's).
#pragma once
#include <algorithm>
#include <exception>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

// ---- Device allocations.  hipFree waits for the device and unmaps, hipMalloc maps again: an entry point that allocates its result (ggml_data_to_tensor, quantize_mxfp8,
// moe_feed_forward) spent 1.6 ms (three results of 70 MB in all) to 3.3 ms (one of 117 MB) per call on them where its kernels take 40 .. 60 us, back to back; with
// freed blocks kept, 0.07 ms for the latter.  So a freed block of at most POOL_BLOCK_MAX bytes is kept for the next request of its size class:
//  * freed blocks are first `dirty`: kernels on any stream may still be using them, exactly as before a hipFree.  They become `clean`, i.e. may be handed out again,
//    after the wait for the device that an hipFree performs - but one for many blocks: when a request finds no clean block of its class while POOL_DIRTY_COUNT
//    blocks of the class (more at each further wait) or POOL_DIRTY_BYTES in all are dirty.  No stream has to be named, no caller synchronises more than it did.  The wait is that of an hipFree of a few bytes allocated
//    for it (1.4 us where the device is idle): an hipDeviceSynchronize is refused during a capture of any thread and ends that capture, an hipFree only during one of its own (measured).
//  * at most POOL_BYTES per device are kept; beyond, blocks of the class used least recently go back to the runtime (what an earlier phase left behind, not the block at hand nor
//    one of the classes in use: 20 and 180 us a call of moe_feed_forward at 32 and 2000 tokens), all of them do before a request is refused for want of memory, and on tga_trim().
//  * size classes are eighths of a power of two (at most 11.1 % of a block is idle).  One mutex.  While its thread captures a stream, tga_free puts any block aside without a call to the runtime (an hipFree would
//    invalidate the capture); one of more than POOL_BLOCK_MAX bytes is freed with the next call of that thread outside a capture.  tga_trim is refused then.
//  * a thread with a capture of its own open gets no block: the replays would go on using one that its call gave back when it returned (and hipMalloc itself refuses then).  Captures that
//    the library did not open are the runtime's to know: an hipFree of nothing is refused during exactly those that hipMalloc is refused during (measured for the three capture modes).
#define POOL_BLOCK_MAX ((size_t)1 << 30)
#define POOL_BYTES ((size_t)4 << 30)
#define POOL_DIRTY_BYTES ((size_t)2 << 30)
#define POOL_DIRTY_COUNT 8                   // of a class at its first wait, twice as many at further ones
#define POOL_DIRTY_COUNT_MAX 32              // (31 us behind running kernels, where a device synchronisation costs 13)

struct PoolClass { std::vector<void*> clean, dirty; size_t due = POOL_DIRTY_COUNT, used = 0; };   // due: dirty blocks at the next wait; used: when one was last taken or put aside
struct Pool { std::map<size_t, PoolClass> classes; size_t kept = 0, dirty = 0, clock = 0; };
static std::mutex g_pool_mutex;
static std::unordered_map<int, Pool> g_pools;                                        // by device
struct PoolBlock { size_t cls; int dev; bool out; };                                  // size class, device, handed out (or kept)
static std::unordered_map<void*, PoolBlock> g_pool_blocks;                           // every block that belongs to a size class

static size_t pool_class(size_t n) {
  if (n <= 4096) return (n + 511) & ~(size_t)511;
  int b = 0; for (size_t t = n - 1; t >>= 1;) b++;                                   // 2^b < n <= 2^(b + 1)
  const size_t step = (size_t)1 << (b - 3);
  return (n + step - 1) & ~(step - 1);
}
static int pool_settle(Pool& p) {                                                     // every dirty block becomes clean (not where there is no memory left: the caller trims then)
  void* few = nullptr;
  if (hipMalloc(&few, 512) != hipSuccess) { (void)hipGetLastError(); return 0; }
  TGA_HIP(hipFree(few));
  for (auto& c : p.classes) { c.second.clean.insert(c.second.clean.end(), c.second.dirty.begin(), c.second.dirty.end()); c.second.dirty.clear(); }
  p.dirty = 0;
  return 0;
}
static int pool_release(Pool& p) {                                                    // everything kept goes back to the runtime (hipFree waits for the block's users)
  for (auto& c : p.classes) {
    for (auto* v : {&c.second.clean, &c.second.dirty}) {
      while (!v->empty()) {                                                           // (out of the lists first: where an hipFree fails, no block that is gone may stay in them)
        void* q = v->back();
        v->pop_back(); g_pool_blocks.erase(q); p.kept -= c.first;
        if (v == &c.second.dirty) p.dirty -= c.first;
        TGA_HIP(hipFree(q));
      }
    }
  }
  p.classes.clear();
  return 0;
}
static int pool_make_room(Pool& p, size_t n) {                                        // blocks of the class that was used least recently go back until n more may be kept
  while (p.kept && p.kept + n > POOL_BYTES) {
    std::pair<const size_t, PoolClass>* idle = nullptr;
    for (auto& c : p.classes) if (c.second.clean.size() + c.second.dirty.size() && (!idle || c.second.used < idle->second.used)) idle = &c;
    std::vector<void*>& v = idle->second.clean.empty() ? idle->second.dirty : idle->second.clean;
    void* q = v.back();
    if (&v == &idle->second.dirty) p.dirty -= idle->first;
    v.pop_back(); g_pool_blocks.erase(q); p.kept -= idle->first;
    TGA_HIP(hipFree(q));
  }
  return 0;
}
static int pool_trim() { for (auto& p : g_pools) if (const int rc = pool_release(p.second)) return rc; return 0; }

static thread_local int t_captures = 0;                                              // captures of this thread (tga_graph_begin .. tga_graph_end / tga_cmdlist_end: they end where they began)
static thread_local std::vector<void*> t_large;                                      // blocks of no size class freed during one
static int pool_free_large() { while (!t_large.empty()) { void* q = t_large.back(); t_large.pop_back(); TGA_HIP(hipFree(q)); } return 0; }
static int pool_malloc_(void** ptr, size_t n) {
  TGA_REQUIRE(!t_captures, "tga_malloc: not while this thread captures a stream");
  if (const int rc = pool_free_large()) return rc;
  TGA_HIP(hipFree(nullptr));                                                          // (0.2 us) a capture that something else opened: refused (error 900) where hipMalloc is, else nothing
  if (n > POOL_BLOCK_MAX) {
    hipError_t e = hipMalloc(ptr, n);
    if (e != hipErrorOutOfMemory) { TGA_HIP(e); return 0; }
    (void)hipGetLastError();
    std::lock_guard<std::mutex> lock(g_pool_mutex);
    if (const int rc = pool_trim()) return rc;
    TGA_HIP(hipMalloc(ptr, n));
    return 0;
  }
  int dev = 0;
  TGA_HIP(hipGetDevice(&dev));
  const size_t cls = pool_class(n);
  std::lock_guard<std::mutex> lock(g_pool_mutex);
  Pool& p = g_pools[dev];
  PoolClass& c = p.classes[cls];
  c.used = ++p.clock;
  if (c.clean.empty() && !c.dirty.empty() && (c.dirty.size() >= c.due || p.dirty >= POOL_DIRTY_BYTES)) {
    if (const int rc = pool_settle(p)) return rc;
    if (c.due < POOL_DIRTY_COUNT_MAX) c.due *= 2;
  }
  if (!c.clean.empty()) { *ptr = c.clean.back(); c.clean.pop_back(); p.kept -= cls; g_pool_blocks[*ptr].out = true; return 0; }
  hipError_t e = hipMalloc(ptr, cls);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    if (const int rc = pool_trim()) return rc;
    e = hipMalloc(ptr, cls);
  }
  TGA_HIP(e);
  try { g_pool_blocks[*ptr] = {cls, dev, true}; } catch (...) { (void)hipFree(*ptr); *ptr = nullptr; throw; }
  return 0;
}
static int pool_free_(void* ptr) {
  if (!t_captures) { if (const int rc = pool_free_large()) return rc; }
  std::lock_guard<std::mutex> lock(g_pool_mutex);
  auto it = g_pool_blocks.find(ptr);
  if (it == g_pool_blocks.end()) {
    if (t_captures) { t_large.push_back(ptr); return 0; }
    TGA_HIP(hipFree(ptr));
    return 0;
  }
  TGA_REQUIRE(it->second.out, "tga_free: the block has been freed before");               // (as hipFree refuses it: kept twice, it would be handed out twice)
  const size_t cls = it->second.cls;
  Pool& p = g_pools[it->second.dev];
  if (!t_captures && p.kept + cls > POOL_BYTES) { if (const int rc = pool_make_room(p, cls)) return rc; }
  PoolClass& c = p.classes[cls];
  c.dirty.push_back(ptr);
  c.used = ++p.clock;
  p.kept += cls; p.dirty += cls; it->second.out = false;
  return 0;
}
// Pinned host memory: a block that is given back waits in a list, without a call to the runtime (an hipHostFree would end a capture of its thread, and a model may be collected during one), for the
// next request or tga_trim(); the list holds no more than what was in use at a time since the last request.
static std::vector<void*> g_pinned, g_pinned_freed;                                   // in use; given back
static int pinned_release() { while (!g_pinned_freed.empty()) { void* q = g_pinned_freed.back(); g_pinned_freed.pop_back(); TGA_HIP(hipHostFree(q)); } return 0; }
static int pinned_malloc_(void** ptr, size_t n) {
  TGA_REQUIRE(!t_captures, "tga_host_malloc: not while this thread captures a stream");
  TGA_HIP(hipFree(nullptr));                                                          // (as in pool_malloc_)
  std::lock_guard<std::mutex> lock(g_pool_mutex);
  if (const int rc = pinned_release()) return rc;
  TGA_HIP(hipHostMalloc(ptr, n, hipHostMallocDefault));
  try { g_pinned.push_back(*ptr); } catch (...) { (void)hipHostFree(*ptr); *ptr = nullptr; throw; }
  return 0;
}
static int pinned_free_(void* ptr) {
  std::lock_guard<std::mutex> lock(g_pool_mutex);
  const auto it = std::find(g_pinned.begin(), g_pinned.end(), ptr);
  TGA_REQUIRE(it != g_pinned.end(), "tga_host_free: no block of tga_host_malloc, or one that has been freed before");      // (in the list it would fail the next caller's request)
  g_pinned_freed.push_back(ptr);
  g_pinned.erase(it);
  return 0;
}
static int pool_give_back_() {
  TGA_REQUIRE(!t_captures, "tga_trim: not while this thread captures a stream");
  if (const int rc = pool_free_large()) return rc;
  std::lock_guard<std::mutex> lock(g_pool_mutex);
  if (const int rc = pinned_release()) return rc;
  return pool_trim();
}
// (the lists may throw where the host has no memory left: an error at the C entries)
template <typename F> static int pool_guarded(const char* who, F f) {
  try { return f(); } catch (const std::exception& e) { return tga_set_error("%s: %s", who, e.what()); }
}
static int pool_malloc(void** ptr, size_t n) { return pool_guarded("tga_malloc", [&] { return pool_malloc_(ptr, n); }); }
static int pool_free(void* ptr) { return pool_guarded("tga_free", [&] { return pool_free_(ptr); }); }
static int pool_give_back() { return pool_guarded("tga_trim", [] { return pool_give_back_(); }); }
static int pinned_malloc(void** ptr, size_t n) { return pool_guarded("tga_host_malloc", [&] { return pinned_malloc_(ptr, n); }); }
static int pinned_free(void* ptr) { return pool_guarded("tga_host_free", [&] { return pinned_free_(ptr); }); }
