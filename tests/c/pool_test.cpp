// The rules of csrc/pool.h against a runtime of this file's own: a device that is busy until something waits for it, calls that a capture refuses, a limit on memory, frees that fail.
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <map>
#include <new>
#include <set>
#include <string>
#include <unordered_map>
#include <vector>

static bool g_no_host_memory = false;
void* operator new(size_t n) { if (g_no_host_memory) throw std::bad_alloc(); if (void* p = malloc(n)) return p; abort(); }
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

typedef int hipError_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorStreamCaptureUnsupported = 900 };
static char g_msg[256] = "";
static int tga_set_error(const char* fmt, ...) { va_list ap; va_start(ap, fmt); vsnprintf(g_msg, sizeof(g_msg), fmt, ap); va_end(ap); return 1; }
#define TGA_HIP(expr) do { hipError_t _e = (expr); if (_e != hipSuccess) return tga_set_error("HIP Error %d [%s]", (int)_e, #expr); } while (0)
#define TGA_REQUIRE(cond, ...) do { if (!(cond)) return tga_set_error(__VA_ARGS__); } while (0)

static std::set<void*> g_live; static uintptr_t g_next = 1 << 20; static size_t g_limit = ~(size_t)0, g_used = 0;
static std::unordered_map<void*, size_t> g_size;
static int g_waits = 0, g_mallocs = 0, g_fail_free_after = -1;
static bool g_capturing = false, g_capture_broken = false;                // a capture of the calling thread that something else opened
static bool g_other_capture = false;                                       // ... and one of another thread: only a device synchronisation is refused then
static hipError_t refused() { if (g_capturing) { g_capture_broken = true; return hipErrorStreamCaptureUnsupported; } return hipSuccess; }
static hipError_t hipMalloc(void** p, size_t n) {
  if (hipError_t e = refused()) return e;
  if (g_used + n > g_limit) return hipErrorOutOfMemory;
  const bool none = g_no_host_memory; g_no_host_memory = false;
  *p = (void*)g_next; g_next += n + 4096; g_live.insert(*p); g_size[*p] = n; g_used += n; g_mallocs++; g_no_host_memory = none;
  return hipSuccess;
}
static hipError_t hipFree(void* p) {
  if (hipError_t e = refused()) return e;
  if (!p) return hipSuccess;
  if (!g_live.count(p)) return hipErrorInvalidValue;
  if (g_fail_free_after == 0) return hipErrorInvalidValue;
  if (g_fail_free_after > 0) g_fail_free_after--;
  g_live.erase(p); g_used -= g_size[p]; g_waits++;                          // (waits for the device)
  return hipSuccess;
}
enum { hipHostMallocDefault = 0 };
static hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
static hipError_t hipHostFree(void* p) { return hipFree(p); }
[[maybe_unused]] static hipError_t hipDeviceSynchronize() { if (hipError_t e = refused()) return e; if (g_other_capture) { g_capture_broken = true; return hipErrorStreamCaptureUnsupported; } g_waits++; return hipSuccess; }
static hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
[[maybe_unused]] static hipError_t hipGetLastError() { return hipSuccess; }

#include "../../tinygrad_amd/csrc/pool.h"

#define CHECK(c) do { if (!(c)) { printf("%s:%d: %s (last error: %s)\n", __FILE__, __LINE__, #c, g_msg); exit(1); } } while (0)

static void freed_twice() {
  void* a; CHECK(!pool_malloc(&a, 1 << 20));
  CHECK(!pool_free(a)); CHECK(pool_free(a) != 0);
  std::set<void*> got;
  for (int i = 0; i < 40; i++) {                                           // every block handed out once, however often the class is settled
    void* b[4]; for (auto& q : b) { CHECK(!pool_malloc(&q, 1 << 20)); CHECK(got.insert(q).second); }
    for (auto& q : b) { CHECK(!pool_free(q)); CHECK(pool_free(q) != 0); got.erase(q); }
  }
}
static void waits_before_handing_out() {
  for (int i = 0; i < 30; i++) {
    void* a; CHECK(!pool_malloc(&a, 3 << 20)); const int w = g_waits; CHECK(!pool_free(a));
    std::vector<void*> got;
    for (int j = 0; j < 40; j++) { void* b; CHECK(!pool_malloc(&b, 3 << 20)); if (b == a) CHECK(g_waits > w); got.push_back(b); }
    for (void* b : got) CHECK(!pool_free(b));
  }
}

static void keep(size_t n, int count) {                                    // so many kept blocks of a class, free to be handed out
  std::vector<void*> b(count + POOL_DIRTY_COUNT_MAX); for (auto& q : b) CHECK(!pool_malloc(&q, n)); for (auto& q : b) CHECK(!pool_free(q));
  void* q; CHECK(!pool_malloc(&q, n)); CHECK(!pool_free(q));
}
static void capture_opened_elsewhere() {
  keep(5 << 20, 8);
  g_capturing = true;
  void* a = nullptr; CHECK(pool_malloc(&a, 5 << 20) != 0 && !a); CHECK(strstr(g_msg, "900"));
  CHECK(pool_malloc(&a, (size_t)2 << 30) != 0 && !a);
  g_capturing = false;
  CHECK(!pool_malloc(&a, 5 << 20)); CHECK(!pool_free(a));
}
static void capture_of_another_thread() {
  g_other_capture = true;
  std::set<void*> seen; int again = 0;
  for (int i = 0; i < 40; i++) {
    void* b[4]; for (auto& q : b) { CHECK(!pool_malloc(&q, 6 << 20)); again += !seen.insert(q).second; }
    for (auto& q : b) CHECK(!pool_free(q));
  }
  CHECK(again && !g_capture_broken);
}
static void a_free_that_fails() {
  keep(5 << 20, 12); keep(1 << 16, 12);
  g_fail_free_after = 7;
  CHECK(pool_give_back() != 0);
  g_fail_free_after = -1;
  size_t kept = 0, dirty = 0;
  for (auto& c : g_pools[0].classes) { kept += c.first * (c.second.clean.size() + c.second.dirty.size()); dirty += c.first * c.second.dirty.size(); }
  CHECK(kept && kept == g_pools[0].kept && dirty == g_pools[0].dirty);
  for (int i = 0; i < 60; i++) { void* q; CHECK(!pool_malloc(&q, i & 1 ? 5 << 20 : 1 << 16)); CHECK(g_live.count(q)); }
}
static void capture_of_its_own() {                                          // (no call of the library may reach the runtime then)
  void *a, *b; CHECK(!pool_malloc(&a, (size_t)3 << 30)); CHECK(!pool_malloc(&b, 1 << 20));
  std::vector<void*> many(12); for (auto& q : many) CHECK(!pool_malloc(&q, (size_t)1 << 29));
  t_captures = 1; g_capturing = true;
  void* c = nullptr; CHECK(pool_malloc(&c, 1 << 20) != 0 && !c);
  CHECK(!pool_free(a)); CHECK(!pool_free(b)); for (auto& q : many) CHECK(!pool_free(q));      // (6 GiB: more than are kept)
  CHECK(pool_give_back() != 0);
  CHECK(!g_capture_broken && g_live.count(a));
  t_captures = 0; g_capturing = false;
  CHECK(!pool_malloc(&c, 1 << 20)); CHECK(!g_live.count(a)); CHECK(!pool_free(c));
  CHECK(!pool_give_back()); CHECK(g_live.empty() && !g_pools[0].kept && !g_pools[0].dirty);
}
static void classes_hold_little_more() {
  for (size_t n = 4097; n <= POOL_BLOCK_MAX; n += 1 + n / 97)
    for (size_t m : {n, n - n % 4096, n - n % 4096 + 1}) {
      if (m < 4097) continue;
      const size_t c = pool_class(m); CHECK(c >= m && (c - m) * 9 <= c && c % 512 == 0 && pool_class(c) == c);
    }
  for (int b = 12; b < 30; b++) { const size_t m = ((size_t)1 << b) + 1, c = pool_class(m); CHECK((c - m) * 9 <= c); }
}
static void no_host_memory() {
  void *a = nullptr, *b; CHECK(!pool_malloc(&b, 1 << 20));
  g_no_host_memory = true;
  const int rc = pool_malloc(&a, 7 << 20), rf = pool_free(b);
  g_no_host_memory = false;
  CHECK(rc && !a && rf && g_live.size() == 1);
  CHECK(!pool_free(b)); CHECK(!pool_malloc(&a, 7 << 20));                  // (the block that could not be listed is still the caller's)
}
static void full_of_other_blocks() {
  for (size_t n : {(size_t)200 << 20, (size_t)300 << 20}) {                // 6 GiB of two classes, all freed: 4 GiB are kept
    std::vector<void*> b(12); for (auto& q : b) CHECK(!pool_malloc(&q, n)); for (auto& q : b) CHECK(!pool_free(q));
  }
  CHECK(g_pools[0].kept <= POOL_BYTES && g_pools[0].kept > POOL_BYTES - 2 * ((size_t)320 << 20));
  for (size_t n : {(size_t)2 << 20, (size_t)90 << 20}) {                   // small blocks, then some that keep more bytes than any other class in the end
    int mallocs = 0;
    for (int i = 0; i < 400; i++) {
      if (i == 200) mallocs = g_mallocs;
      void *a, *b; CHECK(!pool_malloc(&a, n)); CHECK(!pool_malloc(&b, n / 16)); CHECK(!pool_free(a)); CHECK(!pool_free(b));
    }
    CHECK(g_mallocs - mallocs <= 2 * 200 / POOL_DIRTY_COUNT);               // (the few bytes of each wait)
  }
  CHECK(g_pools[0].kept <= POOL_BYTES);
}
static void pinned_freed_in_a_capture() {
  for (int own = 0; own < 2; own++) {                                       // (a capture that something else opened, and one of the library's)
    void *a, *b; CHECK(!pinned_malloc(&a, 64)); CHECK(!pinned_malloc(&b, 64));
    t_captures = own; g_capturing = true;
    CHECK(!pinned_free(a)); CHECK(pinned_free(a) != 0); CHECK(!g_capture_broken && g_live.count(a));
    if (own) { void* c = nullptr; CHECK(pinned_malloc(&c, 64) != 0 && !c); CHECK(!g_capture_broken); }
    t_captures = 0; g_capturing = false;
    void* c; CHECK(!pinned_malloc(&c, 64)); CHECK(!g_live.count(a));
    CHECK(!pinned_free(b)); CHECK(!pinned_free(c)); CHECK(!pool_give_back()); CHECK(g_live.empty());
  }
}
static void pinned_of_someone_else() {
  void *a, *b; int other = 0; CHECK(!pinned_malloc(&a, 64));
  CHECK(pinned_free(&other) != 0); CHECK(pinned_free((char*)a + 4) != 0);      // (refused here and not in the next caller's request)
  CHECK(!pinned_malloc(&b, 64)); CHECK(g_live.count(a) && g_live.count(b));
  CHECK(!pinned_free(a)); CHECK(!pinned_free(b)); CHECK(!pool_give_back()); CHECK(g_live.empty());
}

int main(int argc, char** argv) {
  const std::map<std::string, void (*)()> tests = {{"freed_twice", freed_twice}, {"waits_before_handing_out", waits_before_handing_out}, {"capture_opened_elsewhere", capture_opened_elsewhere}, {"capture_of_another_thread", capture_of_another_thread}, {"a_free_that_fails", a_free_that_fails}, {"capture_of_its_own", capture_of_its_own}, {"classes_hold_little_more", classes_hold_little_more}, {"no_host_memory", no_host_memory}, {"full_of_other_blocks", full_of_other_blocks}, {"pinned_freed_in_a_capture", pinned_freed_in_a_capture}, {"pinned_of_someone_else", pinned_of_someone_else}};
  CHECK(argc == 2 && tests.count(argv[1]));
  tests.at(argv[1])();
  puts("ok");
}
