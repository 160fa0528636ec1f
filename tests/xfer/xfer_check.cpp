// pcx_xfer.hip on the host (tests/xfer/hip): results of many sizes in one and two
// arrays, copies that fail, and threads that cannot be started for want of memory.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>
#include <new>
#include <vector>

int g_fail_copies = 0, g_pinned = 0;
static thread_local bool t_no_memory = false;   // operator new throws in this thread

void* operator new(size_t n) {
  void* p = t_no_memory ? nullptr : std::malloc(n);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

#include "../../lala-pc_amd/csrc/pcx_xfer.hip"

static int check(size_t n, size_t n2, bool no_memory, const char* what) {
  std::vector<unsigned char> src(n + n2), a(n + 1, 0xee), b(n2 + 1, 0xee);
  unsigned v = 12345u + (unsigned)n;
  for (auto& c : src) c = (unsigned char)((v = v * 1664525u + 1013904223u) >> 24);
  t_no_memory = no_memory;
  const hipError_t he = pcx_internal::copy_to_host(a.data(), n, b.data(), n2, src.data(), 0, nullptr);
  t_no_memory = false;
  const bool ok = he == hipSuccess && !std::memcmp(a.data(), src.data(), n) &&
                  !std::memcmp(b.data(), src.data() + n, n2) && a[n] == 0xee && b[n2] == 0xee;
  if (!ok) std::printf("%s: %zu + %zu bytes: status %d\n", what, n, n2, (int)he);
  return !ok;
}

int main() {
  pcx_internal::xfer_acquire();
  int bad = 0;
  const size_t M = (size_t)1 << 20;
  // engines that come and go with a large result each allocate nothing pinned
  for (int i = 0; i < 5; ++i) {
    bad += check(24 * M, 7 * M, false, "one read an engine");
    bad += g_pinned != 0;
    pcx_internal::xfer_release();
    pcx_internal::xfer_acquire();
  }
  bad += check(24 * M, 8 * M, false, "before the slots");
  bad += g_pinned != 0;
  bad += check(2 * M, 0, false, "the first through the slots");
  bad += g_pinned != 1;
  for (size_t n : {(size_t)0, (size_t)1, M - 1, M, M + 1, 2 * M - 4095, 4 * M, 4 * M + 1, 5 * M + 77, 9 * M + 4097})
    for (size_t n2 : {(size_t)0, (size_t)3, M, 3 * M + 5}) {
      bad += check(n, n2, false, "threads");
      bad += check(n, n2, true, "no memory for threads");
    }
  g_fail_copies = 1;
  std::vector<unsigned char> s(3 * M), d(3 * M);
  bad += pcx_internal::copy_to_host(d.data(), 3 * M, nullptr, 0, s.data(), 0, nullptr) == hipSuccess;
  g_fail_copies = 0;
  bad += check(3 * M, 0, false, "after a failure");
  bad += g_pinned != 1;
  pcx_internal::xfer_release();
  bad += g_pinned != 0;
  std::printf(bad ? "failed\n" : "ok\n");
  return bad != 0;
}
