// The pool of idle ray-query stages: which one a query gets, which one leaves, and that no call throws.
// Exit status: number of the failed expectation, 0 if none.
#include "../../naivetrace_amd/csrc/idle_stages.hpp"
#include <cstdio>
#include <cstdlib>
#include <new>
using namespace ttgpu;

struct Stage {
  int device = 0, slots = 0;
  size_t slot_rays = 0;
  int id = 0;
};
using Pool = IdleStages<Stage, 4>;
static_assert(noexcept(std::declval<Pool &>().Put(Stage{})), "a stage comes back from a destructor");
static_assert(noexcept(std::declval<Pool &>().Take(Stage{})) && noexcept(std::declval<Pool &>().Drop()), "");

static bool g_no_memory = false;
void *operator new(size_t n) {
  if (g_no_memory) throw std::bad_alloc();
  return std::malloc(n);
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

static int g_checks = 0, g_failed = 0;
static void expect(bool ok, const char *what) {
  ++g_checks;
  if (!ok) {
    printf("%d: %s\n", g_checks, what);
    if (!g_failed) g_failed = g_checks;
  }
}

int main() {
  const Stage large{0, 3, 1 << 17, 1}, one_k{0, 1, 1 << 10, 2}, one_64k{0, 1, 1 << 16, 3}, other_device{1, 1, 1 << 10, 4};
  Pool p;
  expect(p.Take(one_k).slots == 0, "an empty pool has none");
  g_no_memory = true;
  p.Put(large);
  expect(p.Take(one_k).slots == 0, "a query of one slot leaves the stage of several alone");
  p.Put(one_64k);
  p.Put(other_device);
  p.Put(one_k);
  expect(p.Take(Stage{0, 1, 1 << 10, 0}).id == 2, "the smallest that fits, not the first");
  expect(p.Take(Stage{0, 1, 1 << 11, 0}).id == 3, "the next larger when the small one is out");
  expect(p.Take(Stage{0, 1, 1 << 10, 0}).slots == 0, "not another device's");
  expect(p.Take(large).id == 1, "a large query gets the stage of several slots");
  expect(p.Take(Stage{0, 3, 1 << 17, 0}).slots == 0, "which is then out");
  expect(p.Take(Stage{1, 1, 1 << 10, 0}).id == 4, "the other device's for that device");
  for (int k = 0; k < 4; ++k) expect(p.Put(Stage{0, 1, (size_t)1024 << k, 10 + k}).slots == 0, "room for four");
  expect(p.Put(Stage{0, 1, 4096, 20}).id == 10, "the smallest of five leaves");
  expect(p.Put(Stage{0, 1, 1024, 21}).id == 21, "which may be the one that comes back");
  int left = 0;
  while (p.Drop().slots) ++left;
  expect(left == 4, "all four come out at the end");
  g_no_memory = false;
  printf("%d checks\n", g_checks);
  return g_failed;
}
