// stage_driver.cpp -- a staging lease whose call failed goes back to the pool
// while no memory can be had: nothing may throw there.
#include <cstdio>
#include <cstdlib>
#include <new>

#include "device.hpp"

static thread_local bool g_fail = false;

void *operator new(size_t n) {
  if (g_fail) throw std::bad_alloc();
  if (void *p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

int main() {
  for (int turn = 0; turn < 2 * hsdl::kStagesKept; ++turn) {
    // (no GPU here: taking the stream fails, the stage itself exists)
    hsdl::StageLease a, b;
    const int ra = a.take(0, 100, 1), rb = b.take(0, 100, 2);
    if (ra == HSDL_OK || rb == HSDL_OK) {
      std::puts("a GPU answered");
      return 1;
    }
    g_fail = true;  // both leases end without memory
    a.~StageLease();
    b.~StageLease();
    g_fail = false;
    new (&a) hsdl::StageLease();
    new (&b) hsdl::StageLease();
  }
  hsdl::release_stages(-1);
  std::puts("stages returned");
  return 0;
}
