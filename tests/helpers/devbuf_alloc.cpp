// The growable device buffer over an allocator of this file's own, for the CPU
// test of a failed allocation: no GPU and no HIP library.
#include <cstdlib>

#include "../../adaptive-multiresolution-dg_amd/csrc/context.hpp"

static bool fail_next = false;

extern "C" hipError_t hipMalloc(void** p, size_t n) {
  if (fail_next) return hipErrorOutOfMemory;
  *p = std::malloc(n);
  return hipSuccess;
}
extern "C" hipError_t hipFree(void* p) {
  std::free(p);
  return hipSuccess;
}
void adg::hip_check(hipError_t e, const char* what) {
  if (e != hipSuccess) throw HipError(what);
}

// grows a buffer to `first` values, fails to grow it to `more`, then asks for
// `after`: whether it holds memory for that many values
extern "C" int grow_fail_grow(size_t first, size_t more, size_t after) {
  adg::DevBuf<double> b;
  fail_next = false;
  b.ensure(first);
  fail_next = true;
  bool thrown = false;
  try {
    b.ensure(more);
  } catch (const adg::HipError&) {
    thrown = true;
  }
  fail_next = false;
  if (!thrown) return -1;
  b.ensure(after);
  return b.p != nullptr && b.cap >= after;
}
