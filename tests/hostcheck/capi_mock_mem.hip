// capi_mock_mem.hip -- the host check of capi_mock.hip with a device memory that fills up (test
// infrastructure only).
#include "mock_hip.h"

namespace mock {
inline size_t& limit() { static size_t l = ~size_t(0); return l; }  // bytes of device memory
inline hipError_t limited_malloc(void** p, size_t n) {
  size_t held = 0;
  for (auto& kv : live())
    if (!kv.second.pinned) held += kv.second.n;
  if (held + n > limit()) return hipErrorOutOfMemory;
  return m_hipMalloc(p, n);
}
}  // namespace mock
#undef hipMalloc
#define hipMalloc mock::limited_malloc
#include "capi_mock.hip"

// device bytes beyond those held now that can still be allocated (negative: no limit)
extern "C" void mock_leave_free(long long bytes) {
  size_t held = 0;
  for (auto& kv : mock::live())
    if (!kv.second.pinned) held += kv.second.n;
  mock::limit() = bytes < 0 ? ~size_t(0) : held + (size_t)bytes;
}
