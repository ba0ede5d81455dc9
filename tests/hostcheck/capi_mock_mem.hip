// capi_mock_mem.hip -- the host check of capi_mock.hip with a device memory that fills up and a
// log of the push launches (test infrastructure only).
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
namespace mock {
inline unsigned& push_grid() { static unsigned g = 0; return g; }  // workgroups of the last push
inline void log_launch(const char* kernel, dim3 g) {
  if (!strcmp(kernel, "f")) push_grid() = g.x;  // as launch_push names the kernel it picked
}
}  // namespace mock
#undef hipLaunchKernelGGL
#define hipLaunchKernelGGL(K, G, B, L, S, ...) \
  (mock::log_launch(#K, dim3(G)),              \
   mock_launch((const void*)(K), dim3(G), dim3(B), (size_t)(L), S, __VA_ARGS__))
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
extern "C" unsigned mock_push_workgroups() { return mock::push_grid(); }
