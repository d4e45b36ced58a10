// Whether two streams' launches run side by side: asked when the second lane's stream is made (Context::choose_side).
#include "context.h"

#include <mutex>

namespace tch {
namespace {
// Two of these, one on each of two streams: whether they ran at the same time.  Each raises its flag and looks for the
// other's; both give up after kPolls looks (about a tenth of a millisecond), so both always end.
constexpr int kPolls = 200;
__device__ unsigned g_handshake[4];   // per side: flag, and the token if the other side's flag was seen
__global__ void handshake_kernel(unsigned* state, int side, unsigned token, int polls) {
  if (threadIdx.x != 0) return;
  __hip_atomic_store(state + side, token, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  unsigned seen = 0;
  for (int i = 0; i < polls && !seen; ++i) {
    seen = __hip_atomic_load(state + (side ^ 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) == token ? token : 0u;
    __builtin_amdgcn_s_sleep(8);
  }
  __hip_atomic_store(state + 2 + side, seen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
}  // namespace

int run_at_the_same_time(hipStream_t a, hipStream_t b) {
  static std::mutex mu;   // one pair of flags
  static unsigned token = 0;
  std::lock_guard<std::mutex> lock(mu);
  void* state = nullptr;
  if (hipGetSymbolAddress(&state, HIP_SYMBOL(g_handshake)) != hipSuccess) return -1;
  unsigned* const flags = static_cast<unsigned*>(state);
  // the first launch on a stream makes its queue, which takes longer than the kernels wait
  token += 2;
  hipLaunchKernelGGL(handshake_kernel, dim3(1), dim3(64), 0, b, flags, 1, token - 1, 0);
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(a) != hipSuccess || hipStreamSynchronize(b) != hipSuccess) return -1;
  hipLaunchKernelGGL(handshake_kernel, dim3(1), dim3(64), 0, a, flags, 0, token, kPolls);
  hipLaunchKernelGGL(handshake_kernel, dim3(1), dim3(64), 0, b, flags, 1, token, kPolls);
  unsigned got[4] = {};
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(a) != hipSuccess || hipStreamSynchronize(b) != hipSuccess ||
      hipMemcpy(got, flags, sizeof(got), hipMemcpyDeviceToHost) != hipSuccess)
    return -1;
  return got[2] == token && got[3] == token ? 1 : 0;
}

}  // namespace tch
