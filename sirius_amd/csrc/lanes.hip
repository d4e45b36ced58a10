// Whether two streams' launches run side by side: asked when the second lane's stream is made (Context::choose_side).
// Another thread may be capturing a graph meanwhile, and streams of other libraries may be busy: everything here goes to
// the two streams asked about, nothing to the null stream, and the answer comes back through mapped host memory.
#include "context.h"

#include <mutex>

namespace tch {
namespace {
// Two of these, one on each of two streams: whether they ran at the same time.  Each raises its flag and looks for the
// other's; both give up after kPolls looks (about a tenth of a millisecond), so both always end.
constexpr int kPolls = 200;
__device__ unsigned g_handshake[2];   // per side: the flag
__global__ void handshake_kernel(unsigned* flags, unsigned* answer, int side, unsigned token, int polls) {
  if (threadIdx.x != 0) return;
  __hip_atomic_store(flags + side, token, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  unsigned seen = 0;
  for (int i = 0; i < polls && !seen; ++i) {
    seen = __hip_atomic_load(flags + (side ^ 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) == token ? token : 0u;
    __builtin_amdgcn_s_sleep(8);
  }
  __hip_atomic_store(answer + side, seen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
}  // namespace

// Asked of a stream made just now it takes 45 us where the two meet (35 when asked again) and 85-90 where they do not; the first
// question of a process, which loads the kernel, up to 4 ms.  (Making a stream takes 0.2 ms, 3 where it gets a hardware
// queue that did not exist; giving one back 0.3.  A stream turned down costs 0.75 ms in all.)
int run_at_the_same_time(hipStream_t a, hipStream_t b) {
  static std::mutex mu;   // one pair of flags and answers
  static unsigned token = 0;
  static volatile unsigned* answer = nullptr;   // two words, kept for the process
  std::lock_guard<std::mutex> lock(mu);
  if (!answer) {
    void* p = nullptr;
    if (hipHostMalloc(&p, 2 * sizeof(unsigned), hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) {
      (void)hipGetLastError();
      return -1;
    }
    answer = static_cast<unsigned*>(p);
  }
  void *state = nullptr, *seen = nullptr;
  if (hipGetSymbolAddress(&state, HIP_SYMBOL(g_handshake)) != hipSuccess ||
      hipHostGetDevicePointer(&seen, const_cast<unsigned*>(answer), 0) != hipSuccess)
    return -1;
  unsigned *const flags = static_cast<unsigned*>(state), *const to = static_cast<unsigned*>(seen);
  answer[0] = answer[1] = 0;
  // the first launch on a stream makes its queue, which takes longer than the kernels wait
  token += 2;
  hipLaunchKernelGGL(handshake_kernel, dim3(1), dim3(64), 0, b, flags, to, 1, token - 1, 0);
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(a) != hipSuccess || hipStreamSynchronize(b) != hipSuccess) return -1;
  hipLaunchKernelGGL(handshake_kernel, dim3(1), dim3(64), 0, a, flags, to, 0, token, kPolls);
  hipLaunchKernelGGL(handshake_kernel, dim3(1), dim3(64), 0, b, flags, to, 1, token, kPolls);
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(a) != hipSuccess || hipStreamSynchronize(b) != hipSuccess) return -1;
  return answer[0] == token && answer[1] == token ? 1 : 0;
}

}  // namespace tch
