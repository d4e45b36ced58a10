// The last step of a LayerNorm backward: the per-workgroup partial sums of dgamma and dbeta, added up per column.  A
// launch of its own, or extra workgroups of the weight gradient that is launched next.
#pragma once

#include "kernels.h"

namespace tch {

constexpr int kColSumLds = 32 * 8 * 2;   // doubles of LDS a workgroup needs

// 8 columns x 32 lanes per workgroup of 256, fp64 sums in a fixed order
__device__ __forceinline__ void col_sum_body(const LnSumArgs& p, uint32_t block, double* lds) {
  auto red = reinterpret_cast<double(*)[8][2]>(lds);
  const int cl = threadIdx.x & 7, lane = threadIdx.x >> 3;
  const int c = block * 8 + cl;
  double s = 0.0, q = 0.0;
  if (c < p.C) {
    constexpr int U = 16;   // 512 row blocks in one round trip to memory
    for (int b = lane; b < p.blocks; b += U * 32) {
      float2 v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int bb = b + u * 32;
        v[u] = bb < p.blocks ? *reinterpret_cast<const float2*>(p.partial + (static_cast<int64_t>(bb) * p.C + c) * 2)
                             : make_float2(0.f, 0.f);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        s += v[u].x;
        q += v[u].y;
      }
    }
  }
  red[lane][cl][0] = s;
  red[lane][cl][1] = q;
  __syncthreads();
  for (int off = 16; off > 0; off >>= 1) {
    if (lane < off) {
      red[lane][cl][0] += red[lane + off][cl][0];
      red[lane][cl][1] += red[lane + off][cl][1];
    }
    __syncthreads();
  }
  if (lane == 0 && c < p.C) {
    const float a = static_cast<float>(red[0][cl][0]), b = static_cast<float>(red[0][cl][1]);
    p.out0[c] = p.accumulate ? p.out0[c] + a : a;
    p.out1[c] = p.accumulate ? p.out1[c] + b : b;
  }
}

}  // namespace tch
