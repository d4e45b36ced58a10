// Implicit-GEMM convolution for gfx950: forward, data gradient and weight
// gradient over NHWC activations and KRSC filters, on the 32x32 MFMA tiles
// (v_mfma_f32_32x32x16_bf16; fp32 storage in three bf16 parts, fp32_split.h, or on
// v_mfma_f32_32x32x2_f32), fp32 accumulation, operands staged through LDS in 16-byte chunks.
//
// The reference has no convolution code of its own: its training scripts call
// torchvision's ResNet (train/resnet152.py:22) and the arithmetic is
// F.conv2d / its autograd formulas.  These kernels restate that arithmetic:
//   FWD    y[n,ho,wo,k]  = sum_{r,s,c} x[n, ho*st-p+r, wo*st-p+s, c] * w[k,r,s,c]
//   DGRAD  dx[n,h,w,c]   = sum_{r,s,k} dy[n,(h+p-r)/st,(w+p-s)/st,k] * wt[c,r,s,k]
//   WGRAD  dw[k,r,s,c]   = sum_{n,ho,wo} dy[n,ho,wo,k] * x[n, ho*st-p+r, wo*st-p+s, c]
//
// GEMM view (rows x cols, reduction):
//   FWD    (N*Ho*Wo) x K,        over R*S*C
//   DGRAD  (N*H*W)   x C,        over R*S*K     (filter pre-transposed to [C][R][S][K])
//   WGRAD  K         x (R*S*C),  over N*Ho*Wo, split across workgroups
//
// Kernels: igemm2_kernel (bf16 forward / data gradient, direct-to-LDS), igemm3_kernel (3x3 layers with the activation
// patch in LDS), igemm4_kernel (few output tiles, and fp32: the reduction dealt to the wavefronts of a workgroup),
// igemm_kernel (what those do not take), wgrad_kernel (bf16) / wgrad_f32_kernel.
//
// FWD / DGRAD in igemm_kernel: a tile row in LDS holds one GEMM row (or column) and BK reduction
// elements = 4 chunks of 16 bytes (+1 chunk of padding); a lane's MFMA operand is
// one chunk (lanes 0-31 chunk 2j, lanes 32-63 chunk 2j+1 of their row).
//
// WGRAD: both operands are contiguous along the GEMM row/column (channels) and
// strided along the reduction (pixels), the opposite of what an MFMA operand
// wants.  The tiles are kept as they come, [pixel][channel], and the operand is
// formed by the LDS transpose read of gfx950 (ds_read_b64_tr_b16): a group of 16
// lanes reads a 4-pixel x 16-channel block and every lane receives the 4 pixels
// of ONE channel.
//
// The MFMA is issued with the filter-side fragment as the first operand, so a
// lane's 16 accumulators belong to ONE output row and to groups of 4 consecutive
// output columns: the epilogue moves them through LDS as 16-byte vectors and
// writes (and reads the residual / mask) as full 16-byte chunks per lane.
#include "col_sum.h"
#include "fp32_split.h"
#include "kernels.h"
#include <algorithm>
#include <climits>
#include <iterator>
#include <vector>

#include "context.h"
#include "ops.h"

#include <utility>

#include <mutex>
#include <string>

namespace tch {
namespace {

constexpr int kLdsStride = 5;  // FWD/DGRAD: chunks per LDS tile row: 4 data + 1 pad
constexpr int kRowPad = 4;     // WGRAD, fp32: chunks of padding per [pixel] row (64 bytes)
constexpr int kStagePad = 4;   // epilogue staging: floats of padding per row

enum Mode : int { kFwd = 0, kDgrad = 1, kWgrad = 2 };

struct IgemmArgs {
  const void* a_src;  // FWD: x        DGRAD: dy       WGRAD: dy
  const void* b_src;  // FWD: w        DGRAD: wt       WGRAD: x
  void* out;          // FWD: y        DGRAD: dx       WGRAD: dw (fp32) or split partials
  const void* add;    // optional addend, laid out like out (FWD/DGRAD)
  const void* mask;   // optional: addend counts only where mask > 0
  int add_sub;        // DGRAD: 1 = `add` lives on the stride-2 subsampled pixel grid [N, ceil(H/2), ceil(W/2), C] and
                      // counts at the even (h, w) only (the data gradient of a strided 1x1 convolution, kept compact)
  const float* bias;  // optional per-column bias (FWD)
  const float* scale; // optional per-column factor applied before the bias (FWD: an inference-mode BatchNorm folded in)
  int relu_out;       // FWD: the stored output is max(0, .) of everything above
  float* dbias;       // WGRAD, optional: column sums of dy (the gradient of that bias), [splits][K] partials or final
  float* stats;       // optional: per (row tile, column) pair of sums over the stored output (see finish_tile)
  long long* stat_acc;  // optional, instead of stats: the same pair added to exact accumulators, [copies][4][columns]
  int stat_acc_copies;  // power of two
  const void* bn_mask;      // DGRAD with stats, optional: the stored output is zeroed where bn_mask <= 0
  const void* bn_x;         // DGRAD with stats: input of the BatchNorm this gradient flows into, laid out like out
  const float* bn_mean;     // DGRAD with stats: that BatchNorm's saved batch mean / inverse std per column
  const float* bn_invstd;
  // Optional, with stats: the workgroup that finishes a column tile last also turns the sums into the
  // BatchNorm's per-channel coefficients (no finalize launch).  fin_counters: one int per column tile,
  // zero before the launch; the finishing workgroup leaves it zero again.
  int* fin_counters;
  const float* fin_gamma;
  const float* fin_beta;     // FWD
  float* fin_running_mean;   // FWD, may be null (then fin_running_var is null too)
  float* fin_running_var;
  float* fin_out0;           // FWD: saved batch mean         DGRAD: dgamma
  float* fin_out1;           // FWD: saved inverse std        DGRAD: dbeta
  float* fin_coef;           // FWD: scale[C], shift[C]       DGRAD: coef[3][C] (dx = c0*g + c1*x + c2)
  float fin_momentum, fin_eps;
  int fin_accumulate;        // DGRAD: dgamma / dbeta +=
  int N, H, W, C;     // x side
  int Ho, Wo, K;      // y side
  int R, S, stride, stride_log2, pad;
  int gemm_m, gemm_n, gemm_k;
  int tiles_m, tiles_n, splits;
  int group_rows;   // FWD/DGRAD direct-to-LDS kernel: row tiles per group of the tile order (0 / 1: row-major)
  int k_per_split;  // multiple of BK
  int out_f32;      // FWD/DGRAD: store fp32 instead of T
  int in_fp32;      // fp32, read by the launcher only: no parts (fp32_split.h)
  int accumulate;   // WGRAD with splits == 1: out += result
  int take_pending; // WGRAD, read by the launcher only: the context's pending split reduction rides this launch
  int pointwise;    // 1x1, stride 1, pad 0
  uint32_t a_bytes, b_bytes;  // extents of a_src / b_src for the bounds-checked buffer loads
  FastDiv div_plane;  // pixels per image on the gather side
  FastDiv div_width;  // row width on the gather side
  // The divisions on the way to a kernel's first load, 35 instructions each otherwise.  With these, no tap walk for 1x1 layers, taps
  // by rows and columns, and the operand tiles requested ahead of the epilogue's operands: ResNet-152 of 64 images 13.92 -> 13.78 ms, 2 x 16
  // 13.60 -> 13.38, 20 7.07 -> 6.97, requests of 24 images 2.12 -> 2.07.
  FastDiv div_tiles_n;   // igemm4_kernel: the tiles of a run
  FastDiv div_group;     // FWD/DGRAD: tiles of a group of rows     WGRAD: of a split
  FastDiv div_rows;      // FWD/DGRAD: rows of a group of rows
  FastDiv div_c, div_s;  // WGRAD: C and S
};

// first operand = filter-side fragment (its rows become accumulator registers),
// second operand = activation-side fragment (its rows become accumulator lanes)
template <typename T>
__device__ inline void mma(const Chunk& first, const Chunk& second, f32x16_t& acc);
template <>
__device__ inline void mma<bf16>(const Chunk& first, const Chunk& second, f32x16_t& acc) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(first.h, second.h, acc, 0, 0, 0);
}
template <>
__device__ inline void mma<float>(const Chunk& first, const Chunk& second, f32x16_t& acc) {
#pragma unroll
  for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(first.f[e], second.f[e], acc, 0, 0, 0);
}

// Operand loads go through buffer instructions: an offset outside the declared extent
// returns zeros, so padding, ragged edges and the tail of the reduction need neither a
// branch nor a select, and the loads stay in flight across the multiply of earlier tiles.
typedef unsigned int uint4_t __attribute__((ext_vector_type(4)));
typedef unsigned int uint2_t __attribute__((ext_vector_type(2)));
constexpr uint32_t kOutOfRange = 0x80000000u;

__device__ inline __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), 0x00020000);
}

__device__ inline Chunk load_chunk(__amdgpu_buffer_rsrc_t rsrc, uint32_t byte_off, bool valid) {
  uint4_t v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, static_cast<int>(valid ? byte_off : kOutOfRange), 0, 0);
  Chunk c;
  c.w[0] = v[0];
  c.w[1] = v[1];
  c.w[2] = v[2];
  c.w[3] = v[3];
  return c;
}

// Walks the reduction index of a filter-tap-major operand: (r, s, channel) with
// `channels` per tap, advancing by a fixed step; no division after init.
struct TapWalker {
  int r, s, ch;
  __device__ inline void init(int k, int channels, int S) {
    int tap = k / channels;
    ch = k - tap * channels;
    r = tap / S;
    s = tap - r * S;
  }
  // branch-free; a step covers at most 4 taps (channels >= one chunk, step = 4 chunks)
  __device__ inline void advance(int step, int channels, int S) {
    ch += step;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool wrap = ch >= channels;
      ch -= wrap ? channels : 0;
      s += wrap ? 1 : 0;
      const bool wrap_s = s >= S;
      s = wrap_s ? 0 : s;
      r += wrap_s ? 1 : 0;
    }
  }
};

// Called by every workgroup after it has stored its row of partial sums: the one that arrives last at
// the column tile's counter sums all tiles_m rows of its BN columns (fp64, fixed order) and writes
// the BatchNorm coefficients.  Nobody waits for anybody: a workgroup that is not last just leaves.
// Visibility across the chip's L2 slices without flushing them (a device-scope fence per workgroup
// writes back every dirty line of its L2 slice, the convolution's own output included, and costs
// more than the whole kernel): the partial sums are published with device-scope atomic exchanges,
// whose result the publishing thread waits for before the barrier that precedes the counter bump,
// and the finishing workgroup reads them with device-scope atomic loads.  Atomics execute at the
// point all slices share.
// (Its flag lies in the last word of the staging tile, behind the sums: a variable of its own would cost every kernel 4 bytes
// of LDS, and two workgroups of 80 KB their place on one CU.)
template <int MODE, int BN, int NT, int STAGE_BYTES>
__device__ inline void finalize_column_tile(const IgemmArgs& p, float* stage, int tid, int n0) {
  static_assert(NT * 16 + 4 <= STAGE_BYTES, "sums and flag fit the staging tile");
  int& last_arrival = reinterpret_cast<int*>(stage)[STAGE_BYTES / 4 - 1];
  __syncthreads();
  if (tid == 0) {
    int* counter = p.fin_counters + n0 / BN;
    const int prev = atomicAdd(counter, 1);
    last_arrival = prev == p.tiles_m - 1;
    if (last_arrival) *counter = 0;  // every other workgroup of this column tile has been here already
  }
  __syncthreads();
  if (!last_arrival) return;

  constexpr int PARTS = NT / BN;   // row tiles are dealt round-robin to PARTS threads per column
  const int cl = tid % BN, part = tid / BN;
  double s_part = 0.0, q_part = 0.0;
  if (n0 + cl < p.gemm_n) {
    constexpr int U = 8;
    for (int b = part; b < p.tiles_m; b += U * PARTS) {
      unsigned long long v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int bb = b + u * PARTS;
        v[u] = bb < p.tiles_m
                   ? __hip_atomic_load(reinterpret_cast<const unsigned long long*>(
                                           p.stats + (static_cast<int64_t>(bb) * p.gemm_n + n0 + cl) * 2),
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                   : 0ull;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        s_part += __uint_as_float(static_cast<uint32_t>(v[u]));
        q_part += __uint_as_float(static_cast<uint32_t>(v[u] >> 32));
      }
    }
  }
  double* red = reinterpret_cast<double*>(stage);  // [PARTS][BN][2]
  red[(part * BN + cl) * 2] = s_part;
  red[(part * BN + cl) * 2 + 1] = q_part;
  __syncthreads();
  const int c = n0 + tid;
  if (tid >= BN || c >= p.gemm_n) return;
  double s = 0.0, q = 0.0;
#pragma unroll
  for (int k = 0; k < PARTS; ++k) {
    s += red[(k * BN + tid) * 2];
    q += red[(k * BN + tid) * 2 + 1];
  }
  const double n = static_cast<double>(p.gemm_m);
  const int C = p.gemm_n;
  if (MODE == kFwd) {
    // s = sum x, q = sum x^2  (torch.nn.BatchNorm2d in training mode: biased variance normalises,
    // the unbiased one goes into running_var)
    const double mean = s / n;
    double var = q / n - mean * mean;
    if (var < 0.0) var = 0.0;
    const float invstd = 1.0f / sqrtf(static_cast<float>(var) + p.fin_eps);
    p.fin_out0[c] = static_cast<float>(mean);
    p.fin_out1[c] = invstd;
    if (p.fin_running_mean) {
      const double unbiased = p.gemm_m > 1 ? var * n / (n - 1.0) : var;
      p.fin_running_mean[c] = (1.f - p.fin_momentum) * p.fin_running_mean[c] + p.fin_momentum * static_cast<float>(mean);
      p.fin_running_var[c] = (1.f - p.fin_momentum) * p.fin_running_var[c] + p.fin_momentum * static_cast<float>(unbiased);
    }
    const float sc = p.fin_gamma[c] * invstd;
    p.fin_coef[c] = sc;
    p.fin_coef[C + c] = p.fin_beta[c] - static_cast<float>(mean) * sc;
  } else {
    // s = sum g, q = sum g * xhat
    const float db = static_cast<float>(s), dg = static_cast<float>(q);
    p.fin_out1[c] = p.fin_accumulate ? p.fin_out1[c] + db : db;
    p.fin_out0[c] = p.fin_accumulate ? p.fin_out0[c] + dg : dg;
    const double invstd = p.bn_invstd[c];
    const double scale = static_cast<double>(p.fin_gamma[c]) * invstd;
    const double cb = -scale * invstd * (q / n);
    const double c0 = -scale * (s / n) - cb * p.bn_mean[c];
    p.fin_coef[c] = static_cast<float>(scale);
    p.fin_coef[C + c] = static_cast<float>(cb);
    p.fin_coef[2 * C + c] = static_cast<float>(c0);
  }
}

// Threads of a workgroup that store a tile BN columns wide: whole rows of chunks per visit, a power of two of them (all
// threads, unless the tile is 96 or 192 columns wide).
template <int E, int BN, int NT>
constexpr int storing_threads() {
  int rows = 1;
  while (2 * rows * (BN / E) <= NT) rows *= 2;
  return rows * (BN / E);
}

// The accumulators of one workgroup tile, one 32-row band (index tm) at a time:
// lanes write float4 groups into the staging tile [WM*32][BN + pad], then every
// thread takes E consecutive columns of one row and hands them to `fin` together with the
// number of the visit (tm * ITERS + it, a compile-time constant after unrolling).
template <int E, int WM, int WN, int TM, int TN, typename Fin>
__device__ inline void staged_epilogue(f32x16_t (&acc)[TM][TN], float* stage, int tid, Fin fin) {
  constexpr int BN = WN * TN * 32;
  constexpr int NT = WM * WN * 64;
  constexpr int LD = BN + kStagePad;
  constexpr int CH = BN / E;
  constexpr int NTE = storing_threads<E, BN, NT>();
  constexpr int ITERS = (WM * 32 * CH) / NTE;
  static_assert((WM * 32 * CH) % NTE == 0, "epilogue mapping");
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
#pragma unroll
  for (int tm = 0; tm < TM; ++tm) {
    __syncthreads();
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = wm * 32 + (lane & 31);
        const int c = (wn * TN + tn) * 32 + 8 * j + 4 * (lane >> 5);
        float4 v = make_float4(acc[tm][tn][4 * j], acc[tm][tn][4 * j + 1], acc[tm][tn][4 * j + 2],
                               acc[tm][tn][4 * j + 3]);
        *reinterpret_cast<float4*>(stage + r * LD + c) = v;
      }
    }
    __syncthreads();
    if (NTE < NT && tid >= NTE) continue;
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int q = tid + it * NTE;
      const int r = q / CH, cc = q - r * CH;
      float v[E];
#pragma unroll
      for (int e = 0; e < E; e += 4) {
        float4 t = *reinterpret_cast<const float4*>(stage + r * LD + cc * E + e);
        v[e] = t.x;
        v[e + 1] = t.y;
        v[e + 2] = t.z;
        v[e + 3] = t.w;
      }
      fin(tm * ITERS + it, ((r >> 5) * TM + tm) * 32 + (r & 31), cc * E, v);
    }
  }
}

template <int E>
__device__ inline void store_floats(float* dst, const float* v) {
#pragma unroll
  for (int e = 0; e < E; e += 4) *reinterpret_cast<float4*>(dst + e) = make_float4(v[e], v[e + 1], v[e + 2], v[e + 3]);
}

// ---------------------------------------------------------------------------
// epilogue of forward / data gradient: bias, gated residual, rounding, 16-byte accesses per
// lane; optionally the sums a BatchNorm next to the convolution needs, one pair per (row tile,
// column) at stats[(tile_m * gemm_n + col) * 2], summed in a fixed order:
//   forward:       sum and sum of squares of the values AS STORED (after rounding to T): the
//                  batch statistics of the BatchNorm that follows;
//   data gradient: the output g is the gradient behind a BatchNorm(+ReLU): it is rounded to T,
//                  zeroed where bn_mask <= 0 (the ReLU), stored, and the pair is sum(g) and
//                  sum(g * xhat), xhat = (bn_x - mean) * invstd: the two reductions of the
//                  BatchNorm backward.
// ---------------------------------------------------------------------------
// What the epilogue reads beside the accumulators: per output chunk (a "visit" of a thread) the addend, and for the
// BatchNorm sums the BatchNorm's input and the ReLU's output.  Requested for all chunks of a thread at once, or, where the
// accumulators leave no registers for that, for the chunks of one 32-row band (a data gradient's addend: for one chunk).
// Bounded by latency: reading each chunk's operands when its turn came cost a trip to memory per chunk (the stores between
// them keep the compiler from moving the loads up).  Launches in the step, one at a time: inference convolutions with a
// residual 1-4 us less, data gradients with BatchNorm sums 2-5, with an addend too 5-9; a ResNet-152 request of one image
// 1104 -> 995 us, of 24 images 2288 -> 2148, training steps of 64, 2 x 16 and 20 images 2-3 % shorter.
template <typename T, int MODE, int VISITS, int BAND>
struct EpilogueOperands {
  static constexpr int kGroup = VISITS <= 8 ? VISITS : BAND;
  static constexpr int kAddGroup = MODE == kFwd || VISITS <= 4 ? kGroup : 1;
  static constexpr int E = Elem<T>::kPerChunk;
  Chunk add[kAddGroup], x[kGroup], relu[kGroup];
  // of the thread's columns: scale and bias (forward), mean and inverse std (data gradient with BatchNorm sums)
  float c0[E], c1[E];

  __device__ static inline void request_columns(const float* src, int n, int col, float (&c)[E]) {
    const __amdgpu_buffer_rsrc_t rsrc = make_rsrc(src, static_cast<uint32_t>(n) * 4);
#pragma unroll
    for (int e = 0; e < E; e += 4) {
      const Chunk v = load_chunk(rsrc, static_cast<uint32_t>(col + e) * 4, col < n);
#pragma unroll
      for (int k = 0; k < 4; ++k) c[e + k] = v.f[k];
    }
  }

  // `row`, `col`: of the chunk in the output
  __device__ inline void request_sums(const IgemmArgs& p, int i, int row, int col, bool ok) {
    const uint32_t bytes = static_cast<uint32_t>(p.gemm_m) * p.gemm_n * sizeof(T);
    const uint32_t at = (static_cast<uint32_t>(row) * p.gemm_n + col) * static_cast<uint32_t>(sizeof(T));
    x[i] = load_chunk(make_rsrc(p.bn_x, bytes), at, ok);
    if (p.bn_mask) relu[i] = load_chunk(make_rsrc(p.bn_mask, bytes), at, ok);
  }
  __device__ inline void request_add(const IgemmArgs& p, int i, int row, int col, bool ok) {
    const uint32_t bytes = static_cast<uint32_t>(p.gemm_m) * p.gemm_n * sizeof(T);
    const uint32_t at = (static_cast<uint32_t>(row) * p.gemm_n + col) * static_cast<uint32_t>(sizeof(T));
    if (MODE == kDgrad && p.add_sub) {   // lives on the even pixels: zeros elsewhere
      const uint32_t hs = (p.H + 1) >> 1, ws = (p.W + 1) >> 1;
      uint32_t img, rem, h, w;
      p.div_plane.divmod(static_cast<uint32_t>(row), img, rem);
      p.div_width.divmod(rem, h, w);
      const uint32_t sub = (((img * hs + (h >> 1)) * ws + (w >> 1)) * p.gemm_n + col) * static_cast<uint32_t>(sizeof(T));
      add[i] = load_chunk(make_rsrc(p.add, static_cast<uint32_t>(p.N) * hs * ws * p.gemm_n * sizeof(T)), sub, ok && ((h | w) & 1u) == 0u);
    } else {
      add[i] = load_chunk(make_rsrc(p.add, bytes), at, ok);
    }
  }

  // The operands of the group of chunks that starts at `visit`, if one does.  (NT threads store, a chunk column each;
  // row_of: visit -> row of the tile.)
  template <int BN, int NT, typename RowOf>
  __device__ inline void request_group(const IgemmArgs& p, int visit, bool sums, int tid, int m0, int n0, RowOf row_of) {
    const int col = n0 + (tid % (BN / E)) * E;
    auto stored = [&](int row) { return tid < NT && row < p.gemm_m && col < p.gemm_n; };
    if (MODE == kDgrad && sums && visit % kGroup == 0) {
#pragma unroll
      for (int v = 0; v < kGroup; ++v) request_sums(p, v, m0 + row_of(visit + v), col, stored(m0 + row_of(visit + v)));
    }
    if (p.add && visit % kAddGroup == 0) {
#pragma unroll
      for (int v = 0; v < kAddGroup; ++v) request_add(p, v, m0 + row_of(visit + v), col, stored(m0 + row_of(visit + v)));
    }
  }
  // ahead of the walk over the chunks
  template <int BN, int NT, typename RowOf>
  __device__ inline void request_first(const IgemmArgs& p, int tid, int m0, int n0, RowOf row_of) {
    const int col = n0 + (tid % (BN / E)) * E;
    const bool sums = MODE == kDgrad && (p.stats || p.stat_acc);
    const float* const p0 = MODE == kFwd ? p.scale : sums ? p.bn_mean : nullptr;
    const float* const p1 = MODE == kFwd ? p.bias : sums ? p.bn_invstd : nullptr;
    if (p0) request_columns(p0, p.gemm_n, col, c0);
    if (p1) request_columns(p1, p.gemm_n, col, c1);
    request_group<BN, NT>(p, 0, sums, tid, m0, n0, row_of);
  }
};

// The accumulators reach it through `walk(fin)`, which calls fin(visit, row of the tile, column of the tile, E values) for
// every chunk this thread stores (column chunk tid % CH, so `row_of(visit)` alone names it beforehand); `o` holds the operands
// of its first group of chunks.  NT of the workgroup's BLOCK threads store something; the
// others only keep the barriers company.
template <typename T, int MODE, int BN, int NT, int BLOCK, int VISITS, int BAND, int STAGE_BYTES, typename RowOf, typename Walk>
__device__ inline void finish_walk(const IgemmArgs& p, EpilogueOperands<T, MODE, VISITS, BAND>& o, float* stage, int tid, int m0, int n0,
                                   int tile_m, RowOf row_of, Walk walk) {
  constexpr int E = Elem<T>::kPerChunk;
  constexpr int CH = BN / E;   // column chunks of the tile; a thread always gets chunk tid % CH
  constexpr int ROWS = NT / CH;
  static_assert(NT % CH == 0 && NT <= BLOCK, "stats mapping");
  const bool storing = NT == BLOCK || tid < NT;
  const bool want_stats = p.stats != nullptr || p.stat_acc != nullptr;
  float st_sum[E], st_sq[E];
#pragma unroll
  for (int e = 0; e < E; ++e) st_sum[e] = st_sq[e] = 0.f;
  walk([&](int visit, int tr, int tc, float* v) {
    if (visit > 0) o.template request_group<BN, NT>(p, visit, MODE == kDgrad && want_stats, tid, m0, n0, row_of);
    const int row = m0 + tr, col = n0 + tc;
    if (row >= p.gemm_m || col >= p.gemm_n) return;
    const int64_t idx = static_cast<int64_t>(row) * p.gemm_n + col;
    const int sums_at = visit % o.kGroup, add_at = visit % o.kAddGroup;
    if (MODE == kFwd && p.scale) {
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] *= o.c0[e];
    }
    if (MODE == kFwd && p.bias) {
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] += o.c1[e];
    }
    if (p.add) {
      float a[E];
      chunk_to_float<T>(o.add[add_at], a);
      if (p.mask) {
        Chunk cm;
        cm.u = *reinterpret_cast<const uint4*>(static_cast<const T*>(p.mask) + idx);
        float m[E];
        chunk_to_float<T>(cm, m);
#pragma unroll
        for (int e = 0; e < E; ++e)
          if (!(m[e] > 0.f)) a[e] = 0.f;
      }
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] += a[e];
    }
    if (MODE == kFwd && p.relu_out) {
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = fmaxf(v[e], 0.f);
    }
    if (p.out_f32) {
      store_floats<E>(static_cast<float*>(p.out) + idx, v);
    } else if (MODE == kDgrad && want_stats) {
      Chunk c = float_to_chunk<T>(v);
      chunk_to_float<T>(c, v);
      if (p.bn_mask) {
        float m[E];
        chunk_to_float<T>(o.relu[sums_at], m);
#pragma unroll
        for (int e = 0; e < E; ++e)
          if (!(m[e] > 0.f)) v[e] = 0.f;
        c = float_to_chunk<T>(v);  // exact: every v[e] is a value of T
      }
      *reinterpret_cast<uint4*>(static_cast<T*>(p.out) + idx) = c.u;
      float x[E];
      chunk_to_float<T>(o.x[sums_at], x);
#pragma unroll
      for (int e = 0; e < E; ++e) {
        st_sum[e] += v[e];
        st_sq[e] += v[e] * ((x[e] - o.c0[e]) * o.c1[e]);
      }
    } else {
      const Chunk c = float_to_chunk<T>(v);
      *reinterpret_cast<uint4*>(static_cast<T*>(p.out) + idx) = c.u;
      if (want_stats) {
        chunk_to_float<T>(c, v);  // the statistics are those of the stored values
#pragma unroll
        for (int e = 0; e < E; ++e) {
          st_sum[e] += v[e];
          st_sq[e] += v[e] * v[e];
        }
      }
    }
  });

  if (want_stats) {
    // threads tid, tid + CH, tid + 2 CH, ... hold partial sums of the same E columns
    __syncthreads();
    // [2][E] planes of one float per thread, plane stride NT + 8 floats: the 64 lanes of a store hit 64 consecutive
    // banks, and the 64 lanes of a load below (8 values of e x 8 values of cc) land 8 banks apart per plane: neither
    // has a bank conflict (a [thread][2E] layout made every store a 16-way one)
    constexpr int PS = NT + 8;
    static_assert(2 * E * PS * 4 <= STAGE_BYTES, "the sums fit the staging tile");
    float* red = stage;
    if (storing) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        red[e * PS + tid] = st_sum[e];
        red[(E + e) * PS + tid] = st_sq[e];
      }
    }
    __syncthreads();
    if (tid < BN) {
      const int cc = tid / E, e = tid - cc * E;
      float a = 0.f, b = 0.f;
#pragma unroll 4
      for (int r = 0; r < ROWS; ++r) {   // thread r * CH + cc holds row group r of chunk column cc
        a += red[e * PS + r * CH + cc];
        b += red[(E + e) * PS + r * CH + cc];
      }
      const int col = n0 + tid;
      if (col < p.gemm_n && p.stat_acc) {
        // every row tile adds to the same pair of accumulators: no per-tile partials, nothing to sum up later
        acc_add2(p.stat_acc, p.gemm_n, p.stat_acc_copies, tile_m, col, a, b);
      } else if (col < p.gemm_n) {
        float2* dst = reinterpret_cast<float2*>(p.stats + (static_cast<int64_t>(tile_m) * p.gemm_n + col) * 2);
        if (p.fin_counters) {
          // published for the workgroup that finishes this column tile (see finalize_column_tile)
          const unsigned long long bits = static_cast<unsigned long long>(__float_as_uint(a)) |
                                          (static_cast<unsigned long long>(__float_as_uint(b)) << 32);
          const unsigned long long old = atomicExch(reinterpret_cast<unsigned long long*>(dst), bits);
          asm volatile("" ::"v"(old));  // wait for the exchange itself, not only for its issue
        } else {
          *dst = make_float2(a, b);
        }
      }
    }
    if (p.fin_counters) finalize_column_tile<MODE, BN, NT, STAGE_BYTES>(p, stage, tid, n0);
  }
}

// The form for accumulators spread over the wavefronts of a tile, one 32-row band at a time.  EARLY: the operands are
// requested when the kernel starts and wait in registers until the accumulators are done (the kernels that can spare the
// registers), instead of costing a trip to memory behind the last multiply.  They leave behind the requests of the first operand tiles, which
// then wait for nothing of the epilogue's.  The loop's counted waits do not know of them: requests land in order, so a wait for a
// tile requested behind them waits for them as well, and the first wait, which leaves a fixed number outstanding, for
// as many more operand loads as there are such requests.
template <typename T, int MODE, int WM, int WN, int TM, int TN, bool EARLY>
struct TileEpilogue {
  static constexpr int BN = WN * TN * 32, NT = WM * WN * 64, CH = BN / Elem<T>::kPerChunk;
  static constexpr int NTE = storing_threads<Elem<T>::kPerChunk, BN, NT>();
  static constexpr int ITERS = (WM * 32 * CH) / NTE, VISITS = TM * ITERS;
  EpilogueOperands<T, MODE, VISITS, ITERS> operands;

  __device__ static inline int row_of(int tid, int visit) {
    const int r = (tid + (visit % ITERS) * NTE) / CH;
    return ((r >> 5) * TM + visit / ITERS) * 32 + (r & 31);
  }
  __device__ inline void request(const IgemmArgs& p, int tid, int m0, int n0) {
    operands.template request_first<BN, NTE>(p, tid, m0, n0, [&](int visit) { return row_of(tid, visit); });
  }
  __device__ inline void start(const IgemmArgs& p, int tid, int m0, int n0) {
    if constexpr (EARLY) request(p, tid, m0, n0);
  }
  __device__ inline void finish(const IgemmArgs& p, f32x16_t (&acc)[TM][TN], float* stage, int tid, int m0, int n0, int tile_m) {
    // Nothing but fp32 outputs of a bf16 product (an output head): four columns per thread instead of the eight of a bf16 chunk,
    // so that the lanes of a store lie side by side.  Two stores of every other 16 bytes fill each memory line in two
    // goes (8192 x 50304 over 768, 256 x 256: 842 us with them, 801 so; 2048 rows 234 and 219).
    // Only for the 256 x 256 tile, which large products get; the kernels of the smaller tiles keep their registers.
    if constexpr (MODE == kFwd && sizeof(T) == 2 && WM * TM * WN * TN >= 64) {
      if (p.out_f32 && !p.scale && !p.bias && !p.add && !p.relu_out && !p.stats && !p.stat_acc) {
        staged_epilogue<4, WM, WN, TM, TN>(acc, stage, tid, [&](int, int tr, int tc, const float* v) {
          const int row = m0 + tr, col = n0 + tc;
          if (row < p.gemm_m && col < p.gemm_n)
            store_floats<4>(static_cast<float*>(p.out) + static_cast<int64_t>(row) * p.gemm_n + col, v);
        });
        return;
      }
    }
    if constexpr (!EARLY) request(p, tid, m0, n0);
    finish_walk<T, MODE, BN, NTE, NT, VISITS, ITERS, WM * 32 * (BN + kStagePad) * 4>(
        p, operands, stage, tid, m0, n0, tile_m, [&](int visit) { return row_of(tid, visit); },
        [&](auto fin) { staged_epilogue<Elem<T>::kPerChunk, WM, WN, TM, TN>(acc, stage, tid, fin); });
  }
};

// ---------------------------------------------------------------------------
// forward / data gradient.  PARTS: an fp32 product on the bf16 pipes (fp32_split.h)
// ---------------------------------------------------------------------------
template <typename T, int MODE, int WM, int WN, int TM, int TN, bool PARTS = false>
__global__ __launch_bounds__(WM* WN * 64, PARTS ? 2 : 1) void igemm_kernel(IgemmArgs p) {
  constexpr int E = Elem<T>::kPerChunk;
  constexpr int BK = 4 * E;
  constexpr int BM = WM * TM * 32;
  constexpr int BN = WN * TN * 32;
  constexpr int NT = WM * WN * 64;
  constexpr int EB = sizeof(T);
  constexpr int A_PT = (BM * 4) / NT;
  constexpr int B_PT = (BN * 4) / NT;
  static_assert((BM * 4) % NT == 0 && (BN * 4) % NT == 0, "tile/loader mismatch");
  constexpr int OPER_BYTES = (BM + BN) * kLdsStride * 16 * 2;
  constexpr int STAGE_BYTES = WM * 32 * (BN + kStagePad) * 4;
  constexpr int LDS_BYTES = OPER_BYTES > STAGE_BYTES ? OPER_BYTES : STAGE_BYTES;

  __shared__ uint4 lds[LDS_BYTES / 16];
  uint4* lds_a = lds;                            // [2][BM * kLdsStride]
  uint4* lds_b = lds + 2 * BM * kLdsStride;      // [2][BN * kLdsStride]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;

  uint32_t tile_m, tile_n;
  p.div_tiles_n.divmod(xcd_remap(blockIdx.x, gridDim.x), tile_m, tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int k_end = p.gemm_k;
  const int nk = (k_end + BK - 1) / BK;

  // ---- operand A: gather of activation rows; the chunk column is the same for every i ----
  const int in_h = (MODE == kFwd) ? p.H : p.Ho;
  const int in_w = (MODE == kFwd) ? p.W : p.Wo;
  const int in_c = (MODE == kFwd) ? p.C : p.K;
  const int chunk_col = tid & 3;
  int a_base[A_PT], a_h0[A_PT], a_w0[A_PT];
  bool a_row_ok[A_PT];
  TapWalker walk;
#pragma unroll
  for (int i = 0; i < A_PT; ++i) {
    const int row = m0 + ((tid + i * NT) >> 2);
    a_row_ok[i] = row < p.gemm_m;
    uint32_t img = 0, pix = 0, oh = 0, ow = 0;
    if (a_row_ok[i]) {
      p.div_plane.divmod(static_cast<uint32_t>(row), img, pix);
      p.div_width.divmod(pix, oh, ow);
    }
    if (p.pointwise) {
      a_base[i] = row * in_c;  // dense [gemm_m][in_c]
      a_h0[i] = a_w0[i] = 0;
    } else {
      a_base[i] = static_cast<int>(img) * in_h * in_w * in_c;
      if (MODE == kFwd) {
        a_h0[i] = static_cast<int>(oh) * p.stride - p.pad;
        a_w0[i] = static_cast<int>(ow) * p.stride - p.pad;
      } else {
        a_h0[i] = static_cast<int>(oh) + p.pad;
        a_w0[i] = static_cast<int>(ow) + p.pad;
      }
    }
  }

  // two register sets: the tiles kt+1 and kt+2 are in flight while tile kt is multiplied
  Chunk ra0[A_PT], rb0[B_PT], ra1[A_PT], rb1[B_PT];
  const __amdgpu_buffer_rsrc_t rsrc_a = make_rsrc(p.a_src, p.a_bytes);
  const __amdgpu_buffer_rsrc_t rsrc_b = make_rsrc(p.b_src, p.b_bytes);

  auto load_tiles = [&](int kt, Chunk* ra, Chunk* rb) {
    const int k0 = kt * BK;
    const int kk = k0 + chunk_col * E;
    if (p.pointwise) {
      const bool k_ok = kk < k_end;
#pragma unroll
      for (int i = 0; i < A_PT; ++i)
        ra[i] = load_chunk(rsrc_a, static_cast<uint32_t>(a_base[i] + kk) * EB, a_row_ok[i] && k_ok);
    } else {
      const bool tap_ok = walk.r < p.R && kk < k_end;
#pragma unroll
      for (int i = 0; i < A_PT; ++i) {
        int hi, wi;
        bool ok = a_row_ok[i] && tap_ok;
        if (MODE == kFwd) {
          hi = a_h0[i] + walk.r;
          wi = a_w0[i] + walk.s;
        } else {
          const int th = a_h0[i] - walk.r, tw = a_w0[i] - walk.s;
          const int sm = p.stride - 1;
          ok = ok && th >= 0 && tw >= 0 && ((th & sm) == 0) && ((tw & sm) == 0);
          hi = th >> p.stride_log2;
          wi = tw >> p.stride_log2;
        }
        ok = ok && static_cast<unsigned>(hi) < static_cast<unsigned>(in_h) &&
             static_cast<unsigned>(wi) < static_cast<unsigned>(in_w);
        const uint32_t off = static_cast<uint32_t>(a_base[i] + (hi * in_w + wi) * in_c + walk.ch) * EB;
        ra[i] = load_chunk(rsrc_a, off, ok);
      }
      walk.advance(BK, in_c, p.S);
    }
    // operand B: dense filter rows: FWD reads w[K][R*S*C], DGRAD reads wt[C][R*S*K]
#pragma unroll
    for (int i = 0; i < B_PT; ++i) {
      const int row = n0 + ((tid + i * NT) >> 2);
      const bool ok = row < p.gemm_n && kk < k_end;
      rb[i] = load_chunk(rsrc_b, static_cast<uint32_t>(row * p.gemm_k + kk) * EB, ok);
    }
  };

  auto store_tiles = [&](int buf, const Chunk* ra, const Chunk* rb) {
#pragma unroll
    for (int i = 0; i < A_PT; ++i) {
      const int q = tid + i * NT;
      lds_a[buf * BM * kLdsStride + (q >> 2) * kLdsStride + (q & 3)] = ra[i].u;
    }
#pragma unroll
    for (int i = 0; i < B_PT; ++i) {
      const int q = tid + i * NT;
      lds_b[buf * BN * kLdsStride + (q >> 2) * kLdsStride + (q & 3)] = rb[i].u;
    }
  };

  f32x16_t acc[TM][TN];
  const int frag_row = lane & 31;
  const int frag_half = lane >> 5;
  // the sums of the tile, in `acc`; split_c: in fp32, on the bf16 pipes, small products in `low`
  auto reduce = [&](auto split_c, f32x16_t (&low)[TM][TN]) {
    constexpr bool SPLIT = decltype(split_c)::value;
    clear(acc);
    if constexpr (SPLIT) clear(low);
    walk.init(chunk_col * E, in_c, p.S);
    auto compute = [&](int buf) {
      const uint4* la = lds_a + buf * BM * kLdsStride;
      const uint4* lb = lds_b + buf * BN * kLdsStride;
      auto a_chunk = [&](int tm, int j) {
        Chunk c;
        c.u = la[((wm * TM + tm) * 32 + frag_row) * kLdsStride + 2 * j + frag_half];
        return c;
      };
      auto b_chunk = [&](int tn, int j) {
        Chunk c;
        c.u = lb[((wn * TN + tn) * 32 + frag_row) * kLdsStride + 2 * j + frag_half];
        return c;
      };
      if constexpr (SPLIT) {
        Split8 fb[TN];
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) fb[tn] = split8(b_chunk(tn, 0), b_chunk(tn, 1));
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
          const Split8 fa = split8(a_chunk(tm, 0), a_chunk(tm, 1));
#pragma unroll
          for (int tn = 0; tn < TN; ++tn) mma_split(fb[tn], fa, acc[tm][tn], low[tm][tn]);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          Chunk fa[TM], fb[TN];
#pragma unroll
          for (int tm = 0; tm < TM; ++tm) fa[tm] = a_chunk(tm, j);
#pragma unroll
          for (int tn = 0; tn < TN; ++tn) fb[tn] = b_chunk(tn, j);
#pragma unroll
          for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) mma<T>(fb[tn], fa[tm], acc[tm][tn]);
        }
      }
    };

    // Register set 0 carries the even tiles, set 1 the odd ones.  The loop has no
    // conditionals: tiles past the end of the reduction load as zeros (out-of-range
    // buffer offsets) and multiply to nothing, so an odd tile count costs one empty step.
    load_tiles(0, ra0, rb0);
    load_tiles(1, ra1, rb1);
    store_tiles(0, ra0, rb0);
    __syncthreads();
    load_tiles(2, ra0, rb0);
    for (int kt = 0; kt < nk; kt += 2) {
      compute(0);  // tile kt
      store_tiles(1, ra1, rb1);
      __syncthreads();
      load_tiles(kt + 3, ra1, rb1);
      compute(1);  // tile kt + 1
      store_tiles(0, ra0, rb0);
      __syncthreads();
      load_tiles(kt + 4, ra0, rb0);
    }
  };
  if constexpr (PARTS) {
    f32x16_t low[TM][TN];
    reduce(std::true_type{}, low);
    if (__syncthreads_or(join_split(acc, low))) reduce(std::false_type{}, low);
  } else {
    reduce(std::false_type{}, acc);
  }

  TileEpilogue<T, MODE, WM, WN, TM, TN, false> epilogue;
  epilogue.finish(p, acc, reinterpret_cast<float*>(lds), tid, m0, n0, tile_m);
}

typedef __attribute__((address_space(3))) void* lds_void_ptr;

// 16 bytes per lane from `rsrc` at byte offset voff (+ the wave-uniform soff) to dst + lane*16 in
// LDS; an offset outside the resource stores zeros.  (Kept in a device function: named directly
// in a kernel body, the builtin makes the host pass drop the kernel's launch stub.)
__device__ inline void load_to_lds(__amdgpu_buffer_rsrc_t rsrc, unsigned char* dst, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_ptr)dst, 16, voff, soff, 0, 0);
}

// the registers belong to their values up to this point of the program
template <int A, int B>
__device__ inline void hold(uint4_t (&r)[A][B]) {
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int j = 0; j < B; ++j) asm volatile("" : "+v"(r[i][j]));
}

__device__ inline const void* wave_uniform(const void* ptr) {
  const uint64_t v = reinterpret_cast<uint64_t>(ptr);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
  return reinterpret_cast<const void*>(static_cast<uint64_t>(hi) << 32 | lo);
}

// fn(0), fn(1), .. fn(N - 1) with the index as a constant
template <int... I, typename F>
__device__ __forceinline__ void unrolled_steps(std::integer_sequence<int, I...>, F&& fn) {
  (fn(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void unrolled(F&& fn) {
  unrolled_steps(std::make_integer_sequence<int, N>{}, fn);
}

// All but the newest N of this wave's direct loads have landed, all its LDS accesses are done, and every wave of the
// workgroup is here.  Not __syncthreads(): the compiler puts a wait for EVERY outstanding direct load in front of
// that (a direct load is an LDS write to it), which leaves no tile in flight across the barrier whatever NBUF is:
// each step then pays a whole trip to memory (a 64 x 64 tile: 0.47 us per 64-element step with two buffers or three).
template <int N>
__device__ inline void wait_and_meet() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// ---------------------------------------------------------------------------
// weight gradient
// ---------------------------------------------------------------------------
// The bf16 weight gradient: dy and x tiles of 32 pixels go from global memory straight into LDS rows [pixel][channel]
// and are read transposed (ds_read_b64_tr_b16: a lane gets 4 pixels of one channel).  A 16-byte slot of a row is
// XOR-ed by the row so that the 4 x 32-byte patches of a transposing read spread over all banks although rows are
// unpadded.  64 KB of tiles in flight, four of 128 x 128 or eight of 64 x 64: a workgroup's step is a trip to memory
// divided by the tiles in flight until the operand path of the CU is full (64 x 64, 147 / 75 / 53 us with two / three /
// four tiles where eight steps' worth of splits are missing).  Against the form that staged tiles in registers (two in
// flight, LDS stores of its own): 256 x 2304 over 12 544 pixels 44 -> 31 us, 3072 x 768 over 8192 62 -> 47, 128 x 1152 over
// 50 176 34 -> 26; reading a whole step ahead of its multiplication into a second register set (169 instead of 136
// registers) gained nothing on top, a slice ahead does (128 x 128, below).
// POINTWISE: x is read at dy's pixels (no tap arithmetic).  BIAS: the launch may be asked for the bias gradient.
// 64 x 64 keeps five tiles in LDS instead of eight over up to 60 steps, and over up to 32 where the launch is about one
// workgroup on every compute unit (short_wgrad_ring): the seven requests of the full ring's start are a good part of a short
// reduction, and 40 KB leave room for another workgroup.  ResNet steps in ms with the full ring / five tiles up to 60 steps / this
// rule: of 16 images 6.80 / 6.72 / 6.72, 2 x 16 13.73 / 13.57 / 13.58, 21 7.77 / 7.92 / 7.77, 24 8.13 / 8.27 / 8.13, 28 8.61 / 8.59 /
// 8.55, 32 9.08 / 9.24 / 9.11; of 6-15, 17-20, 40, 48 and 64 images, GPT-2 and Swin-B the same within 0.5 % with all.  Its weight gradients of the third
// stage, 72 of 155: 3 x 3 as 432 workgroups of 33-66 steps are as fast or faster with five tiles, 1 x 1 as 192 of 33 (16
// images) faster, as 256 of 31 (20) the same and of 33-49 (21-32) slower: one workgroup on every compute unit lives off its
// own requests.  With several on each, 60 or 100 steps make no difference.  (Three tiles up to 48 steps: 20 images 7.01 for 7.06,
// but Swin-B of 7 images 4.89 for 4.75.)
constexpr int kWgradRing = 65536, kWgradShortRing = 40960;
inline bool short_wgrad_ring(int64_t workgroups, int steps) { return steps <= (workgroups > 192 && workgroups <= 256 ? 32 : 60); }
template <int WM, int WN, int TM, int TN, int RING>
constexpr int wgrad_direct_buffers() {
  return RING / (32 * (WM * TM + WN * TN) * 64);
}
template <int WM, int WN, int TM, int TN, int RING>
constexpr int wgrad_direct_lds() {
  constexpr int ring = wgrad_direct_buffers<WM, WN, TM, TN, RING>() * 32 * (WM * TM + WN * TN) * 64, stage = WM * 32 * (WN * TN * 32 + kStagePad) * 4;
  return ring > stage ? ring : stage;
}
template <int WM, int WN, int TM, int TN, int RING, bool POINTWISE, bool BIAS>
__device__ __forceinline__ void wgrad_body_direct(const IgemmArgs& p, uint32_t id, unsigned char* lds) {
  constexpr int BKP = 32, NBUF = wgrad_direct_buffers<WM, WN, TM, TN, RING>();
  constexpr int BM = WM * TM * 32, BN = WN * TN * 32, NW = WM * WN;
  constexpr int RA = BM * 2, RB = BN * 2;              // bytes of one pixel row
  constexpr int SA = RA / 16, SB = RB / 16;            // 16-byte slots of it
  constexpr int A_BYTES = BKP * RA, BUF_BYTES = BKP * (RA + RB);
  constexpr int A_LD = A_BYTES / 1024 / NW, B_LD = BKP * RB / 1024 / NW;
  static_assert(A_BYTES % (1024 * NW) == 0 && (BKP * RB) % (1024 * NW) == 0, "tile/loader mismatch");
  static_assert((RA == 256 || RA == 128) && (RB == 256 || RB == 128), "row swizzle");
  static_assert(NBUF * BUF_BYTES <= 65536, "the buffer is part of the reads' immediate offset");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  uint32_t split, tile_m, tile_n;
  p.div_group.divmod(id, split, id);
  p.div_tiles_n.divmod(id, tile_m, tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int k_begin = split * p.k_per_split;
  int k_end = k_begin + p.k_per_split;
  if (k_end > p.gemm_k) k_end = p.gemm_k;
  const int nk = (k_end - k_begin + BKP - 1) / BKP;

  // two 128-byte rows span the 64 banks, or one 256-byte row does: four consecutive rows land on different quarters
  auto swz_a = [](int row) { return RA == 256 ? (row & 3) << 2 : ((row >> 1) & 1) << 2; };
  auto swz_b = [](int row) { return RB == 256 ? (row & 3) << 2 : ((row >> 1) & 1) << 2; };

  // ---- what this lane loads: a fixed channel chunk of dy and of x, one pixel row per direct load ----
  const int a_row = lane / SA, b_row = lane / SB;
  const int a_ch = m0 + ((lane % SA) ^ swz_a(a_row)) * 8;
  const int b_n = n0 + ((lane % SB) ^ swz_b(b_row)) * 8;
  // a channel beyond the tensor has no pixels
  const int a_end = a_ch < p.gemm_m ? k_end : 0, b_end = b_n < p.gemm_n ? k_end : 0;
  // (a grouped launch reads its arguments from memory: told that they are the same in every lane)
  const __amdgpu_buffer_rsrc_t rsrc_a = make_rsrc(wave_uniform(p.a_src), __builtin_amdgcn_readfirstlane(p.a_bytes));
  const __amdgpu_buffer_rsrc_t rsrc_b = make_rsrc(wave_uniform(p.b_src), __builtin_amdgcn_readfirstlane(p.b_bytes));
  int a_pix[A_LD], a_off[A_LD], b_pix[B_LD], b_off[B_LD];   // the pixel each direct load takes next, its byte offset
#pragma unroll
  for (int i = 0; i < A_LD; ++i) {
    a_pix[i] = k_begin + (wave * A_LD + i) * (64 / SA) + a_row;
    a_off[i] = (a_pix[i] * p.K + a_ch) * 2;
  }
  const int a_step = BKP * p.K * 2;
  // Not pointwise: the lane's tap and channel, and every load's place in the input image, moved on by 32 output pixels per step.
  // Row, column and offset move by constants and by others where a row or an image ends: 18 instructions a load, none of them
  // an integer multiplication, which takes the time of four (with seven of those: 256 x 2304 over 12 544 pixels unsplit 65.6 us
  // for 64.1, over 3136 20.4 for 19.5).
  int b_c = b_n, b_h = 0, b_w = 0;
  int b_hi[B_LD], b_wi[B_LD];
  uint32_t step_img = 0, step_oh = 0, step_ow = 0;
  if (!POINTWISE) {
    const int tap = p.div_c.div(b_n);
    const int r = p.div_s.div(tap);
    b_c = b_n - tap * p.C;
    b_h = r - p.pad;
    b_w = tap - r * p.S - p.pad;
    p.div_plane.divmod(BKP, step_img, step_oh);
    p.div_width.divmod(step_oh, step_oh, step_ow);
  }
  const int in_rows = p.Ho * p.stride, in_cols = p.Wo * p.stride;   // what a wrap takes off
  const int h_end = b_h + in_rows, w_end = b_w + in_cols;
  const int step_hi = step_oh * p.stride, step_wi = step_ow * p.stride;
  const int off_step = ((static_cast<int>(step_img) * p.H + step_hi) * p.W + step_wi) * p.C * 2;
  const int off_row = off_step + p.stride * (p.W - p.Wo) * p.C * 2, off_img = (p.H - in_rows) * p.W * p.C * 2;
#pragma unroll
  for (int i = 0; i < B_LD; ++i) {
    b_pix[i] = k_begin + (wave * B_LD + i) * (64 / SB) + b_row;
    b_off[i] = (b_pix[i] * p.C + b_c) * 2;
    b_hi[i] = b_wi[i] = 0;
    if (!POINTWISE) {
      uint32_t img, rem, oh, ow;
      p.div_plane.divmod(static_cast<uint32_t>(b_pix[i]), img, rem);
      p.div_width.divmod(rem, oh, ow);
      b_hi[i] = static_cast<int>(oh) * p.stride + b_h;
      b_wi[i] = static_cast<int>(ow) * p.stride + b_w;
      b_off[i] = (((static_cast<int>(img) * p.H + b_hi[i]) * p.W + b_wi[i]) * p.C + b_c) * 2;
    }
  }
  const int b_step = BKP * p.C * 2;
  // Every lane issues every load whatever it asks for (the counted waits rely on it): an offset out of range where
  // there is no pixel, a tap outside the image, or a tile behind the last one.
  constexpr int LOADS = A_LD + B_LD;
  auto issue_load = [&](int buf, int j) {
    if (j < A_LD) {
      load_to_lds(rsrc_a, lds + buf * BUF_BYTES + (wave * A_LD + j) * 1024, a_pix[j] < a_end ? a_off[j] : static_cast<int>(kOutOfRange), 0);
      a_pix[j] += BKP;
      a_off[j] += a_step;
      return;
    }
    const int i = j - A_LD;
    const int off = b_off[i];
    bool ok = b_pix[i] < b_end;
    if (POINTWISE) {
      b_off[i] += b_step;
    } else {
      ok = ok & (static_cast<unsigned>(b_hi[i]) < static_cast<unsigned>(p.H)) & (static_cast<unsigned>(b_wi[i]) < static_cast<unsigned>(p.W));
      b_wi[i] += step_wi;
      const bool row = b_wi[i] >= w_end;
      b_wi[i] -= row ? in_cols : 0;
      b_hi[i] += row ? step_hi + p.stride : step_hi;
      const bool img = b_hi[i] >= h_end;
      b_hi[i] -= img ? in_rows : 0;
      b_off[i] += row ? off_row : off_step;
      b_off[i] += img ? off_img : 0;
    }
    load_to_lds(rsrc_b, lds + buf * BUF_BYTES + A_BYTES + (wave * B_LD + i) * 1024, ok ? off : static_cast<int>(kOutOfRange), 0);
    b_pix[i] += BKP;
  };

  f32x16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // transposing reads: lane = 16 G + q; the 16 lanes of a group read pixels {8 (G/2) + q/4} x channels {16 (G%2) + 4 (q%4) ..};
  // afterwards lane q owns channel 16 (G%2) + q of the band and four pixels
  const int grp = lane >> 4, q16 = lane & 15;
  const int tr_pix = 8 * (grp >> 1) + (q16 >> 2);
  const int tr_b = (16 * (grp & 1) + 4 * (q16 & 3)) * 2;   // bytes within the 64-byte band
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
  // address of pixel row tr_pix, band w * T + t: the band is four slots, so the row's XOR only moves whole bands
  auto band = [&](int row_bytes, int w_band, int swz) {
    return static_cast<uint32_t>(tr_pix * row_bytes + ((w_band * 4) ^ swz) * 16 + tr_b);
  };
  uint32_t rd_a[TM], rd_b[TN];
#pragma unroll
  for (int t = 0; t < TM; ++t) rd_a[t] = lds_base + band(RA, wm * TM + t, swz_a(tr_pix));
#pragma unroll
  for (int t = 0; t < TN; ++t) rd_b[t] = lds_base + A_BYTES + band(RB, wn * TN + t, swz_b(tr_pix));
  constexpr int SL = BKP / 16, READS = 2 * (TM + TN);
  uint2_t fa[SL][TM][2], fb[SL][TN][2];
  // read i of slice ks of the tile in buffer `buf` (rows + 16 and + 4 keep the row's swizzle, a multiple of four rows)
  auto read_one = [&](auto buf_c, auto ks_c, auto i_c) {
    constexpr int ks = decltype(ks_c)::value, i = decltype(i_c)::value, t = i & 1, j = i >> 1;
    constexpr int AT = decltype(buf_c)::value * BUF_BYTES, ROW = ks * 16 + 4 * t;
    auto &ra = fa;
    auto &rb = fb;
    if constexpr (j < TM) {
      const uint32_t at = rd_a[j];
      asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(ra[ks][j][t]) : "v"(at), "n"(AT + ROW * RA));
    } else {
      const uint32_t at = rd_b[j - TM];
      asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(rb[ks][j - TM][t]) : "v"(at), "n"(AT + ROW * RB));
    }
  };
  auto hold_slice = [&](int ks) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) asm volatile("" : "+v"(fa[ks][tm][t]));
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) asm volatile("" : "+v"(fb[ks][tn][t]));
    }
  };
  auto chunk = [](const uint2_t (&v)[2]) {
    Chunk c;
    c.w[0] = v[0][0];
    c.w[1] = v[0][1];
    c.w[2] = v[1][0];
    c.w[3] = v[1][1];
    return c;
  };

  // The bias gradient of a linear layer is the column sum of dy: the wavefronts of the first column of tiles add up the
  // dy operands they multiply anyway (a lane: one channel of each band, half of the pixels).
  const bool sum_dy = BIAS && p.dbias != nullptr && tile_n == 0 && wn == 0;
  float bsum[TM];
#pragma unroll
  for (int tm = 0; tm < TM; ++tm) bsum[tm] = 0.f;

  constexpr int AHEAD = (NBUF - 2) * LOADS;
  typedef std::integral_constant<int, 0> first_t;
  typedef std::integral_constant<int, 1> second_t;
  static_assert(SL == 2, "two slices a step");
  // multiplies slice ks; `behind(m)` stands behind its m-th MFMA
  auto multiply = [&](int ks, auto behind) {
    Chunk ca[TM], cb[TN];
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) ca[tm] = chunk(fa[ks][tm]);
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) cb[tn] = chunk(fb[ks][tn]);
    unrolled<TM * TN>([&](auto m_c) {
      constexpr int m = decltype(m_c)::value, tm = m / TN, tn = m % TN;
      mma<bf16>(cb[tn], ca[tm], acc[tm][tn]);
      behind(m_c);
    });
    if (sum_dy) {
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) {
        float v[8];
        chunk_to_float<bf16>(ca[tm], v);
#pragma unroll
        for (int e = 0; e < 8; ++e) bsum[tm] += v[e];
      }
    }
  };
  // 64 x 64: all reads of a step, then its multiplies; others as in igemm2_kernel's interleaved tilings: while slice ks is
  // multiplied, the slice behind it is read into the other registers and a half of the direct loads goes out.  The barrier that
  // hands over the next tile stands in front of a tile's last slice, which is in registers by then: the buffer takes another
  // tile from there on.  128 x 128 alone on a CU: 0.249 -> 0.203 us a step (3072 x 768 over 8192
  // rows unsplit 71 -> 59.5).  What bounds it with two workgroups on a CU is LDS, 24 KB in and out per 16 pixels: 0.179 both ways.  (64 x 64 has one MFMA to put four reads and a
  // load behind: 1 x 1 the same, 3 x 3 66 -> 78 us.)
  constexpr bool INTERLEAVED = TM * TN > 1;
  constexpr int EARLY = INTERLEAVED ? LOADS / 2 : 0;   // of a tile's loads, behind the second slice; the others behind the next first one
  auto slice = [&](auto ks_c, auto buf_c, auto ld_buf_c) {   // multiplies slice ks; reads the other one from `buf`
    constexpr int ks = decltype(ks_c)::value, FROM = ks == 1 ? 0 : EARLY, AUX = READS + (ks == 1 ? EARLY : LOADS - EARLY);
    constexpr int PER = (AUX + TM * TN - 1) / (TM * TN);
    multiply(ks, [&](auto m_c) {
      unrolled<PER>([&](auto a_c) {
        constexpr int a = decltype(m_c)::value * PER + decltype(a_c)::value;
        if constexpr (a < READS) read_one(buf_c, std::integral_constant<int, ks ^ 1>{}, std::integral_constant<int, a>{});
        else if constexpr (a < AUX) issue_load(decltype(ld_buf_c)::value, FROM + a - READS);
      });
      __builtin_amdgcn_sched_barrier(0);
    });
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    hold_slice(ks ^ 1);
  };
  auto step = [&](auto u_c) {
    constexpr int u = decltype(u_c)::value, before = (u + NBUF - 1) % NBUF;
    if constexpr (INTERLEAVED) {
      slice(first_t{}, u_c, std::integral_constant<int, before>{});
      wait_and_meet<AHEAD>();
      slice(second_t{}, std::integral_constant<int, (u + 1) % NBUF>{}, u_c);
    } else {
      wait_and_meet<AHEAD>();
      unrolled<READS>([&](auto i_c) { read_one(u_c, first_t{}, i_c); });
      unrolled<READS>([&](auto i_c) { read_one(u_c, second_t{}, i_c); });
#pragma unroll
      for (int j = 0; j < LOADS; ++j) issue_load(before, j);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      hold_slice(0);
      hold_slice(1);
      multiply(0, [](auto) {});
      multiply(1, [](auto) {});
      __builtin_amdgcn_sched_barrier(0);   // the next step's addresses stay in the next step (36 registers less)
    }
  };
#pragma unroll
  for (int s = 0; s < NBUF - 1; ++s)
#pragma unroll
    for (int j = 0; j < LOADS; ++j) issue_load(s, j);
  if constexpr (INTERLEAVED) {
#pragma unroll
    for (int j = 0; j < EARLY; ++j) issue_load(NBUF - 1, j);
    wait_and_meet<AHEAD + EARLY>();
    unrolled<READS>([&](auto i_c) { read_one(first_t{}, first_t{}, i_c); });
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    hold_slice(0);
  }
  int kt = 0;
  for (; kt + NBUF <= nk; kt += NBUF) unrolled<NBUF>(step);
  unrolled<NBUF - 1>([&](auto u_c) {
    if (kt + decltype(u_c)::value < nk) step(u_c);
  });
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the zeros behind the last tile: the epilogue uses their place

  float* out = static_cast<float*>(p.out);
  if (p.splits > 1) out += static_cast<int64_t>(split) * p.gemm_m * p.gemm_n;
  const bool accumulate = p.splits == 1 && p.accumulate;
  staged_epilogue<Elem<bf16>::kPerChunk, WM, WN, TM, TN>(acc, reinterpret_cast<float*>(lds), tid, [&](int, int tr, int tc, float* v) {
    const int row = m0 + tr, col = n0 + tc;
    if (row >= p.gemm_m || col >= p.gemm_n) return;
    float* dst = out + static_cast<int64_t>(row) * p.gemm_n + col;
    if (accumulate) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] += dst[e];
    }
    store_floats<8>(dst, v);
  });
  if (sum_dy) {
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
      const float sum = bsum[tm] + __shfl_xor(bsum[tm], 32, 64);
      const int ch = m0 + (wm * TM + tm) * 32 + (lane & 31);
      if (lane < 32 && ch < p.gemm_m) {
        float* dst = p.dbias + (p.splits > 1 ? static_cast<int64_t>(split) * p.gemm_m : 0) + ch;
        *dst = accumulate ? *dst + sum : sum;
      }
    }
  }
}

// `id`: the workgroup's place among the tiles_m * tiles_n * splits workgroups of this weight gradient
template <int WM, int WN, int TM, int TN, bool PARTS>
__device__ __forceinline__ void wgrad_body_f32(const IgemmArgs& p, uint32_t id) {
  typedef float T;
  constexpr int E = Elem<T>::kPerChunk;
  constexpr int BKP = 4 * E;  // pixels per reduction step
  constexpr int BM = WM * TM * 32;
  constexpr int BN = WN * TN * 32;
  constexpr int NT = WM * WN * 64;
  constexpr int EB = sizeof(T);
  constexpr int CA = BM / E, CB = BN / E;        // data chunks per [pixel] row
  constexpr int LDA = CA + kRowPad, LDB = CB + kRowPad;  // row stride in chunks
  constexpr int A_PT = (BKP * CA) / NT;
  constexpr int B_PT = (BKP * CB) / NT;
  static_assert((BKP * CA) % NT == 0 && (BKP * CB) % NT == 0, "tile/loader mismatch");
  static_assert(NT % CA == 0 && NT % CB == 0, "a thread keeps one chunk column");
  constexpr int OPER_BYTES = 2 * BKP * (LDA + LDB) * 16;
  constexpr int STAGE_BYTES = WM * 32 * (BN + kStagePad) * 4;
  // three parts of bf16 per value: [buffer][dy, x][part][pixel][channel], rows unpadded, 16-byte slots XOR-ed by the row as
  // in wgrad_body_direct
  constexpr int RA = BM * 2, RB = BN * 2;
  constexpr int A_PART = BKP * RA, B_PART = BKP * RB, PARTS_BYTES = 3 * (A_PART + B_PART);
  static_assert((RA == 256 || RA == 128) && (RB == 256 || RB == 128), "row swizzle");
  constexpr int LDS_BYTES = std::max({OPER_BYTES, STAGE_BYTES, PARTS ? 2 * PARTS_BYTES : 0});

  __shared__ uint4 lds[LDS_BYTES / 16];
  uint4* lds_a = lds;                      // [2][BKP][LDA]
  uint4* lds_b = lds + 2 * BKP * LDA;      // [2][BKP][LDB]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;

  uint32_t split, tile_m, tile_n;
  p.div_group.divmod(id, split, id);
  p.div_tiles_n.divmod(id, tile_m, tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int k_begin = split * p.k_per_split;
  int k_end = k_begin + p.k_per_split;
  if (k_end > p.gemm_k) k_end = p.gemm_k;
  const int nk = (k_end - k_begin + BKP - 1) / BKP;

  // operand A = dy[pixel][K]: this thread's channel chunk and first pixel row
  const int a_cc = tid % CA, a_prow = tid / CA;
  const int a_ch = m0 + a_cc * E;
  const bool a_ch_ok = a_ch < p.gemm_m;
  // operand B = x gathered: column n = (tap, channel) is fixed per thread
  const int b_cc = tid % CB, b_prow = tid / CB;
  const int b_n = n0 + b_cc * E;
  const bool b_n_ok = b_n < p.gemm_n;
  int b_r = 0, b_s = 0, b_c = 0;
  if (b_n_ok) {
    const int tap = p.div_c.div(b_n);
    b_c = b_n - tap * p.C;
    b_r = p.div_s.div(tap);
    b_s = tap - b_r * p.S;
  }

  Chunk ra0[A_PT], rb0[B_PT], ra1[A_PT], rb1[B_PT];
  const __amdgpu_buffer_rsrc_t rsrc_a = make_rsrc(p.a_src, p.a_bytes);
  const __amdgpu_buffer_rsrc_t rsrc_b = make_rsrc(p.b_src, p.b_bytes);

  auto load_tiles = [&](int kt, Chunk* ra, Chunk* rb) {
    const int k0 = k_begin + kt * BKP;
#pragma unroll
    for (int i = 0; i < A_PT; ++i) {
      const int pix = k0 + a_prow + i * (NT / CA);
      ra[i] = load_chunk(rsrc_a, static_cast<uint32_t>(pix * p.K + a_ch) * EB, a_ch_ok && pix < k_end);
    }
#pragma unroll
    for (int i = 0; i < B_PT; ++i) {
      const int pix = k0 + b_prow + i * (NT / CB);
      bool ok = b_n_ok && pix < k_end;
      uint32_t off;
      if (p.pointwise) {
        off = static_cast<uint32_t>(pix * p.C + b_c) * EB;
      } else {
        uint32_t img, rem, oh, ow;
        p.div_plane.divmod(static_cast<uint32_t>(pix), img, rem);
        p.div_width.divmod(rem, oh, ow);
        const int hi = static_cast<int>(oh) * p.stride - p.pad + b_r;
        const int wi = static_cast<int>(ow) * p.stride - p.pad + b_s;
        ok = ok && static_cast<unsigned>(hi) < static_cast<unsigned>(p.H) &&
             static_cast<unsigned>(wi) < static_cast<unsigned>(p.W);
        off = static_cast<uint32_t>((static_cast<int>(img) * p.H * p.W + hi * p.W + wi) * p.C + b_c) * EB;
      }
      rb[i] = load_chunk(rsrc_b, off, ok);
    }
  };

  // The bias gradient of a linear layer is the column sum of dy: the workgroups of the first column tile add
  // up the dy chunks they stage anyway (every pixel of the split passes through exactly once).
  const bool sum_dy = p.dbias != nullptr && tile_n == 0;
  float bsum[E];

  auto swz = [](int row_bytes, int row) { return row_bytes == 256 ? (row & 3) << 2 : ((row >> 1) & 1) << 2; };
  unsigned char* const parts = reinterpret_cast<unsigned char*>(lds);
  // four channels of one pixel into the three parts of their operand
  auto store_parts = [&](unsigned char* tile, int part_bytes, int row_bytes, int row, int cc, const Chunk& c) {
    uint2 w[3];
    split4(c, w);
    unsigned char* dst = tile + row * row_bytes + ((cc >> 1) ^ swz(row_bytes, row)) * 16 + (cc & 1) * 8;
#pragma unroll
    for (int k = 0; k < 3; ++k) *reinterpret_cast<uint2*>(dst + k * part_bytes) = w[k];
  };
  // transposing reads: see wgrad_body_direct
  const int grp = lane >> 4, q16 = lane & 15;
  const int tr_pix = 8 * (grp >> 1) + (q16 >> 2);
  auto band = [&](int row_bytes, int w_band) {
    return tr_pix * row_bytes + ((w_band * 4) ^ swz(row_bytes, tr_pix)) * 16 + (16 * (grp & 1) + 4 * (q16 & 3)) * 2;
  };
  auto read_parts = [&](const unsigned char* tile, int part_bytes, int row_bytes, int w_band) {
    Split8 f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const unsigned char* src = tile + k * part_bytes + band(row_bytes, w_band);
      f.part[k] = read_transposed(src, src + 4 * row_bytes);
    }
    return f;
  };

  f32x16_t acc[TM][TN];
  // the sums of the tile, in `acc`; split_c: on the bf16 pipes, small products in `low`
  auto reduce = [&](auto split_c, f32x16_t (&low)[TM][TN]) {
    constexpr bool SPLIT = decltype(split_c)::value;
    clear(acc);
    if constexpr (SPLIT) clear(low);
#pragma unroll
    for (int e = 0; e < E; ++e) bsum[e] = 0.f;

    auto store_tiles = [&](int buf, const Chunk* ra, const Chunk* rb) {
      if constexpr (SPLIT) {
        unsigned char* a_tile = parts + buf * PARTS_BYTES;
#pragma unroll
        for (int i = 0; i < A_PT; ++i) store_parts(a_tile, A_PART, RA, a_prow + i * (NT / CA), a_cc, ra[i]);
#pragma unroll
        for (int i = 0; i < B_PT; ++i) store_parts(a_tile + 3 * A_PART, B_PART, RB, b_prow + i * (NT / CB), b_cc, rb[i]);
      } else {
#pragma unroll
        for (int i = 0; i < A_PT; ++i) lds_a[(buf * BKP + a_prow + i * (NT / CA)) * LDA + a_cc] = ra[i].u;
#pragma unroll
        for (int i = 0; i < B_PT; ++i) lds_b[(buf * BKP + b_prow + i * (NT / CB)) * LDB + b_cc] = rb[i].u;
      }
      if (sum_dy) {
#pragma unroll
        for (int i = 0; i < A_PT; ++i) {
          float v[E];
          chunk_to_float<T>(ra[i], v);
#pragma unroll
          for (int e = 0; e < E; ++e) bsum[e] += v[e];
        }
      }
    };

    auto compute = [&](int buf) {
      if constexpr (SPLIT) {
        const unsigned char* a_tile = parts + buf * PARTS_BYTES;
        Split8 fb[TN];
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) fb[tn] = read_parts(a_tile + 3 * A_PART, B_PART, RB, wn * TN + tn);
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
          const Split8 fa = read_parts(a_tile, A_PART, RA, wm * TM + tm);
#pragma unroll
          for (int tn = 0; tn < TN; ++tn) mma_split(fb[tn], fa, acc[tm][tn], low[tm][tn]);
        }
      } else {
        // one reduction element per lane and MFMA, no transposition needed
        const float* la = reinterpret_cast<const float*>(lds_a + buf * BKP * LDA);
        const float* lb = reinterpret_cast<const float*>(lds_b + buf * BKP * LDB);
#pragma unroll
        for (int ks = 0; ks < BKP / 2; ++ks) {
          const int prow = ks * 2 + (lane >> 5);
          float fa[TM], fb[TN];
#pragma unroll
          for (int tm = 0; tm < TM; ++tm) fa[tm] = la[prow * (LDA * 4) + (wm * TM + tm) * 32 + (lane & 31)];
#pragma unroll
          for (int tn = 0; tn < TN; ++tn) fb[tn] = lb[prow * (LDB * 4) + (wn * TN + tn) * 32 + (lane & 31)];
#pragma unroll
          for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int tn = 0; tn < TN; ++tn)
              acc[tm][tn] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[tn], fa[tm], acc[tm][tn], 0, 0, 0);
        }
      }
    };

    // Register set 0 carries the even tiles, set 1 the odd ones.  The loop has no
    // conditionals: tiles past the end of the reduction load as zeros (out-of-range
    // buffer offsets) and multiply to nothing, so an odd tile count costs one empty step.
    load_tiles(0, ra0, rb0);
    load_tiles(1, ra1, rb1);
    store_tiles(0, ra0, rb0);
    __syncthreads();
    load_tiles(2, ra0, rb0);
    for (int kt = 0; kt < nk; kt += 2) {
      compute(0);  // tile kt
      store_tiles(1, ra1, rb1);
      __syncthreads();
      load_tiles(kt + 3, ra1, rb1);
      compute(1);  // tile kt + 1
      store_tiles(0, ra0, rb0);
      __syncthreads();
      load_tiles(kt + 4, ra0, rb0);
    }
  };
  if constexpr (PARTS) {
    f32x16_t low[TM][TN];
    reduce(std::true_type{}, low);
    if (__syncthreads_or(join_split(acc, low))) reduce(std::false_type{}, low);
  } else {
    reduce(std::false_type{}, acc);
  }

  float* out = static_cast<float*>(p.out);
  if (p.splits > 1) out += static_cast<int64_t>(split) * p.gemm_m * p.gemm_n;
  const bool accumulate = p.splits == 1 && p.accumulate;
  staged_epilogue<Elem<T>::kPerChunk, WM, WN, TM, TN>(acc, reinterpret_cast<float*>(lds), tid, [&](int, int tr, int tc, float* v) {
    const int row = m0 + tr, col = n0 + tc;
    if (row >= p.gemm_m || col >= p.gemm_n) return;
    float* dst = out + static_cast<int64_t>(row) * p.gemm_n + col;
    if (accumulate) {
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] += dst[e];
    }
    store_floats<E>(dst, v);
  });
  if (sum_dy) {
    // NT / CA threads hold partial sums of the same E channels: through LDS, then one thread per channel
    float* red = reinterpret_cast<float*>(lds);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; ++e) red[a_prow * BM + a_cc * E + e] = bsum[e];
    __syncthreads();
    if (tid < BM && m0 + tid < p.gemm_m) {
      float s = 0.f;
#pragma unroll
      for (int r = 0; r < NT / CA; ++r) s += red[r * BM + tid];
      float* dst = p.dbias + (p.splits > 1 ? static_cast<int64_t>(split) * p.gemm_m : 0) + m0 + tid;
      *dst = accumulate ? *dst + s : s;
    }
  }
}

__device__ __forceinline__ void splitk_reduce_body(const ReduceArgs& p, uint32_t block);

// One weight gradient, and optionally, as the workgroups from gemm_wgs on:
//  - the split reduction of the weight gradient launched BEFORE it on the same stream: its partials are complete by
//    stream order, so the reduction needs no launch of its own and runs beside this gradient's multiplications;
//  - the column sums of the LayerNorm backward before it.  As launches of their own they were bound by latency on the
//    main lane (6-11 us each, 25 in a GPT-2 step, 53 in a Swin-B step); here they are free.  Steps, before and after:
//    Swin-B x32 11.96 -> 11.63 ms, x7 5.30 -> 5.16, GPT-2 8x256 4.74 -> 4.60, 2x256 in fp32 7.34 -> 6.99.
struct WgradArgs {
  IgemmArgs a;
  ReduceArgs red;      // from gemm_wgs on, red_blocks workgroups (0: none)
  LnSumArgs cols;      // behind them, the column sums of a LayerNorm backward: the workgroups that are left
  uint32_t gemm_wgs, red_blocks;
};

// what a workgroup beyond the gradient's own does; lds: at least kColSumLds doubles
__device__ __forceinline__ void wgrad_passenger(const WgradArgs& w, double* lds) {
  const uint32_t id = blockIdx.x - w.gemm_wgs;
  if (id < w.red_blocks)
    splitk_reduce_body(w.red, id);
  else
    col_sum_body(w.cols, id - w.red_blocks, lds);
}

template <int WM, int WN, int TM, int TN, bool PARTS>
__global__ __launch_bounds__(WM* WN * 64) void wgrad_f32_kernel(WgradArgs w) {
  if (blockIdx.x >= w.gemm_wgs) {
    __shared__ double red[kColSumLds];
    wgrad_passenger(w, red);
    return;
  }
  wgrad_body_f32<WM, WN, TM, TN, PARTS>(w.a, xcd_remap(blockIdx.x, w.gemm_wgs));
}

template <int WM, int WN, int TM, int TN, int RING, bool POINTWISE, bool BIAS>
__global__ __launch_bounds__(WM* WN * 64) void wgrad_kernel(WgradArgs w) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds[wgrad_direct_lds<WM, WN, TM, TN, RING>()];
  if (blockIdx.x >= w.gemm_wgs) {
    wgrad_passenger(w, reinterpret_cast<double*>(lds));
    return;
  }
  wgrad_body_direct<WM, WN, TM, TN, RING, POINTWISE, BIAS>(w.a, xcd_remap(blockIdx.x, w.gemm_wgs), lds);
}

// The weight gradients of several convolutions in one launch.  `table` holds one argument block per convolution,
// `map` one entry per workgroup: (which convolution, which of its workgroups).  Neighbouring entries of the map
// are workgroups of the same convolution and split, so that after the XCD remap the workgroups that share
// operand rows also share an L2.  Both arrays are read with wave-uniform addresses.
// With fewer workgroups than entries a workgroup takes every gridDim.x-th entry: a launch that is meant to run
// beside other kernels for a long time on a share of every CU instead of flooding the chip.
struct WgradGroupArgs {
  const IgemmArgs* table;
  const uint2* map;
  uint32_t entries;
};

template <typename T, int WM, int WN, int TM, int TN>
__global__ __launch_bounds__(WM* WN * 64) void wgrad_group_kernel(WgradGroupArgs g) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds[sizeof(T) == 2 ? wgrad_direct_lds<WM, WN, TM, TN, kWgradRing>() : 16];
  for (uint32_t gid = xcd_remap(blockIdx.x, gridDim.x); gid < g.entries; gid += gridDim.x) {
    const uint2 e = g.map[gid];
    const IgemmArgs p = g.table[__builtin_amdgcn_readfirstlane(e.x)];
    const uint32_t id = __builtin_amdgcn_readfirstlane(e.y);
    if constexpr (sizeof(T) == 4) wgrad_body_f32<WM, WN, TM, TN, false>(p, id);
    else if (p.pointwise) wgrad_body_direct<WM, WN, TM, TN, kWgradRing, true, true>(p, id, lds);
    else wgrad_body_direct<WM, WN, TM, TN, kWgradRing, false, true>(p, id, lds);
    __syncthreads();   // the next entry's operand tiles overwrite what the epilogue staged in LDS
  }
}

// ---------------------------------------------------------------------------
// forward / data gradient, bf16, channel counts that are multiples of 64
// ---------------------------------------------------------------------------
// Same GEMM view as igemm_kernel, restructured around what gfx950 offers:
//   * operand tiles go from global memory straight into LDS (buffer_load ... lds, 16 bytes
//     per lane, out-of-range offsets land as zeros): no staging registers, no LDS stores;
//   * one reduction step is 64 elements = one 128-byte LDS row per GEMM row, unpadded, with
//     the 16-byte slot index XOR-ed by (row >> 1) & 7 so that a 16-lane group of an MFMA
//     operand read touches every bank once;
//   * a step never straddles a filter tap (channels % 64 == 0), so the tap walk is scalar:
//     a lane keeps one byte offset and one validity bit per tap for each row it loads;
//   * NBUF tiles in LDS, one barrier per step: one is multiplied, one is being requested, and NBUF - 2 are in flight
//     across the barrier (none with two, where the other workgroups of the CU fill the trip to memory);
//   * ROT = 1 is the rotated, interleaved loop (see there) with eight wavefronts per tile: two on every SIMD, one multiplies
//     while the other waits.  What bounds a tile then is the operand path of the CU (direct loads reach 135 B/ns, LDS reads
//     600; the loop alone 1.65 PFLOP/s at 128 x 192, MFMA alone 1.84 where 2.5 is the peak).  8192 x 768 over 3072: 43.7 us
//     as 128 x 128 on four wavefronts without it, 37.2 as 128 x 192; 8192 x 2304 over 768 44.8 and 41.1 (128 x 128),
//     2048 x 2304 15.3 and 12.3 (128 x 192); 12 544 x 256 over 1024 with batch sums 14.6 and 12.3 (128 x 128, three tiles);
//   * ROT = 2 reads the operands of the next step into a second register set while this step is multiplied: the barrier
//     hands over a tile one step before it is needed and the LDS latency passes behind the multiplies.  What bounds
//     the small tiles then is LDS itself (a 64 x 64 tile: 32 KB read, 16 KB written per step).  1024 x 768 over 3072:
//     24.3 us with a whole trip to memory per step (0.47 us each), 16.3 with the loads really in flight, 13.5 pipelined;
//     2048 rows 25.3 / 20.6 / 17.8 (128 x 64 on eight wavefronts);
//   * KS = 32 halves the step (64-byte rows, sixteen rows per direct load): half the LDS per tile in flight, so
//     more workgroups share a CU and a small grid is resident in one round.
constexpr int kStep2 = 64;                  // reduction elements per step
constexpr int kRowBytes2 = kStep2 * 2;      // 128

// Whether a kernel can keep the epilogue's operands in registers from its start: by what LDS leaves of the registers (512
// per lane of a SIMD, shared by the wavefronts on it).
template <int MODE, int WAVES, int FRAGS, int RING_BYTES>
constexpr bool igemm2_early() {
  constexpr int per_simd = 163840 / RING_BYTES * WAVES / 4, registers = 512 / per_simd;
  return FRAGS <= (MODE == kFwd ? 3 : 2) && registers >= (MODE == kFwd ? 80 : 160);
}

// Row `row` of a convolution's GEMM as its operand loads need it: element offset of tap (0, 0) in the gathered tensor and one bit
// per tap that exists for this row: where its filter row does and its filter column does.
template <int MODE>
__device__ inline void row_taps(const IgemmArgs& p, int row, int in_h, int in_w, int in_c, int& base, uint32_t& taps) {
  base = 0;
  taps = 0;
  if (row >= p.gemm_m) return;
  if (p.pointwise) {
    base = row * in_c;
    taps = 1u;
    return;
  }
  uint32_t img, pix, oh, ow;
  p.div_plane.divmod(static_cast<uint32_t>(row), img, pix);
  p.div_width.divmod(pix, oh, ow);
  const int sl = p.stride_log2, sm = p.stride - 1;
  int h0, w0;
  if (MODE == kFwd) {
    h0 = static_cast<int>(oh) * p.stride - p.pad;
    w0 = static_cast<int>(ow) * p.stride - p.pad;
    base = ((static_cast<int>(img) * in_h + h0) * in_w + w0) * in_c;
  } else {
    h0 = static_cast<int>(oh) + p.pad;
    w0 = static_cast<int>(ow) + p.pad;
    base = ((static_cast<int>(img) * in_h + (h0 >> sl)) * in_w + (w0 >> sl)) * in_c;
  }
  auto exists = [&](int at, int tap, int extent) {
    if (MODE == kFwd) return static_cast<unsigned>(at + tap) < static_cast<unsigned>(extent);
    const int t = at - tap;
    return t >= 0 && (t & sm) == 0 && (t >> sl) < extent;
  };
  uint32_t cols = 0;
  for (int s = 0; s < p.S; ++s) cols |= exists(w0, s, in_w) ? 1u << s : 0u;
  for (int r = 0; r < p.R; ++r) taps |= exists(h0, r, in_h) ? cols << (r * p.S) : 0u;
}

// The output tile with number `id`.  Wide outputs (group_rows > 1): consecutive ids walk down group_rows row tiles before they move
// one column tile on, so that the tiles an XCD works on at one time form a squarish block (fewer distinct operand rows
// through its L2).
struct Place {
  int tile_m, tile_n;
};
__device__ inline Place place_of(const IgemmArgs& p, uint32_t id) {
  uint32_t q, rem;
  if (p.group_rows <= 1) {
    p.div_tiles_n.divmod(id, q, rem);
    return {static_cast<int>(q), static_cast<int>(rem)};
  }
  p.div_group.divmod(id, q, rem);
  const uint32_t row0 = q * p.group_rows, rows = min(static_cast<uint32_t>(p.group_rows), static_cast<uint32_t>(p.tiles_m) - row0);
  // rem / rows for the rows of a full group and of the last, shorter one
  const uint32_t col = rows == static_cast<uint32_t>(p.group_rows) ? p.div_rows.div(rem) : rem / rows;
  return {static_cast<int>(row0 + (rem - col * rows)), static_cast<int>(col)};
}

template <int MODE, int WM, int WN, int TM, int TN, int NBUF, int ROT = 0, int KS = kStep2>
__global__ __launch_bounds__(WM* WN * 64) void igemm2_kernel(IgemmArgs p) {
  using T = bf16;
  constexpr int E = 8;
  constexpr int BM = WM * TM * 32;
  constexpr int BN = WN * TN * 32;
  constexpr int NW = WM * WN;
  static_assert(KS == 64 || KS == 32, "reduction elements per step");
  constexpr int RB = KS * 2;             // bytes of one LDS row
  constexpr int SLOTS = RB / 16;         // 16-byte slots per row: 8 or 4
  constexpr int SLOT_SH = KS == 64 ? 3 : 2;
  constexpr int LD_ROWS = 1024 / RB;     // rows one direct load of a wave fills: 8 or 16
  constexpr int A_LD = BM / LD_ROWS / NW;  // direct loads per wave and step for the activation tile
  constexpr int B_LD = BN / LD_ROWS / NW;
  static_assert(BM % (LD_ROWS * NW) == 0 && BN % (LD_ROWS * NW) == 0, "tile/loader mismatch");
  constexpr int A_BYTES = BM * RB, B_BYTES = BN * RB;
  // slot = chunk ^ swizzle(row): with 128-byte rows two rows span the 64 banks and (row >> 1) & 7 spreads sixteen
  // rows of one chunk over all of them; with 64-byte rows four rows span them and (row >> 2) & 3 does the same
  auto swizzle = [](int row) { return KS == 64 ? (row >> 1) & 7 : (row >> 2) & 3; };
  constexpr int BUF_BYTES = A_BYTES + B_BYTES;
  constexpr int STAGE_BYTES = WM * 32 * (BN + kStagePad) * 4;
  constexpr int LDS_BYTES = NBUF * BUF_BYTES > STAGE_BYTES ? NBUF * BUF_BYTES : STAGE_BYTES;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[LDS_BYTES];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;

  const Place place = place_of(p, xcd_remap(blockIdx.x, gridDim.x));
  const int tile_m = place.tile_m, tile_n = place.tile_n;
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  TileEpilogue<T, MODE, WM, WN, TM, TN, igemm2_early<MODE, WM * WN, TM * TN, NBUF * BUF_BYTES>()> epilogue;

  const int in_h = (MODE == kFwd) ? p.H : p.Ho;
  const int in_w = (MODE == kFwd) ? p.W : p.Wo;
  const int in_c = (MODE == kFwd) ? p.C : p.K;
  const int cblocks = in_c / KS;
  const int nk = p.R * p.S * cblocks;
  const int sl = p.stride_log2;

  // ---- per lane: the rows it feeds, their byte offset at tap (0,0) and which taps exist ----
  const int sub_row = lane >> SLOT_SH, slot = lane & (SLOTS - 1);
  int a_off[A_LD];
  uint32_t a_taps[A_LD];
#pragma unroll
  for (int j = 0; j < A_LD; ++j) {
    const int trow = (wave * A_LD + j) * LD_ROWS + sub_row;
    const int chunk = slot ^ swizzle(trow);
    const int row = m0 + trow;
    uint32_t taps;
    int base;
    row_taps<MODE>(p, row, in_h, in_w, in_c, base, taps);
    a_off[j] = (base + chunk * E) * 2;
    a_taps[j] = taps;
  }
  int b_off[B_LD];
#pragma unroll
  for (int j = 0; j < B_LD; ++j) {
    const int trow = (wave * B_LD + j) * LD_ROWS + sub_row;
    const int chunk = slot ^ swizzle(trow);
    const int row = n0 + trow;
    b_off[j] = row < p.gemm_n ? (row * p.gemm_k + chunk * E) * 2 : static_cast<int>(kOutOfRange);
  }

  const __amdgpu_buffer_rsrc_t rsrc_a = make_rsrc(p.a_src, p.a_bytes);
  const __amdgpu_buffer_rsrc_t rsrc_b = make_rsrc(p.b_src, p.b_bytes);

  // scalar walk over (tap, channel block)
  int ld_r = 0, ld_s = 0, ld_cb = 0, ld_t = 0, ld_kt = 0;
  // direct load j (of the A_LD + B_LD) of the tile the walk stands at
  auto issue_load = [&](int buf, int j) {
    // element offset of this tap relative to tap (0,0), then bytes
    const int tap_elems = (MODE == kFwd) ? (ld_r * in_w + ld_s) * in_c : -((ld_r >> sl) * in_w + (ld_s >> sl)) * in_c;
    const int a_step = (tap_elems + ld_cb * KS) * 2;
    const int b_step = ld_kt * RB;
    // a tile behind the last one: every offset out of range, so zeros land and memory is not asked
    const uint32_t tap_bit = ld_kt < nk ? 1u << ld_t : 0u;
    const int beyond = ld_kt < nk ? 0 : static_cast<int>(kOutOfRange);
    if (j < A_LD) {
      const bool ok = (a_taps[j] & tap_bit) != 0;
      const int off = ok ? a_off[j] + a_step : static_cast<int>(kOutOfRange);
      load_to_lds(rsrc_a, lds + buf * BUF_BYTES + (wave * A_LD + j) * 1024, off, 0);
    } else {
      load_to_lds(rsrc_b, lds + buf * BUF_BYTES + A_BYTES + (wave * B_LD + j - A_LD) * 1024, b_off[j - A_LD] | beyond, b_step);
    }
  };
  auto next_tile = [&] {
    ++ld_kt;
    // selects, not branches: no block boundary while operand reads are in flight
    const int next_tap = ++ld_cb == cblocks ? 1 : 0;
    ld_cb = next_tap ? 0 : ld_cb;
    ld_t += next_tap;
    ld_s += next_tap;
    const int next_row = ld_s == p.S ? 1 : 0;
    ld_s = next_row ? 0 : ld_s;
    ld_r += next_row;
  };
  auto issue_loads = [&](int buf) {
#pragma unroll
    for (int j = 0; j < A_LD + B_LD; ++j) issue_load(buf, j);
    next_tile();
  };

  f32x16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // operand reads: row = tile row of the lane, slot = chunk ^ swizzle(row); the tile bases are
  // multiples of 32 rows, so the swizzle term depends on the lane only
  const int frag_row = lane & 31, frag_half = lane >> 5;
  const int swz = swizzle(frag_row);
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
  const uint32_t a_rd = lds_base + (wm * TM * 32 + frag_row) * RB + swz * 16;
  const uint32_t b_rd = lds_base + A_BYTES + (wn * TN * 32 + frag_row) * RB + swz * 16;
  // The operand reads are written as asm: the compiler orders every LDS read it can see behind
  // ALL outstanding direct-to-LDS loads (vmcnt(0)), which would serialise the prefetch of the
  // next tiles with the multiply of this one.  Which loads must have landed is known here (the
  // counted wait + barrier at the top of a step), so the reads carry their own lgkmcnt waits.
  auto read_frags = [&](int buf, int kk, uint4_t* fa, uint4_t* fb) {
    const uint32_t cx = (2 * kk + frag_half) * 16;
    const uint32_t pa = (a_rd ^ cx) + buf * BUF_BYTES, pb = (b_rd ^ cx) + buf * BUF_BYTES;
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[tm]) : "v"(pa), "n"(tm * 32 * RB));
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[tn]) : "v"(pb), "n"(tn * 32 * RB));
  };
  auto multiply = [&](uint4_t* fa, uint4_t* fb) {
    // ties the registers to the wait that precedes this call in program order
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) asm volatile("" : "+v"(fa[tm]));
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) asm volatile("" : "+v"(fb[tn]));
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
        acc[tm][tn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, fb[tn]),
                                                              __builtin_bit_cast(bf16x8_t, fa[tm]), acc[tm][tn], 0, 0, 0);
  };
  auto compute = [&](int buf) {
    uint4_t fa0[TM], fb0[TN], fa1[TM], fb1[TN];
    read_frags(buf, 0, fa0, fb0);
    read_frags(buf, 1, fa1, fb1);
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(TM + TN));
    multiply(fa0, fb0);
    if constexpr (KS == 32) {   // a 32-element step holds two 16-element slices
      asm volatile("s_waitcnt lgkmcnt(0)");
      multiply(fa1, fb1);
      return;
    }
    read_frags(buf, 2, fa0, fb0);
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(TM + TN));
    multiply(fa1, fb1);
    read_frags(buf, 3, fa1, fb1);
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(TM + TN));
    multiply(fa0, fb0);
    asm volatile("s_waitcnt lgkmcnt(0)");
    multiply(fa1, fb1);
  };

  // at most this many of a wave's loads may still be in flight when its part of the oldest tile must have landed
  constexpr int LOADS = A_LD + B_LD;
  constexpr int AHEAD = (NBUF - 2) * LOADS;
  static_assert(AHEAD < 64, "vmcnt range");

  // One step = wait until only the newer tiles' loads are outstanding (then this wave's part of tile kt has
  // landed; near the end fewer newer tiles exist, so wait for everything), barrier (every wave's part is in
  // LDS and every wave is done with tile kt-1), request the tile NBUF-1 steps ahead into the buffer that just
  // became free, multiply.  The main loop takes NBUF steps per trip with the buffer index a constant and the
  // multiply outside every conditional (inside one, the compiler moves the 64 accumulators between register
  // classes in every step); the last nk % NBUF steps follow one by one.
  auto step = [&](int kt, int u) {
    if (kt + NBUF - 1 <= nk)
      wait_and_meet<AHEAD>();
    else
      wait_and_meet<0>();
    if (kt + NBUF - 1 < nk) issue_loads((u + NBUF - 1) % NBUF);
    compute(u);
  };
  if constexpr (ROT == 2) {
    // Pipelined over the reduction steps: the operands of tile kt+1 are read into a second register set while tile kt
    // is multiplied.
    static_assert(NBUF == 4, "two register sets, alternating with the buffers");
    constexpr int SL = KS / 16;
    uint4_t fa[2][SL][TM], fb[2][SL][TN];
    // the buffer is part of the reads' immediate offset where that reaches (64 KB)
    auto read_tile = [&](auto buf_c, uint4_t (&ra)[SL][TM], uint4_t (&rb)[SL][TN]) {
      constexpr int AT = decltype(buf_c)::value * BUF_BYTES;
      constexpr bool IMM = AT + BUF_BYTES <= 65536;
#pragma unroll
      for (int kk = 0; kk < SL; ++kk) {
        const uint32_t cx = (2 * kk + frag_half) * 16;
        const uint32_t pa = (a_rd ^ cx) + (IMM ? 0 : AT), pb = (b_rd ^ cx) + (IMM ? 0 : AT);
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
          asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(ra[kk][tm]) : "v"(pa), "n"(tm * 32 * RB + (IMM ? AT : 0)));
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
          asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(rb[kk][tn]) : "v"(pb), "n"(tn * 32 * RB + (IMM ? AT : 0)));
      }
    };
#pragma unroll
    for (int s = 0; s < NBUF; ++s) issue_loads(s);
    epilogue.start(p, tid, m0, n0);
    wait_and_meet<(NBUF - 1) * LOADS>();
    read_tile(std::integral_constant<int, 0>{}, fa[0], fb[0]);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    auto pstep = [&](auto u_c) {
      constexpr int u = decltype(u_c)::value, set = u & 1;
      wait_and_meet<AHEAD>();
      read_tile(std::integral_constant<int, (u + 1) % NBUF>{}, fa[set ^ 1], fb[set ^ 1]);
      issue_loads(u);
#pragma unroll
      for (int kk = 0; kk < SL; ++kk) multiply(fa[set][kk], fb[set][kk]);
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      // the registers being filled stay theirs until here, also behind the last tile where nobody multiplies them
      hold(fa[set ^ 1]);
      hold(fb[set ^ 1]);
    };
    int kt0 = 0;
    for (; kt0 + NBUF <= nk; kt0 += NBUF) unrolled<NBUF>(pstep);
    unrolled<NBUF - 1>([&](auto u_c) {
      if (kt0 + decltype(u_c)::value < nk) pstep(u_c);
    });
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the zeros behind the last tile: the epilogue uses their place
  } else if constexpr (ROT == 1) {
    // Rotated and interleaved: while the 16-element slice s of a tile is multiplied, slice s+1 is read into the other register set and
    // a part of the direct loads goes out, an instruction or two behind every MFMA, so that nothing but the barrier
    // leaves the matrix pipe without work.  The barrier that hands over tile kt+1 stands in front of tile kt's last slice,
    // which is in registers by then, as is everything else of tile kt: its buffer takes tile kt+NBUF from there on.
    // With two buffers that tile is waited for SL slices later, and what goes out behind the last slices has no time to
    // land: it all goes out behind the first half of them (65 536 x 4096 x 4096 as 256 x 256 1808 us when spread over all
    // four, 1677 over two, 1754 in one; GPT-2's output head at 8192 rows 896, 842, 885; 12 544 x 256 over 1024 as 128 x 128
    // 14.9, 14.0, 14.5).
    constexpr int SL = KS / 16, LOAD_SL = NBUF == 2 ? SL / 2 : SL;
    uint4_t fa[2][TM], fb[2][TN];
    uint32_t a_sl[SL], b_sl[SL];
#pragma unroll
    for (int kk = 0; kk < SL; ++kk) {
      a_sl[kk] = a_rd ^ static_cast<uint32_t>((2 * kk + frag_half) * 16);
      b_sl[kk] = b_rd ^ static_cast<uint32_t>((2 * kk + frag_half) * 16);
    }
    auto read_one = [&](int buf, int kk, int set, int i) {   // operand i (of the TM + TN) of slice kk
      const uint32_t at = buf * BUF_BYTES;
      if (i < TM)
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[set][i]) : "v"(a_sl[kk] + at), "n"(i * 32 * RB));
      else
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[set][i - TM]) : "v"(b_sl[kk] + at), "n"((i - TM) * 32 * RB));
    };
    auto hold_set = [&](int set) {
#pragma unroll
      for (int i = 0; i < TM; ++i) asm volatile("" : "+v"(fa[set][i]));
#pragma unroll
      for (int i = 0; i < TN; ++i) asm volatile("" : "+v"(fb[set][i]));
    };
    // multiplies the slice in `set`; meanwhile slice kk of the tile in `buf` is read into the other set and part `q` of the
    // loads goes to `ld_buf`
    auto slice = [&](auto set_c, auto buf_c, auto kk_c, auto q_c, auto ld_buf_c) {
      constexpr int set = decltype(set_c)::value, buf = decltype(buf_c)::value, kk = decltype(kk_c)::value;
      constexpr int q = decltype(q_c)::value, ld_buf = decltype(ld_buf_c)::value;
      constexpr int READS = TM + TN, FIRST = (q < LOAD_SL ? q : LOAD_SL) * LOADS / LOAD_SL, MF = TM * TN;
      constexpr int AUX = READS + (q < LOAD_SL ? (q + 1) * LOADS / LOAD_SL - FIRST : 0);
      constexpr int PER = (AUX + MF - 1) / MF > 2 ? (AUX + MF - 1) / MF : 2;
      unrolled<MF>([&](auto m_c) {
        constexpr int m = decltype(m_c)::value, tm = m / TN, tn = m % TN;
        acc[tm][tn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, fb[set][tn]),
                                                              __builtin_bit_cast(bf16x8_t, fa[set][tm]), acc[tm][tn], 0, 0, 0);
        unrolled<PER>([&](auto a_c) {
          constexpr int a = m * PER + decltype(a_c)::value;
          if constexpr (a < READS) read_one(buf, kk, set ^ 1, a);
          else if constexpr (a < AUX) issue_load(ld_buf, FIRST + a - READS);
        });
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr (q == LOAD_SL - 1) next_tile();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      hold_set(set ^ 1);
    };
    auto istep = [&](auto u_c) {
      constexpr int u = decltype(u_c)::value, before = (u + NBUF - 1) % NBUF;
      unrolled<SL - 1>([&](auto s_c) {
        constexpr int s = decltype(s_c)::value;
        slice(std::integral_constant<int, (s & 1)>{}, u_c, std::integral_constant<int, s + 1>{}, std::integral_constant<int, s + 1>{},
              std::integral_constant<int, before>{});
      });
      wait_and_meet<AHEAD>();
      slice(std::integral_constant<int, ((SL - 1) & 1)>{}, std::integral_constant<int, (u + 1) % NBUF>{}, std::integral_constant<int, 0>{},
            std::integral_constant<int, 0>{}, u_c);
    };
#pragma unroll
    for (int s = 0; s < NBUF - 1; ++s) issue_loads(s);
#pragma unroll
    for (int j = 0; j < LOADS / LOAD_SL; ++j) issue_load(NBUF - 1, j);
    epilogue.start(p, tid, m0, n0);
    wait_and_meet<AHEAD + LOADS / LOAD_SL>();
#pragma unroll
    for (int i = 0; i < TM + TN; ++i) read_one(0, 0, 0, i);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    hold_set(0);
    int kt0 = 0;
    for (; kt0 + NBUF <= nk; kt0 += NBUF) unrolled<NBUF>(istep);
    unrolled<NBUF - 1>([&](auto u_c) {
      if (kt0 + decltype(u_c)::value < nk) istep(u_c);
    });
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the zeros behind the last tile: the epilogue uses their place
  } else {
#pragma unroll
    for (int s = 0; s < NBUF - 1; ++s)
      if (s < nk) issue_loads(s);
    epilogue.start(p, tid, m0, n0);
    int kt0 = 0;
    for (; kt0 + NBUF <= nk; kt0 += NBUF) {
#pragma unroll
      for (int u = 0; u < NBUF; ++u) step(kt0 + u, u);
    }
#pragma unroll
    for (int u = 0; u < NBUF - 1; ++u)
      if (kt0 + u < nk) step(kt0 + u, u);
  }

  epilogue.finish(p, acc, reinterpret_cast<float*>(lds), tid, m0, n0, tile_m);
}

// ---------------------------------------------------------------------------
// forward / data gradient of a 1x1 layer, bf16, on a persistent grid: a workgroup walks several output tiles
// ---------------------------------------------------------------------------
// igemm2_kernel's interleaved loop (ROT = 1) with the tiles of a workgroup as ONE sequence of reduction steps: the loads of the
// next tile's first steps go out during this tile's last ones, its first operands are read behind this tile's last multiplies,
// and the output leaves straight from the accumulators, so that between two tiles there is neither a trip to memory nor a barrier
// nor LDS taken from the operands.  Over 768 reduction elements (12 steps) that used to be 4 us of a tile's 12.
// Alone, the fastest of the other tilings and 128 x 192 here: 8192 x 2304 over 768 38.4 -> 32.1 us, 8192 x 3072 46.3 -> 40.7 (256 x 128 the
// same), 8192 x 768 13.8 -> 12.5, over 3072 36.4 -> 34.9; 25088 x 768 over 256 20.3 -> 18.7, 6272 x 1536 over 512 18.4 -> 15.9.
// GPT-2 8 x 1024 11.72 -> 11.26 ms, 4 x 1024 7.40 -> 6.90, Swin-B of 32 images 9.85 -> 9.74.
// What bounds it now is power: on operands that are all zeros 8192 x 768 over 3072 takes 28 us, on random ones 38 on the same
// machine.  A fourth LDS tile gained nothing.  fp32 outputs lose here (an output head 790 us as 256 x 256, 842 so).
template <int WM, int WN, int TM, int TN, int NBUF>
__global__ __launch_bounds__(WM* WN * 64) void igemm5_kernel(IgemmArgs p) {
  constexpr int E = 8, KS = kStep2, RB = kRowBytes2, SL = KS / 16;
  constexpr int BM = WM * TM * 32, BN = WN * TN * 32, NW = WM * WN;
  constexpr int A_LD = BM / 8 / NW, B_LD = BN / 8 / NW, LOADS = A_LD + B_LD;   // direct loads (eight rows each) per wave and step
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "tile/loader mismatch");
  constexpr int A_BYTES = BM * RB, BUF_BYTES = A_BYTES + BN * RB;
  // The bias of a wavefront's columns travels with the operands: requested with the first step of a tile, which is up to NBUF
  // tiles ahead of the epilogue that adds it.
  constexpr int BIAS_BYTES = TN * 32 * 4, BIAS_OFF = NBUF * BUF_BYTES;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[BIAS_OFF + NW * (NBUF + 1) * BIAS_BYTES];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int frag_row = lane & 31, frag_half = lane >> 5;
  const int nk = p.gemm_k / KS;
  const int tiles = p.tiles_m * p.tiles_n;
  const int first = static_cast<int>(xcd_remap(blockIdx.x, gridDim.x));

  auto locate = [&](int id, int& m0, int& n0) {   // the order of igemm2_kernel, within every round of workgroups
    const Place at = place_of(p, static_cast<uint32_t>(id));
    m0 = at.tile_m * BM;
    n0 = at.tile_n * BN;
  };

  const __amdgpu_buffer_rsrc_t rsrc_a = make_rsrc(p.a_src, p.a_bytes);
  const __amdgpu_buffer_rsrc_t rsrc_b = make_rsrc(p.b_src, p.b_bytes);
  const __amdgpu_buffer_rsrc_t rsrc_bias = make_rsrc(p.bias, p.bias ? static_cast<uint32_t>(p.gemm_n) * 4u : 0u);

  // ---- the walk of the loads: the lane's rows of tile ld_id, step ld_kt; behind the last tile every offset is out of range ----
  const int sub_row = lane >> 3, slot = lane & 7;
  int a_off[A_LD], b_off[B_LD];
  int ld_id = first, ld_kt = 0, ld_bias = 0;
  auto enter_tile = [&] {
    int m0 = 0, n0 = 0;
    const bool any = ld_id < tiles;
    if (any) locate(ld_id, m0, n0);
#pragma unroll
    for (int j = 0; j < A_LD; ++j) {
      const int trow = (wave * A_LD + j) * 8 + sub_row, row = m0 + trow;
      a_off[j] = any && row < p.gemm_m ? (row * p.gemm_k + (slot ^ ((trow >> 1) & 7)) * E) * 2 : static_cast<int>(kOutOfRange);
    }
#pragma unroll
    for (int j = 0; j < B_LD; ++j) {
      const int trow = (wave * B_LD + j) * 8 + sub_row, row = n0 + trow;
      b_off[j] = any && row < p.gemm_n ? (row * p.gemm_k + (slot ^ ((trow >> 1) & 7)) * E) * 2 : static_cast<int>(kOutOfRange);
    }
    if (p.bias) {
      unsigned char* dst = lds + BIAS_OFF + (wave * (NBUF + 1) + ld_bias) * BIAS_BYTES;
      const int col = n0 + wn * TN * 32 + lane * 4;
      if (lane < TN * 8) load_to_lds(rsrc_bias, dst, any && col < p.gemm_n ? col * 4 : static_cast<int>(kOutOfRange), 0);
      ld_bias = ld_bias == NBUF ? 0 : ld_bias + 1;
    }
  };
  auto issue_load = [&](uint32_t buf, int j) {   // direct load j of the step the walk stands at
    if (j < A_LD)
      load_to_lds(rsrc_a, lds + buf + (wave * A_LD + j) * 1024, a_off[j], ld_kt * RB);
    else
      load_to_lds(rsrc_b, lds + buf + A_BYTES + (wave * B_LD + j - A_LD) * 1024, b_off[j - A_LD], ld_kt * RB);
  };
  auto next_step = [&] {
    if (++ld_kt == nk) {
      ld_kt = 0;
      ld_id += gridDim.x;
      enter_tile();
    }
  };

  f32x16_t acc[TM][TN];
  clear(acc);
  const int swz = (frag_row >> 1) & 7;
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
  const uint32_t a_rd = lds_base + (wm * TM * 32 + frag_row) * RB + swz * 16;
  const uint32_t b_rd = lds_base + A_BYTES + (wn * TN * 32 + frag_row) * RB + swz * 16;
  uint4_t fa[2][TM], fb[2][TN];
  auto read_one = [&](uint32_t pa, uint32_t pb, int set, int i) {   // operand i (of the TM + TN) of a slice
    if (i < TM)
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[set][i]) : "v"(pa), "n"(i * 32 * RB));
    else
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[set][i - TM]) : "v"(pb), "n"((i - TM) * 32 * RB));
  };
  auto hold_set = [&](int set) {
#pragma unroll
    for (int i = 0; i < TM; ++i) asm volatile("" : "+v"(fa[set][i]));
#pragma unroll
    for (int i = 0; i < TN; ++i) asm volatile("" : "+v"(fb[set][i]));
  };
  // as in igemm2_kernel: multiplies the slice in `set`; meanwhile slice kk of the step in `buf` is read into the other set and
  // part `q` of the loads goes to `ld_buf`
  auto slice = [&](auto set_c, uint32_t buf, auto kk_c, auto q_c, uint32_t ld_buf) {
    constexpr int set = decltype(set_c)::value, kk = decltype(kk_c)::value, q = decltype(q_c)::value;
    constexpr int READS = TM + TN, FIRST = q * LOADS / SL, MF = TM * TN;
    constexpr int AUX = READS + (q + 1) * LOADS / SL - FIRST;
    constexpr int PER = (AUX + MF - 1) / MF > 2 ? (AUX + MF - 1) / MF : 2;
    const uint32_t pa = (a_rd ^ static_cast<uint32_t>((2 * kk + frag_half) * 16)) + buf;
    const uint32_t pb = (b_rd ^ static_cast<uint32_t>((2 * kk + frag_half) * 16)) + buf;
    unrolled<MF>([&](auto m_c) {
      constexpr int m = decltype(m_c)::value, tm = m / TN, tn = m % TN;
      acc[tm][tn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, fb[set][tn]),
                                                            __builtin_bit_cast(bf16x8_t, fa[set][tm]), acc[tm][tn], 0, 0, 0);
      unrolled<PER>([&](auto a_c) {
        constexpr int a = m * PER + decltype(a_c)::value;
        if constexpr (a < READS) read_one(pa, pb, set ^ 1, a);
        else if constexpr (a < AUX) issue_load(ld_buf, FIRST + a - READS);
      });
      __builtin_amdgcn_sched_barrier(0);
    });
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    hold_set(set ^ 1);
  };

  // ---- the output: a lane's accumulators are four consecutive columns of one row at a time; two lanes 32 apart exchange every
  // second group so that each stores 16 bytes of bf16 ----
  // The addend of a tile is requested a whole tile ahead (a request behind the last multiply cost 4 us a tile).
  uint2_t add[TM][TN][4];
  const __amdgpu_buffer_rsrc_t rsrc_add = make_rsrc(p.add, static_cast<uint32_t>(p.gemm_m) * p.gemm_n * 2u);
  auto request_add = [&](int id) {
    if (!p.add || id >= tiles) return;
    int m0, n0;
    locate(id, m0, n0);
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int row = m0 + (wm * TM + tm) * 32 + frag_row, col = n0 + (wn * TN + tn) * 32 + 8 * j + 4 * frag_half;
          add[tm][tn][j] = __builtin_amdgcn_raw_buffer_load_b64(
              rsrc_add, row < p.gemm_m && col < p.gemm_n ? (row * p.gemm_n + col) * 2 : static_cast<int>(kOutOfRange), 0, 0);
        }
  };
  int bias_at = 0;
  auto epilogue = [&](int id) {
    int m0, n0;
    locate(id, m0, n0);
    const int col0 = n0 + wn * TN * 32;
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      float bias[16];
      if (p.bias) {
        uint4_t b[4];
        const uint32_t at = lds_base + BIAS_OFF + (wave * (NBUF + 1) + bias_at) * BIAS_BYTES + tn * 128 + frag_half * 16;
#pragma unroll
        for (int j = 0; j < 4; ++j) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(b[j]) : "v"(at), "n"(j * 32));
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          asm volatile("" : "+v"(b[j]));
#pragma unroll
          for (int i = 0; i < 4; ++i) bias[4 * j + i] = __uint_as_float(b[j][i]);
        }
      }
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) {
        const int row = m0 + (wm * TM + tm) * 32 + frag_row;
        float v[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          v[e] = acc[tm][tn][e];
          acc[tm][tn][e] = 0.f;
        }
        if (p.bias) {
#pragma unroll
          for (int e = 0; e < 16; ++e) v[e] += bias[e];
        }
        const int64_t at = static_cast<int64_t>(row) * p.gemm_n + col0 + tn * 32;
        if (p.add) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint2_t u = add[tm][tn][j];
            v[4 * j] += __uint_as_float(u[0] << 16);
            v[4 * j + 1] += __uint_as_float(u[0] & 0xffff0000u);
            v[4 * j + 2] += __uint_as_float(u[1] << 16);
            v[4 * j + 3] += __uint_as_float(u[1] & 0xffff0000u);
          }
        }
#pragma unroll
        for (int j = 0; j < 4; j += 2) {
          const Chunk c = float_to_chunk<bf16>(v + 4 * j);   // words 0, 1: group j; 2, 3: group j + 1
          const auto x = __builtin_amdgcn_permlane32_swap(c.w[0], c.w[2], false, false);
          const auto y = __builtin_amdgcn_permlane32_swap(c.w[1], c.w[3], false, false);
          const int cc = 8 * (j + frag_half);
          if (row < p.gemm_m && col0 + tn * 32 + cc < p.gemm_n)
            *reinterpret_cast<uint4*>(static_cast<bf16*>(p.out) + at + cc) = make_uint4(x[0], y[0], x[1], y[1]);
        }
      }
    }
    bias_at = bias_at == NBUF ? 0 : bias_at + 1;
    return m0 + BM <= p.gemm_m && n0 + BN <= p.gemm_n;   // every lane stored everything
  };

  constexpr int AHEAD = (NBUF - 2) * LOADS;
  constexpr int STORES = TM * TN * 2;   // of a bf16 epilogue, at least
  request_add(first);
  enter_tile();
#pragma unroll
  for (int s = 0; s < NBUF - 1; ++s) {
#pragma unroll
    for (int j = 0; j < LOADS; ++j) issue_load(s * BUF_BYTES, j);
    next_step();
  }
#pragma unroll
  for (int j = 0; j < LOADS / SL; ++j) issue_load((NBUF - 1) * BUF_BYTES, j);
  wait_and_meet<AHEAD + LOADS / SL>();
#pragma unroll
  for (int i = 0; i < TM + TN; ++i) read_one(a_rd ^ static_cast<uint32_t>(frag_half * 16), b_rd ^ static_cast<uint32_t>(frag_half * 16), 0, i);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  hold_set(0);
  uint32_t buf = 0, before = (NBUF - 1) * BUF_BYTES;
  bool stored = false;
  for (int id = first; id < tiles; id += gridDim.x) {
    for (int kt = 0; kt < nk; ++kt) {
      unrolled<SL - 1>([&](auto s_c) {
        constexpr int s = decltype(s_c)::value;
        slice(std::integral_constant<int, (s & 1)>{}, buf, std::integral_constant<int, s + 1>{}, std::integral_constant<int, s + 1>{}, before);
      });
      next_step();
      // behind an epilogue its stores are among the newest requests
      if (stored && kt == 0)
        wait_and_meet<AHEAD + STORES>();
      else
        wait_and_meet<AHEAD>();
      before = buf;
      buf = buf == (NBUF - 1) * BUF_BYTES ? 0 : buf + BUF_BYTES;
      slice(std::integral_constant<int, ((SL - 1) & 1)>{}, buf, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, before);
    }
    stored = epilogue(id);
    request_add(id + gridDim.x);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the zeros behind the last tile land before the LDS goes
}

// ---------------------------------------------------------------------------
// forward / data gradient where the grid of output tiles cannot fill the chip (fp32: where it has fewer than one and a
// half 128 x 128 tiles per compute unit): the reduction is dealt out to the KG wavefronts of a workgroup
// ---------------------------------------------------------------------------
// What bounds it: the trip to memory behind every launch boundary and the chain of steps behind it.  196 x 256 over 2304 (a
// 3x3 layer of one image) 13.2 -> 6.1 us, 784 x 512 over 4608 36.9 -> 14.8, fp32 784 x 256 over 2304 77.6 -> 14.8 against
// 64 x 64 tiles of igemm2_kernel / igemm_kernel; the 151 launches of a ResNet-152 request take 4.4-6.9 us each.
// Every wavefront owns the WHOLE TM*32 x TN*32 tile for every KG-th reduction step and has a ring of NBUF operand
// tiles of its own in LDS, filled with direct loads: nothing is shared before the end, so the main loop has no
// barrier and a wavefront waits for its own loads only.  The partial tiles meet in LDS once and are added in the
// order of the wavefronts.  What this buys where workgroups are few: KG * (NBUF - 1) operand tiles in flight per
// compute unit and a serial chain of nk / KG steps instead of nk.
// A step is one 64-byte LDS row per GEMM row (32 bf16 or 16 fp32 elements), laid out as in igemm2_kernel with
// 32-element steps; in_c must be a multiple of the step.
// FS = 16 (bf16): tiles of 16 x 16 per MFMA, a whole step each.  What bounds a launch that leaves compute units without a workgroup is
// the 77 bytes / ns that direct loads bring into the LDS of one: four times the workgroups load half as many bytes each.
// In a request of one image, 196 rows and 256 channels over 1024 and over 2304: 6.2 us on average on 56 workgroups of 32 x 32, 4.9 on 208;
// 1024 channels over 256, where 224 fill the chip, 4.0 and 6.6 on 832.
// PARTS: an fp32 product on the bf16 pipes (fp32_split.h).
template <typename T, int MODE, int TM, int TN, int KG, int NBUF, int FS = 32, bool PARTS = false>
__global__ __launch_bounds__(KG * 64, 2) void igemm4_kernel(IgemmArgs p) {
  constexpr int E = Elem<T>::kPerChunk;
  constexpr int EB = sizeof(T);
  static_assert(FS == 32 || (FS == 16 && sizeof(T) == 2 && TM == 1 && TN == 1), "the shapes of the multiplies below");
  constexpr int BM = TM * FS, BN = TN * FS;
  constexpr int RB = 64;                 // bytes of one LDS row
  constexpr int KS = RB / EB;            // reduction elements per step
  constexpr int A_LD = BM / 16, B_LD = BN / 16;   // direct loads (sixteen rows each) per step
  constexpr int A_BYTES = BM * RB, BUF_BYTES = (BM + BN) * RB;
  constexpr int NT = KG * 64;
  constexpr int CH = BN / E;
  constexpr int ITEMS = BM * CH;
  constexpr int NTE = ITEMS < NT ? ITEMS : NT;     // threads that store
  constexpr int VISITS = (ITEMS + NT - 1) / NT;
  static_assert(ITEMS % NTE == 0, "epilogue mapping");
  constexpr int LD = BN + kStagePad;
  constexpr int RED_BYTES = KG * BM * LD * 4;
  constexpr int RING_BYTES = KG * NBUF * BUF_BYTES;
  constexpr int LDS_BYTES = RED_BYTES > RING_BYTES ? RED_BYTES : RING_BYTES;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[LDS_BYTES];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // group_rows != 0: consecutive ids (one XCD) walk down the row tiles of one column tile, sharing its filter rows;
  // 0: along the column tiles of one row tile, sharing its activation rows
  uint32_t slow, fast;
  p.div_tiles_n.divmod(xcd_remap(blockIdx.x, gridDim.x), slow, fast);
  const int tile_m = p.group_rows ? fast : slow, tile_n = p.group_rows ? slow : fast;
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  auto row_of = [&](int visit) { return (tid + visit * NT) / CH; };
  EpilogueOperands<T, MODE, VISITS, VISITS> operands;

  const int in_h = (MODE == kFwd) ? p.H : p.Ho;
  const int in_w = (MODE == kFwd) ? p.W : p.Wo;
  const int in_c = (MODE == kFwd) ? p.C : p.K;
  const int cblocks = in_c / KS;
  const int nk = p.R * p.S * cblocks;
  const int sl = p.stride_log2;

  // ---- per lane: the rows it feeds, their byte offset at tap (0,0) and which taps exist ----
  const int sub_row = lane >> 2, slot = lane & 3;
  int a_off[A_LD];
  uint32_t a_taps[A_LD];
#pragma unroll
  for (int j = 0; j < A_LD; ++j) {
    const int trow = j * 16 + sub_row;
    const int chunk = slot ^ ((trow >> 2) & 3);
    const int row = m0 + trow;
    uint32_t taps;
    int base;
    row_taps<MODE>(p, row, in_h, in_w, in_c, base, taps);
    a_off[j] = (base + chunk * E) * EB;
    a_taps[j] = taps;
  }
  int b_off[B_LD];
#pragma unroll
  for (int j = 0; j < B_LD; ++j) {
    const int trow = j * 16 + sub_row;
    const int chunk = slot ^ ((trow >> 2) & 3);
    const int row = n0 + trow;
    b_off[j] = row < p.gemm_n ? (row * p.gemm_k + chunk * E) * EB : static_cast<int>(kOutOfRange);
  }
  const __amdgpu_buffer_rsrc_t rsrc_a = make_rsrc(p.a_src, p.a_bytes);
  const __amdgpu_buffer_rsrc_t rsrc_b = make_rsrc(p.b_src, p.b_bytes);

  // ---- this wavefront's steps: wave, wave + KG, ... as a scalar walk over (tap, channel block) ----
  const int my_steps = nk > wave ? (nk - wave + KG - 1) / KG : 0;
  int ld_kt, ld_t, ld_cb, ld_r, ld_s;
  auto rewind = [&] {
    ld_kt = wave;
    ld_t = wave / cblocks;
    ld_cb = wave - ld_t * cblocks;
    ld_r = ld_t / p.S;
    ld_s = ld_t - ld_r * p.S;
  };
  unsigned char* ring = lds + wave * (NBUF * BUF_BYTES);
  auto issue_loads = [&](int buf) {
    const int tap_elems = (MODE == kFwd) ? (ld_r * in_w + ld_s) * in_c : -((ld_r >> sl) * in_w + (ld_s >> sl)) * in_c;
    const int a_step = (tap_elems + ld_cb * KS) * EB;
    const int b_step = ld_kt * RB;
    unsigned char* dst = ring + buf * BUF_BYTES;
#pragma unroll
    for (int j = 0; j < A_LD; ++j) {
      const bool ok = (a_taps[j] >> ld_t) & 1u;
      load_to_lds(rsrc_a, dst + j * 1024, ok ? a_off[j] + a_step : static_cast<int>(kOutOfRange), 0);
    }
#pragma unroll
    for (int j = 0; j < B_LD; ++j) load_to_lds(rsrc_b, dst + A_BYTES + j * 1024, b_off[j], b_step);
    ld_kt += KG;
    ld_cb += KG;
    while (ld_cb >= cblocks) {
      ld_cb -= cblocks;
      ++ld_t;
      if (++ld_s == p.S) {
        ld_s = 0;
        ++ld_r;
      }
    }
  };

  typedef std::conditional_t<FS == 32, f32x16_t, f32x4_t> acc_t;
  acc_t acc[TM][TN];
  const int frag_row = lane & (FS - 1), frag_half = lane / FS;   // which chunk of a row's slice
  const int swz = (frag_row >> 2) & 3;
  const uint32_t ring_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(ring));
  const uint32_t rd = ring_base + frag_row * RB + swz * 16;
  auto read_frags = [&](int buf, int kk, uint4_t* fa, uint4_t* fb) {
    const uint32_t pa = (rd ^ static_cast<uint32_t>((2 * kk + frag_half) * 16)) + buf * BUF_BYTES;
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[tm]) : "v"(pa), "n"(tm * FS * RB));
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[tn]) : "v"(pa), "n"(A_BYTES + tn * FS * RB));
  };
  auto hold_frags = [&](uint4_t* fa, uint4_t* fb) {
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) asm volatile("" : "+v"(fa[tm]));
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) asm volatile("" : "+v"(fb[tn]));
  };
  auto chunk = [](const uint4_t& v) {
    Chunk c;
    c.h = __builtin_bit_cast(bf16x8_t, v);
    return c;
  };
  auto multiply = [&](uint4_t* fa, uint4_t* fb) {
    hold_frags(fa, fb);
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) {
        const Chunk a = chunk(fa[tm]), b = chunk(fb[tn]);
        if constexpr (FS == 32)
          mma<T>(b, a, acc[tm][tn]);
        else
          acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b.h, a.h, acc[tm][tn], 0, 0, 0);
      }
  };

  // The tile of step i lands when at most the NBUF-2 tiles requested behind it are outstanding (near the end fewer
  // follow: wait for everything).  The reads of step i-1 were waited for before its multiplies, so its buffer is free.
  constexpr int AHEAD = (NBUF - 2) * (A_LD + B_LD);
  static_assert(AHEAD < 64, "vmcnt range");
  // this wavefront's share of the sums, in `acc`; split_c: in fp32, on the bf16 pipes, small products in `low`
  // The epilogue's operands are requested behind the first loads, except beside the 128 accumulators of a 64 x 64 tile in parts, where there
  // are no registers for them.
  constexpr bool EARLY = !(PARTS && TM * TN == 4);
  auto request_operands = [&] { operands.template request_first<BN, NTE>(p, tid, m0, n0, row_of); };
  auto reduce = [&](auto split_c, acc_t (&low)[TM][TN], bool request) {
    constexpr bool SPLIT = decltype(split_c)::value;
    rewind();
    if constexpr (FS == 16) {
      acc[0][0] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    } else {
      clear(acc);
      if constexpr (SPLIT) clear(low);
    }
    auto step = [&](int i, int buf) {
      if (i + NBUF - 1 <= my_steps)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AHEAD) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (i + NBUF - 1 < my_steps) issue_loads((buf + NBUF - 1) % NBUF);
      uint4_t fa0[TM], fb0[TN], fa1[TM], fb1[TN];
      read_frags(buf, 0, fa0, fb0);
      if constexpr (FS == 16) {   // the whole step is one operand
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        multiply(fa0, fb0);
      } else {
        read_frags(buf, 1, fa1, fb1);
        if constexpr (SPLIT) {
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          hold_frags(fa0, fb0);
          hold_frags(fa1, fb1);
          Split8 sb[TN];
#pragma unroll
          for (int tn = 0; tn < TN; ++tn) sb[tn] = split8(chunk(fb0[tn]), chunk(fb1[tn]));
#pragma unroll
          for (int tm = 0; tm < TM; ++tm) {
            const Split8 sa = split8(chunk(fa0[tm]), chunk(fa1[tm]));
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) mma_split(sb[tn], sa, acc[tm][tn], low[tm][tn]);
          }
        } else {
          asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(TM + TN) : "memory");
          multiply(fa0, fb0);
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          multiply(fa1, fb1);
        }
      }
    };
#pragma unroll
    for (int i = 0; i < NBUF - 1; ++i)
      if (i < my_steps) issue_loads(i);
    if (request) request_operands();
    int i0 = 0;
    for (; i0 + NBUF <= my_steps; i0 += NBUF) {
#pragma unroll
      for (int u = 0; u < NBUF; ++u) step(i0 + u, u);
    }
#pragma unroll
    for (int u = 0; u < NBUF - 1; ++u)
      if (i0 + u < my_steps) step(i0 + u, u);
  };
  if constexpr (PARTS) {
    f32x16_t low[TM][TN];
    reduce(std::true_type{}, low, EARLY);
    if (__any(join_split(acc, low))) reduce(std::false_type{}, low, false);
    if constexpr (!EARLY) request_operands();
  } else {
    reduce(std::false_type{}, acc, true);
  }

  // ---- the partial tiles meet: [wave][BM][LD] fp32, over the rings ----
  float* red = reinterpret_cast<float*>(lds);
  finish_walk<T, MODE, BN, NTE, NT, VISITS, VISITS, LDS_BYTES>(
      p, operands, red, tid, m0, n0, tile_m, row_of, [&](auto fin) {
        __syncthreads();   // every wavefront is done with its ring
        float* mine = red + wave * (BM * LD);
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
          for (int tn = 0; tn < TN; ++tn)
#pragma unroll
            for (int j = 0; j < (FS == 32 ? 4 : 1); ++j)
              *reinterpret_cast<float4*>(mine + (tm * FS + frag_row) * LD + tn * FS + 8 * j + 4 * frag_half) =
                  make_float4(acc[tm][tn][4 * j], acc[tm][tn][4 * j + 1], acc[tm][tn][4 * j + 2], acc[tm][tn][4 * j + 3]);
        __syncthreads();
        if (NTE < NT && tid >= NTE) return;
#pragma unroll
        for (int visit = 0; visit < VISITS; ++visit) {
          const int q = tid + visit * NT;
          const int r = q / CH, c = (q - r * CH) * E;
          float v[E];
#pragma unroll
          for (int e = 0; e < E; ++e) v[e] = 0.f;
#pragma unroll
          for (int g = 0; g < KG; ++g)
#pragma unroll
            for (int e = 0; e < E; e += 4) {
              const float4 t = *reinterpret_cast<const float4*>(red + (g * BM + r) * LD + c + e);
              v[e] += t.x;
              v[e + 1] += t.y;
              v[e + 2] += t.z;
              v[e + 3] += t.w;
            }
          fin(visit, r, c, v);
        }
      });
}

// ---------------------------------------------------------------------------
// 3x3, stride 1, pad 1 (forward and data gradient), 32*WM x 64*TN tile: the activation side of the nine
// taps of a channel block is ONE patch in LDS.  The output pixels of a tile are consecutive in the
// flattened (image, row, column) order, and the input pixel of tap (r, s) lies (r-1)*W + (s-1) places
// further in the same order, so the patch is the contiguous range of pixels from W+1 before the tile to
// W+1 behind it (32*WM + 2W + 2 rows of 64 channels), loaded once per channel block instead of nine
// shifted copies of the tile.  A tap that falls outside its image (the zero padding) reads a row of
// zeros kept in LDS instead.  The filter tiles stream per (channel block, tap), NBUF of them in LDS; the
// patch of the next channel block is requested one load per tap, so that no step waits for all of it.
// The reduction runs channel block by channel block (taps innermost), so sums round differently from
// igemm2_kernel's tap-major order.
//
// What bounds it is the operand path into LDS where workgroups share a CU (a patch takes a third of igemm2's
// bytes for the activations) and the latency of a filter tile where one stands alone (with nine of them in
// LDS the loads run a whole channel block ahead).  A wavefront's reads, loads and multiplies are interleaved
// slice by slice as in igemm2's tilings of eight wavefronts; before, all reads of a step stood in front of its
// multiplies.  Warm, 7x7 of 64 images, 512 channels: 27.0 -> 20.5 us; in place, 14x14 of 16 images, 256
// channels: forward 16.4 -> 14.1, data gradient with sums 17.7 -> 14.6.
// ---------------------------------------------------------------------------
// Of the `steps` steps up to the one with tap `tap`, how many request a load of the next patch in this channel block.  (Those of the
// block before do not count: the first block has none before it, whose patch is older than every filter.)
template <int P_LD>
constexpr int patch_loads_among(int tap, int steps) {
  int n = 0;
  for (int i = 0; i < steps && i <= tap; ++i) n += tap - i < P_LD ? 1 : 0;
  return n;
}

template <int MODE, int WM, int TN, int P_LD, int NBUF>
__global__ __launch_bounds__(WM * 128) void igemm3_kernel(IgemmArgs p) {
  using T = bf16;
  constexpr int E = 8, WN = 2, NW = WM * WN;
  constexpr int BM = WM * 32, BN = WN * TN * 32;
  constexpr int B_LD = BN / 8 / NW;
  constexpr int PATCH_BYTES = P_LD * NW * 8 * kRowBytes2, B_BYTES = BN * kRowBytes2;
  constexpr int B_OFF = 2 * PATCH_BYTES, ZERO_OFF = B_OFF + NBUF * B_BYTES;
  constexpr int STAGE_BYTES = WM * 32 * (BN + kStagePad) * 4;
  constexpr int LDS_BYTES = ZERO_OFF + kRowBytes2 > STAGE_BYTES ? ZERO_OFF + kRowBytes2 : STAGE_BYTES;
  static_assert(9 % NBUF == 0, "the buffer of a step is a constant of its tap");
  static_assert(P_LD <= 9, "the next patch is requested, a load per step");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[LDS_BYTES];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  uint32_t tile_m, tile_n;
  p.div_tiles_n.divmod(xcd_remap(blockIdx.x, gridDim.x), tile_m, tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;

  const int in_c = (MODE == kFwd) ? p.C : p.K;
  const int cblocks = in_c / kStep2;
  const int W = p.W, H = p.H, halo = W + 1;

  // ---- loaders: patch rows (wave * P_LD + j) * 8 + lane / 8, filter rows as in igemm2_kernel ----
  const int sub_row = lane >> 3, slot = lane & 7;
  int p_off[P_LD];
#pragma unroll
  for (int j = 0; j < P_LD; ++j) {
    const int prow = (wave * P_LD + j) * 8 + sub_row;
    const int chunk = slot ^ ((prow >> 1) & 7);
    const int grow = m0 - halo + prow;
    const bool ok = grow >= 0 && grow < p.gemm_m && prow < BM + 2 * halo;
    p_off[j] = ok ? (grow * in_c + chunk * E) * 2 : static_cast<int>(kOutOfRange);
  }
  int b_off[B_LD];
#pragma unroll
  for (int j = 0; j < B_LD; ++j) {
    const int trow = (wave * B_LD + j) * 8 + sub_row;
    const int chunk = slot ^ ((trow >> 1) & 7);
    const int row = n0 + trow;
    b_off[j] = row < p.gemm_n ? (row * p.gemm_k + chunk * E) * 2 : static_cast<int>(kOutOfRange);
  }
  const __amdgpu_buffer_rsrc_t rsrc_a = make_rsrc(p.a_src, p.a_bytes);
  const __amdgpu_buffer_rsrc_t rsrc_b = make_rsrc(p.b_src, p.b_bytes);
  // Every wavefront makes every request (the waits count them): behind the last channel block zeros land.
  auto issue_patch = [&](int cb, int j) {
    const int beyond = cb < cblocks ? 0 : static_cast<int>(kOutOfRange);
    load_to_lds(rsrc_a, lds + (cb & 1) * PATCH_BYTES + (wave * P_LD + j) * 1024, p_off[j] | beyond, cb * kRowBytes2);
  };
  auto issue_filter = [&](int cb, int tap, int buf, int j) {
    const int beyond = cb < cblocks ? 0 : static_cast<int>(kOutOfRange);
    load_to_lds(rsrc_b, lds + B_OFF + buf * B_BYTES + (wave * B_LD + j) * 1024, b_off[j] | beyond, (tap * in_c + cb * kStep2) * 2);
  };
  // Requests leave in this order: patch 0, filters 0 .. NBUF-2, the first load of filter NBUF-1.  Then, in step kt with tap t: the other
  // loads of filter kt + NBUF-1 behind the multiplies of slice 0, one load of the next channel block's patch (t < P_LD) behind those of
  // slice 1, and the first load of filter kt + NBUF behind those of the last slice, whose barrier has freed the buffer of filter kt.
  // (The row of zeros first: the compiler keeps an LDS store behind every direct load.)
  if (tid < 8) *reinterpret_cast<uint4*>(lds + ZERO_OFF + tid * 16) = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
  for (int j = 0; j < P_LD; ++j) issue_patch(0, j);
#pragma unroll
  for (int t = 0; t < NBUF - 1; ++t)
#pragma unroll
    for (int j = 0; j < B_LD; ++j) issue_filter(0, t, t, j);
  issue_filter(0, NBUF - 1, NBUF - 1, 0);
  TileEpilogue<T, MODE, WM, WN, 1, TN, true> epilogue;
  epilogue.start(p, tid, m0, n0);

  // ---- the row this lane feeds to the MFMAs and which of its nine taps lie inside the image ----
  const int frag_row = lane & 31, frag_half = lane >> 5;
  uint32_t taps = 0;
  {
    const int row = m0 + wm * 32 + frag_row;
    if (row < p.gemm_m) {
      uint32_t img, pix, oh, ow, cols = 0;
      p.div_plane.divmod(static_cast<uint32_t>(row), img, pix);
      p.div_width.divmod(pix, oh, ow);
#pragma unroll
      for (int s2 = 0; s2 < 3; ++s2) {
        const int iw = (MODE == kFwd) ? static_cast<int>(ow) + s2 - 1 : static_cast<int>(ow) + 1 - s2;
        if (static_cast<unsigned>(iw) < static_cast<unsigned>(W)) cols |= 1u << s2;
      }
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        const int ih = (MODE == kFwd) ? static_cast<int>(oh) + r - 1 : static_cast<int>(oh) + 1 - r;
        if (static_cast<unsigned>(ih) < static_cast<unsigned>(H)) taps |= cols << (r * 3);
      }
    }
  }

  f32x16_t acc[1][TN];
  clear(acc);
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
  const uint32_t b_rd = lds_base + B_OFF + (wn * TN * 32 + frag_row) * kRowBytes2 + ((frag_row >> 1) & 7) * 16;
  // LDS address of this lane's patch row for a tap (slot swizzle of that row included), or of the row of zeros
  auto patch_row = [&](int cb, int tap) {
    const int r = tap / 3, s2 = tap - 3 * r;
    const int tapoff = (MODE == kFwd) ? r * W + s2 : (2 - r) * W + (2 - s2);
    const uint32_t prow = static_cast<uint32_t>(wm * 32 + frag_row + tapoff);
    const uint32_t in_patch = lds_base + (cb & 1) * PATCH_BYTES + prow * kRowBytes2 + ((prow >> 1) & 7) * 16;
    return ((taps >> tap) & 1u) ? in_patch : lds_base + ZERO_OFF;
  };
  uint4_t fa[2], fb[2][TN];
  auto read_one = [&](uint32_t pa, uint32_t pb, int set, int i) {   // operand i (of the 1 + TN) of a slice
    if (i == 0)
      asm volatile("ds_read_b128 %0, %1" : "=v"(fa[set]) : "v"(pa));
    else
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[set][i - 1]) : "v"(pb), "n"((i - 1) * 32 * kRowBytes2));
  };
  auto hold_set = [&](int set) {
    asm volatile("" : "+v"(fa[set]));
#pragma unroll
    for (int i = 0; i < TN; ++i) asm volatile("" : "+v"(fb[set][i]));
  };
  // Multiplies the slice in `set`; meanwhile slice kk of the step with patch row `row` and filter buffer `buf` is read into the other
  // set, and `request` runs behind the last of these.
  auto slice = [&](auto set_c, uint32_t row, auto buf_c, auto kk_c, auto request) {
    constexpr int set = decltype(set_c)::value, kk = decltype(kk_c)::value;
    const uint32_t cx = (2 * kk + frag_half) * 16;
    const uint32_t pa = row ^ cx, pb = (b_rd ^ cx) + decltype(buf_c)::value * B_BYTES;
    unrolled<TN>([&](auto m_c) {
      constexpr int m = decltype(m_c)::value;
      acc[0][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, fb[set][m]), __builtin_bit_cast(bf16x8_t, fa[set]),
                                                          acc[0][m], 0, 0, 0);
      constexpr int PER = 2;
      unrolled<PER>([&](auto a_c) {
        constexpr int a = m * PER + decltype(a_c)::value;
        if constexpr (a < 1 + TN) read_one(pa, pb, set ^ 1, a);
      });
      if constexpr (m == TN - 1) request();
      __builtin_amdgcn_sched_barrier(0);
    });
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    hold_set(set ^ 1);
  };

  wait_and_meet<(NBUF - 2) * B_LD + 1>();   // patch 0 and filter 0
  uint32_t row = patch_row(0, 0);
#pragma unroll
  for (int i = 0; i < 1 + TN; ++i)
    read_one(row ^ static_cast<uint32_t>(frag_half * 16), b_rd ^ static_cast<uint32_t>(frag_half * 16), 0, i);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  hold_set(0);
  for (int cb = 0; cb < cblocks; ++cb) {
    unrolled<9>([&](auto t_c) {
      constexpr int tap = decltype(t_c)::value, u = tap % NBUF;
      using std::integral_constant;
      constexpr int ahead = (tap + NBUF - 1) % 9, ahead1 = (tap + NBUF) % 9;
      const int cb_ahead = cb + (tap + NBUF - 1) / 9, cb_ahead1 = cb + (tap + NBUF) / 9;
      slice(integral_constant<int, 0>{}, row, integral_constant<int, u>{}, integral_constant<int, 1>{}, [&] {
#pragma unroll
        for (int j = 1; j < B_LD; ++j) issue_filter(cb_ahead, ahead, (u + NBUF - 1) % NBUF, j);
      });
      slice(integral_constant<int, 1>{}, row, integral_constant<int, u>{}, integral_constant<int, 2>{}, [&] {
        if constexpr (tap < P_LD) issue_patch(cb + 1, tap);
      });
      slice(integral_constant<int, 0>{}, row, integral_constant<int, u>{}, integral_constant<int, 3>{}, [&] {});
      // Filter kt + 1 has landed when only what was requested behind it is outstanding: filters kt + 2 .. kt + NBUF-1 and the loads
      // of the next patch in this step and the NBUF-2 before it.  In front of the next channel block its patch has to be there as well,
      // whose last load has the filter loads of 9 - P_LD steps behind it.
      constexpr int newer = (NBUF - 2) * B_LD + patch_loads_among<P_LD>(tap, NBUF - 1);
      wait_and_meet<tap == 8 ? std::min(newer, (9 - P_LD) * B_LD) : newer>();
      row = patch_row(tap == 8 ? cb + 1 : cb, (tap + 1) % 9);
      slice(integral_constant<int, 1>{}, row, integral_constant<int, (u + 1) % NBUF>{}, integral_constant<int, 0>{},
            [&] { issue_filter(cb_ahead1, ahead1, u, 0); });
    });
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the zeros behind the last tile: the epilogue uses their place
  epilogue.finish(p, acc, reinterpret_cast<float*>(lds), tid, m0, n0, tile_m);
}

__device__ __forceinline__ void splitk_reduce_body(const ReduceArgs& p, uint32_t block) {
  if (block >= p.first_blocks) {
    const int i = (block - p.first_blocks) * 256 + threadIdx.x;
    if (i >= p.n2) return;
    float s = 0.f;
    constexpr int U2 = 8;
    for (int k0 = 0; k0 < p.splits; k0 += U2) {
      float v[U2];
#pragma unroll
      for (int u = 0; u < U2; ++u) v[u] = p.partial2[static_cast<int64_t>(k0 + u < p.splits ? k0 + u : p.splits - 1) * p.n2 + i];
#pragma unroll
      for (int u = 0; u < U2; ++u)
        if (k0 + u < p.splits) s += v[u];
    }
    p.out2[i] = p.accumulate ? p.out2[i] + s : s;
    return;
  }
  int64_t i = (static_cast<int64_t>(block) * 256 + threadIdx.x) * 4;
  if (i >= p.n) return;
  // Eight partials are requested before any is added (a request past the last split repeats it and does not
  // count): the kernel costs its dependent round trips to memory, one per trip here instead of one per split.
  // The additions keep the order of the splits.
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  constexpr int U = 8;
  for (int k0 = 0; k0 < p.splits; k0 += U) {
    float4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u < p.splits ? k0 + u : p.splits - 1;
      v[u] = *reinterpret_cast<const float4*>(p.partial + static_cast<int64_t>(k) * p.n + i);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (k0 + u < p.splits) {
        s.x += v[u].x;
        s.y += v[u].y;
        s.z += v[u].z;
        s.w += v[u].w;
      }
  }
  float4* o = reinterpret_cast<float4*>(p.out + i);
  if (p.accumulate) {
    float4 c = *o;
    s.x += c.x;
    s.y += c.y;
    s.z += c.z;
    s.w += c.w;
  }
  *o = s;
}

__global__ __launch_bounds__(256) void splitk_reduce_kernel(ReduceArgs p) { splitk_reduce_body(p, blockIdx.x); }

// The split reductions of several weight gradients in one launch (table / map as in wgrad_group_kernel).
struct ReduceGroupArgs {
  const ReduceArgs* table;
  const uint2* map;
};

__global__ __launch_bounds__(256) void splitk_reduce_group_kernel(ReduceGroupArgs g) {
  const uint2 e = g.map[blockIdx.x];
  const ReduceArgs p = g.table[__builtin_amdgcn_readfirstlane(e.x)];
  splitk_reduce_body(p, __builtin_amdgcn_readfirstlane(e.y));
}

int ilog2_exact(int v) {
  int l = 0;
  while ((1 << l) < v) ++l;
  return ((1 << l) == v) ? l : -1;
}

template <typename T, int MODE, int WM, int WN, int TM, int TN, bool PARTS = false>
const char* igemm_name() {
  static const std::string name = std::string(MODE == kWgrad ? "wgrad_kernel<" : "igemm_kernel<") +
                                  (sizeof(T) == 2 ? "bf16" : "f32") + "," +
                                  (MODE == kFwd ? "fwd," : MODE == kDgrad ? "dgrad," : "") +
                                  std::to_string(WM * TM * 32) + "x" + std::to_string(WN * TN * 32) + (PARTS ? ",parts>" : ">");
  return name.c_str();
}

// Algorithmic bytes of one convolution launch: each operand read once, the result written once (the partial
// results of a split reduction are the kernel's own choice and do not count).  Many of these layers do fewer
// flops per byte than the chip can feed, so the profiler is told the bytes beside the flops.
template <int MODE>
double conv_bytes(const IgemmArgs& a, int eb) {
  const double x = static_cast<double>(a.N) * a.H * a.W * a.C, y = static_cast<double>(a.N) * a.Ho * a.Wo * a.K;
  const double w = static_cast<double>(a.K) * a.R * a.S * a.C;
  if (MODE == kWgrad) return (x + y) * eb + w * 4;
  const double out = MODE == kFwd ? y : x;
  const int extra = (a.add ? 1 : 0) + (a.add && a.mask ? 1 : 0) + (a.bn_x ? 1 : 0) + (a.bn_mask ? 1 : 0);
  return ((MODE == kFwd ? x : y) + w + out * extra) * eb + out * (a.out_f32 ? 4 : eb);
}

// what the kernels divide by on their way to the first load; tiles_m, tiles_n and group_rows are set
void bind_divisions(IgemmArgs& a, int run) {
  a.div_tiles_n = FastDiv(run);
  a.div_group = FastDiv(static_cast<uint32_t>(a.group_rows > 1 ? a.group_rows : a.tiles_m) * a.tiles_n);
  a.div_rows = FastDiv(a.group_rows > 1 ? a.group_rows : 1);
  a.div_c = FastDiv(a.C);
  a.div_s = FastDiv(a.S);
}

// Which fp32 products go through the bf16 pipes (fp32_split.h); the others are multiplied in fp32 by kernels that hold nothing else.
// What decides is whether a SIMD has a second wavefront: taking operands apart does not pass behind a wavefront's own
// multiplies, but behind those of another one.  Then, how many of its instructions a multiply costs.  Times alone in parts as shares of those
// in fp32, over the layers of the three models at 64-8192 rows and 1-32 images (244 forward products and data gradients, 122 weight
// gradients):
//   128 x 128 tiles 0.84-1.00, 128 x 64 0.88-0.98, 64 x 64 split over wavefronts 0.74-0.91 (one wavefront on a SIMD: 1.05-1.10)
//   64 x 32 over 512 - 8192: 0.85-1.00.  Over 16384 and more 0.97-1.07 (2331 x 768: 1.01, over 50304 1.07; 2048 x 768 over that 0.87)
//   32 x 32 over eight wavefronts, K >= 1024: 0.94-1.00 (1.04 once); over four, less than 512 1.00-1.03, one wavefront on a SIMD 1.00-1.20
//   weight gradients: 128 x 128, which have four workgroups on a CU, 0.80-0.90; 64 x 64 with more than one 0.89-1.00, up to four reduction
//   steps 1.01-1.07; else 0.97-1.09
// Data gradients run beside weight gradients, whose work fills what a second wavefront leaves.  Steps with tiles below 64 x 64 in parts
// for both / for forward products only: ResNet-152 of 16 images 17.40 / 17.05 ms, Swin-B of 2 images 6.34 / 6.24 (fp32 multiplies 17.2, 6.26),
// the other steps the same; 32 x 32 tiles over four wavefronts forward: GPT-2 of 2 x 256 5.97 / 5.89 without.
// Never: what was asked for front to back (every tile adds up the same bits), and a convolution whose output a training BatchNorm takes.  Behind
// it stands a ReLU, and whichever of two equally good roundings a pre-activation gets near zero, another one opens or closes gates, each
// of which moves a gradient by more than all other rounding does (ResNet-152 of 4 images, the gradients against those of fp32
// multiplies: 2e-7 relative without a gate, 7.5e-5 with two).  Data and weight gradients are smooth.
template <typename T, int MODE, int BM, int BN, int KG>
constexpr bool parts_tile() {   // KG: wavefronts a reduction is split over (1: igemm_kernel, whose 64 x 64 tiles take two operands apart per product)
  return sizeof(T) == 4 && (BM * BN > 64 * 64 || (KG > 1 && (BM * BN == 64 * 64 || (MODE == kFwd && (BM > 32 || KG == 8)))));
}
template <int MODE, int BM, int BN>
bool product_in_parts(const IgemmArgs& a, int64_t wavefronts) {
  if (a.in_fp32 || (MODE == kFwd && (a.stats || a.stat_acc))) return false;
  const int from = BM * BN == 32 * 32 ? 1024 : 256, to = BM * BN == 64 * 32 ? 16384 : INT_MAX;
  return wavefronts > 4 * 256 && a.gemm_k >= from && a.gemm_k < to;
}
bool wgrad_in_parts(const IgemmArgs& a, int64_t workgroups) { return workgroups > 256 && a.k_per_split > 4 * 16; }

template <int WM, int WN, int TM, int TN, int RING>
void (*wgrad_direct_kernel(const IgemmArgs& a))(WgradArgs) {
  if (a.pointwise) return a.dbias ? wgrad_kernel<WM, WN, TM, TN, RING, true, true> : wgrad_kernel<WM, WN, TM, TN, RING, true, false>;
  return a.dbias ? wgrad_kernel<WM, WN, TM, TN, RING, false, true> : wgrad_kernel<WM, WN, TM, TN, RING, false, false>;
}

template <typename T, int MODE, int WM, int WN, int TM, int TN>
int launch_cfg(Context* ctx, IgemmArgs& a, double flops) {
  constexpr int BM = WM * TM * 32, BN = WN * TN * 32;
  a.tiles_m = (a.gemm_m + BM - 1) / BM;
  a.tiles_n = (a.gemm_n + BN - 1) / BN;
  int64_t wgs = static_cast<int64_t>(a.tiles_m) * a.tiles_n * a.splits;
  if (wgs <= 0 || wgs > 0x7fffffff) {
    set_error("igemm: grid out of range");
    return -22;
  }
  a.group_rows = 0;
  bind_divisions(a, a.tiles_n);
  const dim3 grid(static_cast<unsigned>(wgs)), block(WM * WN * 64);
  if constexpr (MODE == kWgrad) {
    static_assert(WM * WN * 64 == 256, "the split reduction that may ride along is written for 256 threads");
    WgradArgs w{};
    w.a = a;
    w.gemm_wgs = static_cast<uint32_t>(wgs);
    double bytes = conv_bytes<MODE>(a, sizeof(T));
    auto& tr = ctx->trailing_reduce;
    unsigned blocks = grid.x;
    if (a.take_pending && tr.valid) {
      // the launch keeps its own algorithmic bytes (operands once, the filter gradient once): the partial filters
      // the extra workgroups read are traffic, not work
      w.red = tr.args;
      w.red_blocks = tr.blocks;
      blocks += tr.blocks;
      tr.valid = false;
    }
    auto& cs = ctx->trailing_col_sum;
    if (a.take_pending && cs.valid) {
      w.cols = cs.args;
      blocks += (cs.args.C + 7) / 8;
      cs.valid = false;
    }
    void (*kernel)(WgradArgs);
    const char* name = igemm_name<T, MODE, WM, WN, TM, TN>();
    if constexpr (sizeof(T) == 4) {
      const bool parts = wgrad_in_parts(a, wgs);
      kernel = parts ? wgrad_f32_kernel<WM, WN, TM, TN, true> : wgrad_f32_kernel<WM, WN, TM, TN, false>;
      if (parts) name = igemm_name<T, MODE, WM, WN, TM, TN, true>();
    } else if (TM * TN == 1 && short_wgrad_ring(wgs, (a.k_per_split + 31) / 32))
      kernel = wgrad_direct_kernel<WM, WN, TM, TN, TM * TN == 1 ? kWgradShortRing : kWgradRing>(a);
    else
      kernel = wgrad_direct_kernel<WM, WN, TM, TN, kWgradRing>(a);
    return launch(ctx, kernel, dim3(blocks), block, w, name, flops, 0, bytes);
  } else {
    const char* name = igemm_name<T, MODE, WM, WN, TM, TN>();
    const double bytes = conv_bytes<MODE>(a, sizeof(T));
    if constexpr (parts_tile<T, MODE, BM, BN, 1>())
      if (product_in_parts<MODE, BM, BN>(a, wgs * 4))
        return launch(ctx, igemm_kernel<T, MODE, WM, WN, TM, TN, true>, grid, block, a, igemm_name<T, MODE, WM, WN, TM, TN, true>(), flops, 0, bytes);
    return launch(ctx, igemm_kernel<T, MODE, WM, WN, TM, TN>, grid, block, a, name, flops, 0, bytes);
  }
}

template <int MODE, int WM, int WN, int TM, int TN, int NBUF, int ROT = 0, int KS = kStep2>
int launch_cfg2(Context* ctx, IgemmArgs& a, double flops) {
  constexpr int BM = WM * TM * 32, BN = WN * TN * 32;
  static const std::string name = std::string("igemm2_kernel<bf16,") + (MODE == kFwd ? "fwd," : "dgrad,") +
                                  std::to_string(BM) + "x" + std::to_string(BN) + "," + std::to_string(NBUF) + "buf" +
                                  (WM * WN == 8 ? ",8w" : "") + (KS == 32 ? ",k32" : "") + (ROT == 1 ? ",rot>" : ROT == 2 ? ",pipe>" : ">");
  a.tiles_m = (a.gemm_m + BM - 1) / BM;
  a.tiles_n = (a.gemm_n + BN - 1) / BN;
  static const int group_env = [] {
    const char* e = getenv("TCH_IGEMM_GROUP_ROWS");
    return e ? atoi(e) : -1;
  }();
  a.group_rows = group_env >= 0 ? group_env : (a.tiles_n > 8 ? 4 : 0);
  int64_t wgs = static_cast<int64_t>(a.tiles_m) * a.tiles_n;
  if (wgs <= 0 || wgs > 0x7fffffff) {
    set_error("igemm: grid out of range");
    return -22;
  }
  bind_divisions(a, a.tiles_n);
  return launch(ctx, igemm2_kernel<MODE, WM, WN, TM, TN, NBUF, ROT, KS>, dim3(static_cast<unsigned>(wgs)), dim3(WM * WN * 64), a,
                name.c_str(), flops, 0, conv_bytes<MODE>(a, 2));
}

template <int MODE, int WM, int WN, int TM, int TN, int NBUF>
int launch_cfg5(Context* ctx, IgemmArgs& a, double flops) {
  constexpr int BM = WM * TM * 32, BN = WN * TN * 32;
  static const std::string name = std::string("igemm5_kernel<bf16,") + (MODE == kFwd ? "fwd," : "dgrad,") + std::to_string(BM) + "x" +
                                  std::to_string(BN) + "," + std::to_string(NBUF) + "buf,persistent>";
  a.tiles_m = (a.gemm_m + BM - 1) / BM;
  a.tiles_n = (a.gemm_n + BN - 1) / BN;
  a.group_rows = a.tiles_n > 8 ? 4 : 0;
  const int64_t tiles = static_cast<int64_t>(a.tiles_m) * a.tiles_n;
  if (tiles <= 0 || tiles > 0x3fffffff) {
    set_error("igemm: grid out of range");
    return -22;
  }
  bind_divisions(a, a.tiles_n);
  return launch(ctx, igemm5_kernel<WM, WN, TM, TN, NBUF>, dim3(static_cast<unsigned>(std::min<int64_t>(tiles, 256))), dim3(WM * WN * 64), a,
                name.c_str(), flops, 0, conv_bytes<MODE>(a, 2));
}

template <typename T, int MODE, int TM, int TN, int KG, int NBUF, int FS = 32>
int launch_cfg4(Context* ctx, IgemmArgs& a, double flops) {
  constexpr int BM = TM * FS, BN = TN * FS;
  static const std::string name = std::string("igemm4_kernel<") + (sizeof(T) == 2 ? "bf16," : "f32,") +
                                  (MODE == kFwd ? "fwd," : "dgrad,") + std::to_string(BM) + "x" + std::to_string(BN) + "," +
                                  std::to_string(KG) + "way," + std::to_string(NBUF) + "buf>";
  static const std::string parts_name = name.substr(0, name.size() - 1) + ",parts>";
  a.tiles_m = (a.gemm_m + BM - 1) / BM;
  a.tiles_n = (a.gemm_n + BN - 1) / BN;
  const int64_t wgs = static_cast<int64_t>(a.tiles_m) * a.tiles_n;
  if (wgs <= 0 || wgs > 0x7fffffff) {
    set_error("igemm: grid out of range");
    return -22;
  }
  // the larger operand is the one an XCD should fetch once
  a.group_rows = static_cast<int64_t>(a.gemm_n) * a.gemm_k > static_cast<int64_t>(a.a_bytes / sizeof(T)) ? 1 : 0;
  bind_divisions(a, a.group_rows ? a.tiles_m : a.tiles_n);
  const dim3 grid(static_cast<unsigned>(wgs)), block(KG * 64);
  const double bytes = conv_bytes<MODE>(a, sizeof(T));
  if constexpr (parts_tile<T, MODE, BM, BN, KG>())
    if (product_in_parts<MODE, BM, BN>(a, wgs * KG))
      return launch(ctx, igemm4_kernel<T, MODE, TM, TN, KG, NBUF, FS, true>, grid, block, a, parts_name.c_str(), flops, 0, bytes);
  return launch(ctx, igemm4_kernel<T, MODE, TM, TN, KG, NBUF, FS>, grid, block, a, name.c_str(), flops, 0, bytes);
}

// The 3x3 patch kernel: stride 1, pad 1, input channels in blocks of 64, rows short enough for the patch
bool patch_kernel_fits(const ConvShape& s, int in_c) {
  return s.R == 3 && s.S == 3 && s.stride == 1 && s.pad == 1 && in_c % kStep2 == 0 && 128 + 2 * (s.W + 1) <= 256;
}
template <int MODE>
bool patch_kernel_fits(const IgemmArgs& a) {
  const int in_c = MODE == kFwd ? a.C : a.K;
  return a.R == 3 && a.S == 3 && a.stride == 1 && a.pad == 1 && a.H == a.Ho && a.W == a.Wo && in_c % kStep2 == 0 &&
         128 + 2 * (a.W + 1) <= 256;
}

template <int MODE, int WM, int TN, int P_LD, int NBUF>
int launch_cfg3_rows(Context* ctx, IgemmArgs& a, double flops) {
  constexpr int BM = WM * 32, BN = 64 * TN;
  static const std::string name = std::string("igemm3_kernel<bf16,") + (MODE == kFwd ? "fwd," : "dgrad,") + std::to_string(BM) + "x" +
                                  std::to_string(BN) + "," + std::to_string(NBUF) + "buf," + (WM == 4 ? "8w," : "") + "patch" + std::to_string(P_LD * WM * 16) + ">";
  a.tiles_m = (a.gemm_m + BM - 1) / BM;
  a.tiles_n = (a.gemm_n + BN - 1) / BN;
  const int64_t wgs = static_cast<int64_t>(a.tiles_m) * a.tiles_n;
  if (wgs <= 0 || wgs > 0x7fffffff) {
    set_error("igemm: grid out of range");
    return -22;
  }
  a.group_rows = 0;
  bind_divisions(a, a.tiles_n);
  return launch(ctx, igemm3_kernel<MODE, WM, TN, P_LD, NBUF>, dim3(static_cast<unsigned>(wgs)), dim3(WM * 128), a, name.c_str(), flops, 0,
                conv_bytes<MODE>(a, 2));
}

// the number of patch rows: WM * 32 and a halo of W + 1 on both sides, loaded WM * 16 at a time
template <int MODE, int WM, int TN, int NBUF>
int launch_cfg3(Context* ctx, IgemmArgs& a, double flops) {
  const int loads = (WM * 32 + 2 * (a.W + 1) + WM * 16 - 1) / (WM * 16);
  if (loads <= 3) return launch_cfg3_rows<MODE, WM, TN, 3, NBUF>(ctx, a, flops);
  if (WM == 4 || loads <= 4) return launch_cfg3_rows<MODE, WM, TN, 4, NBUF>(ctx, a, flops);
  return launch_cfg3_rows<MODE, WM, TN, WM == 4 ? 4 : 6, NBUF>(ctx, a, flops);
}

// TCH_IGEMM2 = 0 keeps every convolution on igemm_kernel, whatever tiling is asked for; 2 or 3 picks the number of
// LDS tiles of tilings 0 - 2 (default: 2 for 128x128, 3 for 128x64 and 64x64)
int igemm2_setting() {
  static const int v = [] {
    const char* e = getenv("TCH_IGEMM2");
    return e ? atoi(e) : -1;
  }();
  return v;
}

// TCH_IGEMM_K32 = 0: the library's own choice leaves out the tilings with 32-element reduction steps
bool short_steps() {
  static const bool on = [] {
    const char* e = getenv("TCH_IGEMM_K32");
    return !(e && atoi(e) == 0);
  }();
  return on;
}

// Tilings of igemm4_kernel (tile, wavefronts the reduction is dealt to, LDS tiles in flight of each).  LDS decides how
// many workgroups share a CU: one (kSplit32Deep, kSplit64, kSplit64x32Deep) or two (the others).
enum SplitTile : int {
  kSplit32 = 15,         // 32 x 32, 4, 4
  kSplit32Deep = 16,     // 32 x 32, 8, 2
  kSplit64x32 = 17,      // 64 x 32, 4, 3
  kSplit64 = 18,         // 64 x 64, 4, 4 (fp32: 8, 2)
  kSplit64Pair = 19,     // 64 x 64, 4, 2
  kSplit64x32Deep = 20,  // 64 x 32, 8, 3
  kSplit16 = 32,         // 16 x 16, 8, 4 (bf16)
};

// Tilings of igemm2_kernel with pipelined operand reads
enum PipeTile : int {
  kPipe64 = 21,       // 64 x 64, operand reads pipelined over the steps, four LDS tiles
  kMix128x64 = 22,    // interleaved, eight wavefronts: 128 x 64, four LDS tiles
  kMix128 = 23,       // 128 x 128, three (tiling 0 has two, and a second workgroup beside it on its CU)
  kMix128x192 = 24,   // 128 x 192, three
};

// Tilings of igemm5_kernel (persistent grid, interleaved, eight wavefronts, three LDS tiles).  What the kernel does not take
// runs as kMix128x192 or kMix128, which have the same row tiles (no statistics are taken by kWalk256x128).
enum WalkTile : int {
  kWalk128x192 = 25,
  kWalk128 = 26,       // 128 x 128
  kWalk256x128 = 27,
};
bool walk_tile_fits(const IgemmArgs& a) {
  return igemm2_setting() != 0 && a.pointwise && a.gemm_k % kStep2 == 0 && !a.out_f32 && !a.scale && !a.relu_out && !a.mask && !a.add_sub &&
         !a.stats && !a.stat_acc;
}

// Tilings of igemm3_kernel (the 3x3 patch kernel) beside 5 = 128 x 64.  Convolutions it does not take run as tiling 1, kMix128, kPipe64,
// kPipe64 and kMix128x64, which have the same row tiles.
enum PatchTile : int {
  kPatch128 = 28,          // 128 x 128, three filter tiles in LDS as 5 (128 x 64) has
  kPatch64 = 29,           // 64 x 64, four wavefronts
  kPatch64Deep = 30,       // the same with nine filter tiles in LDS instead of three
  kPatch128x64Deep = 31,   // 5 with nine
};
bool patch_tile(int tile_cfg) { return tile_cfg == 5 || (tile_cfg >= kPatch128 && tile_cfg <= kPatch128x64Deep); }
bool patch_64_rows(int tile_cfg) { return tile_cfg == kPatch64 || tile_cfg == kPatch64Deep; }

// the tiling of the same shape that runs where a pipelined one does not exist
int pipe_stand_in(int tile_cfg) { return tile_cfg == kPipe64 || patch_64_rows(tile_cfg) ? 2 : tile_cfg == kMix128x64 || tile_cfg == kPatch128x64Deep ? 1 : 0; }

// The weight-gradient kernel's tile (0 = 128 x 128, 1 = 128 x 64, 2 = 64 x 64) for a tiling number: the same shape where
// there is one.  How the other kernels walk a tile (steps, LDS tiles, reductions split over wavefronts, the 3x3 patch) has
// no meaning here, whose reduction is split over workgroups.
int wgrad_tile(int tile_cfg) {
  switch (tile_cfg) {
    case 0:
    case 9:
    case 10:
    case 11:
    case 12:
    case kMix128:
    case kMix128x192:
    case kWalk128x192:
    case kWalk128:
    case kWalk256x128:
    case kPatch128:
      return 0;
    case 1:
    case 5:
    case 6:
    case 13:
    case kMix128x64:
    case kPatch128x64Deep:
      return 1;
    default:
      return 2;
  }
}

template <typename T>
int launch_wgrad(Context* ctx, IgemmArgs& a, int tile_cfg, double flops) {
  switch (wgrad_tile(tile_cfg)) {
    case 0:
      return launch_cfg<T, kWgrad, 2, 2, 2, 2>(ctx, a, flops);
    case 1:
      return launch_cfg<T, kWgrad, 2, 2, 2, 1>(ctx, a, flops);
    default:
      return launch_cfg<T, kWgrad, 2, 2, 1, 1>(ctx, a, flops);
  }
}

// forward and data gradient
template <typename T, int MODE>
int launch_mode(Context* ctx, IgemmArgs& a, int tile_cfg, double flops) {
  static_assert(MODE == kFwd || MODE == kDgrad, "weight gradients go through launch_wgrad");
  switch (tile_cfg) {
    case kSplit16:
      if constexpr (sizeof(T) == 2) {
        return launch_cfg4<T, MODE, 1, 1, 8, 4, 16>(ctx, a, flops);
      } else {   // effective_tile() gives fp32 kSplit32Deep, whose row tiles are others
        set_error("igemm: 16 x 16 tiles are for bf16");
        return -22;
      }
    case kSplit32:
      return launch_cfg4<T, MODE, 1, 1, 4, 4>(ctx, a, flops);
    case kSplit32Deep:
      return launch_cfg4<T, MODE, 1, 1, 8, 2>(ctx, a, flops);
    case kSplit64x32:
      return launch_cfg4<T, MODE, 2, 1, 4, 3>(ctx, a, flops);
    case kSplit64x32Deep:
      return launch_cfg4<T, MODE, 2, 1, 8, 3>(ctx, a, flops);
    case kSplit64:   // fp32 is bound by the matrix pipes: two wavefronts on each
      if constexpr (sizeof(T) == 2) return launch_cfg4<T, MODE, 2, 2, 4, 4>(ctx, a, flops);
      else return launch_cfg4<T, MODE, 2, 2, 8, 2>(ctx, a, flops);
    case kSplit64Pair:
      return launch_cfg4<T, MODE, 2, 2, 4, 2>(ctx, a, flops);
    default:
      break;
  }
  if constexpr (sizeof(T) == 2) {
    const int in_c = MODE == kFwd ? a.C : a.K;
    const int setting = igemm2_setting();
    if (patch_tile(tile_cfg)) {   // the 3x3 patch in LDS
      if (setting != 0 && patch_kernel_fits<MODE>(a)) {
        if (tile_cfg == 5) return launch_cfg3<MODE, 4, 1, 3>(ctx, a, flops);
        if (tile_cfg == kPatch128) return launch_cfg3<MODE, 4, 2, 3>(ctx, a, flops);
        if (tile_cfg == kPatch64) return launch_cfg3<MODE, 2, 1, 3>(ctx, a, flops);
        return tile_cfg == kPatch64Deep ? launch_cfg3<MODE, 2, 1, 9>(ctx, a, flops) : launch_cfg3<MODE, 4, 1, 9>(ctx, a, flops);
      }
      tile_cfg = tile_cfg == 5 ? 1 : tile_cfg == kPatch128 ? kMix128 : tile_cfg == kPatch128x64Deep ? kMix128x64 : kPipe64;
    }
    // 9 / 10: 256 x 256 on eight wavefronts (128 x 64 each), two LDS tiles, plain / rotated loop: for products with a
    // thousand such tiles or more (65 536 x 4096 x 4096: 1.18 and 1.31 PFLOP/s, 1.03 for 128 x 128; slower than 128 x 128 on
    // the other layers of the three models, by up to 1.7x)
    if (tile_cfg >= kWalk128x192 && tile_cfg <= kWalk256x128) {
      if (walk_tile_fits(a)) {
        if (tile_cfg == kWalk128x192) return launch_cfg5<MODE, 4, 2, 1, 3, 3>(ctx, a, flops);
        if (tile_cfg == kWalk128) return launch_cfg5<MODE, 4, 2, 1, 2, 3>(ctx, a, flops);
        return launch_cfg5<MODE, 4, 2, 2, 2, 3>(ctx, a, flops);
      }
      tile_cfg = tile_cfg == kWalk128x192 ? kMix128x192 : kMix128;
    }
    if (tile_cfg == 9 || tile_cfg == 10) {
      if (setting != 0 && in_c % kStep2 == 0 && a.R * a.S <= 32)
        return tile_cfg == 9 ? launch_cfg2<MODE, 2, 4, 4, 2, 2>(ctx, a, flops) : launch_cfg2<MODE, 2, 4, 4, 2, 2, 1>(ctx, a, flops);
      tile_cfg = 0;
    }
    // 11 - 14: 32-element reduction steps.  11 / 12: 128 x 128 with three / two LDS tiles in flight (48 / 34 KB:
    // three / four workgroups per CU), 13: 128 x 64 and 14: 64 x 64 with three (36 / 24 KB)
    if (tile_cfg >= 11 && tile_cfg <= 14) {
      if (setting != 0 && in_c % kStep2 == 0 && a.R * a.S <= 32) {
        if (tile_cfg == 11) return launch_cfg2<MODE, 2, 2, 2, 2, 3, 0, 32>(ctx, a, flops);
        if (tile_cfg == 12) return launch_cfg2<MODE, 2, 2, 2, 2, 2, 0, 32>(ctx, a, flops);
        if (tile_cfg == 13) return launch_cfg2<MODE, 2, 2, 2, 1, 3, 0, 32>(ctx, a, flops);
        return launch_cfg2<MODE, 2, 2, 1, 1, 3, 0, 32>(ctx, a, flops);
      }
      tile_cfg = tile_cfg <= 12 ? 0 : tile_cfg - 12;
    }
    // 6 / 7: tilings 1 / 2 with two LDS tiles in flight instead of three (48 / 32 KB of LDS: three or four
    // workgroups per CU, which the memory-bound data gradients of the large feature maps prefer)
    if (tile_cfg == 6 || tile_cfg == 7) {
      if (setting != 0 && in_c % kStep2 == 0 && a.R * a.S <= 32)
        return tile_cfg == 6 ? launch_cfg2<MODE, 2, 2, 2, 1, 2>(ctx, a, flops) : launch_cfg2<MODE, 2, 2, 1, 1, 2>(ctx, a, flops);
      tile_cfg -= 5;
    }
    // 21: operand reads pipelined over the steps, 22 - 24: interleaved on eight wavefronts (as tiling 0; see igemm2_kernel)
    if (tile_cfg >= kPipe64 && setting != 0 && in_c % kStep2 == 0 && a.R * a.S <= 32) {
      if (tile_cfg == kPipe64) return launch_cfg2<MODE, 2, 2, 1, 1, 4, 2>(ctx, a, flops);
      if (tile_cfg == kMix128) return launch_cfg2<MODE, 4, 2, 1, 2, 3, 1>(ctx, a, flops);
      if (tile_cfg == kMix128x192) return launch_cfg2<MODE, 4, 2, 1, 3, 3, 1>(ctx, a, flops);
      return launch_cfg2<MODE, 4, 2, 1, 1, 4, 1>(ctx, a, flops);
    }
    if (setting != 0 && in_c % kStep2 == 0 && a.R * a.S <= 32 && tile_cfg >= 0 && tile_cfg <= 2) {
      if (tile_cfg == 0)
        return setting == 3 ? launch_cfg2<MODE, 4, 2, 1, 2, 3, 1>(ctx, a, flops) : launch_cfg2<MODE, 4, 2, 1, 2, 2, 1>(ctx, a, flops);
      if (tile_cfg == 1)
        return setting == 2 ? launch_cfg2<MODE, 2, 2, 2, 1, 2>(ctx, a, flops) : launch_cfg2<MODE, 2, 2, 2, 1, 3>(ctx, a, flops);
      return setting == 2 ? launch_cfg2<MODE, 2, 2, 1, 1, 2>(ctx, a, flops) : launch_cfg2<MODE, 2, 2, 1, 1, 3>(ctx, a, flops);
    }
  }
  if (tile_cfg == 5) tile_cfg = 1;
  if (tile_cfg == 6 || tile_cfg == 7) tile_cfg -= 5;
  if (tile_cfg == 9 || tile_cfg == 10) tile_cfg = 0;
  if (tile_cfg >= 11 && tile_cfg <= 14) tile_cfg = tile_cfg <= 12 ? 0 : tile_cfg - 12;
  if (tile_cfg >= kPipe64) tile_cfg = pipe_stand_in(tile_cfg);
  switch (tile_cfg) {
    case 0:
      return launch_cfg<T, MODE, 2, 2, 2, 2>(ctx, a, flops);  // 128 x 128
    case 1:
      return launch_cfg<T, MODE, 2, 2, 2, 1>(ctx, a, flops);  // 128 x 64
    default:
      return launch_cfg<T, MODE, 2, 2, 1, 1>(ctx, a, flops);  // 64 x 64 (2, and 3 = never the direct-to-LDS kernel)
  }
}

// 2 * N*Ho*Wo * K * R*S*C: the same for forward, data gradient and weight gradient;
// zero-padded input channels do no algorithmic work
double conv_flops(const ConvShape& s, int Ho, int Wo) {
  const int c = (s.c_logical > 0 && s.c_logical < s.C) ? s.c_logical : s.C;
  return 2.0 * s.N * Ho * Wo * static_cast<double>(s.K) * s.R * s.S * c;
}

// rows of the workgroup tile of a tiling number (5 = the 3x3 patch kernel, or tiling 1 where it does not fit)
int tile_rows(int tile_cfg) {
  if (tile_cfg == 9 || tile_cfg == 10) return 256;
  if (tile_cfg == kSplit16) return 16;
  if (tile_cfg >= kPipe64) return tile_cfg == kPipe64 || patch_64_rows(tile_cfg) ? 64 : 128;
  if (tile_cfg >= kSplit32) return tile_cfg <= kSplit32Deep ? 32 : 64;
  if (tile_cfg >= 11 && tile_cfg <= 14) return tile_cfg == 14 ? 64 : 128;
  return (tile_cfg == 5 || tile_cfg == 6) ? 128 : tile_cfg >= 2 ? 64 : 128;
}

// column tiles of 32: callers of the in-kernel finalize provide a counter per 64 columns
bool narrow_tile(int tile_cfg) {
  return tile_cfg == kSplit16 || tile_cfg == kSplit32 || tile_cfg == kSplit32Deep || tile_cfg == kSplit64x32 || tile_cfg == kSplit64x32Deep;
}

int64_t tiles_for(int m, int n, int bm, int bn) {
  return static_cast<int64_t>((m + bm - 1) / bm) * ((n + bn - 1) / bn);
}

// Whether the 256 x 256 tiling (10) is worth asking for: the kernel it needs is at hand (bf16, reduction in whole
// 64-channel steps, few taps) and the product has at least four full rounds of such tiles.
bool wants_huge_tile(int dtype, int gemm_m, int gemm_n, int in_c, int taps) {
  return dtype == kBF16 && in_c % 64 == 0 && taps <= 32 && igemm2_setting() != 0 &&
         tiles_for(gemm_m, gemm_n, 256, 256) >= 1024;
}

// igemm4_kernel: whole 64-byte steps of input channels, one bit per tap
bool split_tile_fits(int dtype, int in_c, int taps) {
  return in_c % (dtype == kBF16 ? 32 : 16) == 0 && taps <= 32 && igemm2_setting() != 0;
}

// igemm2_kernel: whole 128-byte steps of bf16 input channels, one bit per tap
bool direct_tile_fits(int dtype, int in_c, int taps) {
  return dtype == kBF16 && in_c % 64 == 0 && taps <= 32 && igemm2_setting() != 0;
}

// The tiling that runs when `tile_cfg` is asked for: the 256 x 256 tilings exist for the direct-to-LDS kernel only
// and stand for 128 x 128 elsewhere (the statistics' row tiles follow the tiling that runs).
int effective_tile(int tile_cfg, int dtype, int in_c, int taps) {
  if ((tile_cfg == 9 || tile_cfg == 10) && !(dtype == kBF16 && in_c % 64 == 0 && taps <= 32 && igemm2_setting() != 0))
    return 0;
  if (tile_cfg == kSplit16) return !split_tile_fits(dtype, in_c, taps) ? 2 : dtype == kBF16 ? tile_cfg : kSplit32Deep;
  if (tile_cfg >= kPipe64) return direct_tile_fits(dtype, in_c, taps) ? tile_cfg : pipe_stand_in(tile_cfg);
  if (tile_cfg >= kSplit32 && !split_tile_fits(dtype, in_c, taps)) return 2;
  return tile_cfg;
}

// Enough workgroups to give each of the 256 CUs some, with bigger tiles as
// soon as the problem can afford them.  fp32 over short reductions is epilogue and latency: small tiles share a CU and
// overlap theirs (data gradients with the batch sums, 12544 x 256 over 64: 16.8 us as 128 x 128, 14.8 as 64 x 64; 25088
// rows 26.8 and 21.8).
int pick_tile(int dtype, int gemm_m, int gemm_n, int gemm_k) {
  if (dtype == kF32 && gemm_k <= 128) return 2;
  if (gemm_n > 64 && tiles_for(gemm_m, gemm_n, 128, 128) >= 384) return 0;
  if (tiles_for(gemm_m, gemm_n, 128, 64) >= 384) return 1;
  return 2;
}

// What a bf16 product on the direct-to-LDS kernels takes with each of the tilings worth having, in microseconds:
//   start + round * r + steps * max(alone, shared * r) + store * (outputs / 10^6)
// with r = workgroups per compute unit, rounded up, and steps = 64-element reduction steps.  `alone` is a step of one
// workgroup on a CU (a chain of latencies), `shared` what a step costs each of several that share the CU's operand
// path; `round` is what each further one adds to the epilogue: for eight of the plain tilings the fit leaves it at 0, and the
// epilogue is then in `start`, which also holds the 3 us of event, and in `store`.  How many workgroups fit on a CU at a time
// is not in the price; the exceptions below are what that costs.  The constants are least-squares fits (mean error 3-8 %) to
// 556 different convolutions where they stand in a step or request, one launch at a time (operands as cold or warm as their
// producers leave them; 3 us of event among it), each with every tiling: ResNet-152 at 1-64 images, GPT-2 at 512-8192
// tokens, Swin-B at 3-32 images; the second table for ResNet's data gradients with the BatchNorm sums, whose epilogue
// reads two more tensors.  (The patch tilings, 5 and 28-31, were fitted in the same way to ResNet-152's 3x3 convolutions alone: one
// round of workgroups is fastest with nine filter tiles, several with three, of which two workgroups fit on a CU.  kSplit16: two points
// of requests of one image, 208 and 832 workgroups.  The 302 products of 7-512 rows for which it is the choice from these prices, kernel
// times on filters that four launches in turn have read, as shares of the fastest of kSplit32, kSplit32Deep and kSplit64x32, forward / data
// gradient: over 1024 and more 0.85 / 0.86, 768 0.92 / 0.94, 512 0.94 / 0.98, 256 0.97 / 1.01, 128 0.99 / 1.05: from 256 on.)  (Fits to
// launches repeated on warm operands prefer large tiles: a request of 24 images took 2437 us with them, 2098 with these.)  Against the fastest of all tilings per launch, summed over a step or request: 1-2 %, one image 3.
// Tilings without an entry (3, 6, 7, 11, kSplit64, kSplit64Pair, kSplit64x32Deep: for callers that ask, and for tuners) are
// the fastest on some launches, by 1 % on average and 9 % at most.
struct TileCost {
  int cfg, bm, bn;
  float start, round, alone, shared, store;
};
const TileCost kPlainCost[] = {
    {0, 128, 128, 6.49f, 0.18f, 0.893f, 0.491f, 0.61f}, {1, 128, 64, 6.69f, 0.03f, 0.419f, 0.308f, 0.88f},
    {2, 64, 64, 6.39f, 0.00f, 0.343f, 0.209f, 0.68f}, {5, 128, 64, 6.34f, 0.00f, 0.237f, 0.291f, 1.12f},
    {12, 128, 128, 7.89f, 0.00f, 1.073f, 0.602f, 0.37f}, {13, 128, 64, 6.82f, 0.00f, 0.640f, 0.407f, 0.44f},
    {14, 64, 64, 6.44f, 0.00f, 0.598f, 0.265f, 0.41f}, {kSplit32, 32, 32, 6.13f, 0.00f, 0.108f, 0.114f, 2.05f},
    {kSplit32Deep, 32, 32, 5.70f, 0.00f, 0.148f, 0.117f, 3.12f}, {kSplit64x32, 64, 32, 6.05f, 0.00f, 0.208f, 0.160f, 1.53f},
    {kPipe64, 64, 64, 6.24f, 0.00f, 0.264f, 0.194f, 1.40f}, {kMix128x64, 128, 64, 5.60f, 1.22f, 0.336f, 0.340f, 0.83f},
    {kMix128, 128, 128, 5.74f, 1.31f, 0.542f, 0.493f, 0.72f}, {kMix128x192, 128, 192, 5.38f, 3.00f, 0.677f, 0.639f, 0.53f},
    {kPatch128, 128, 128, 6.02f, 0.53f, 0.404f, 0.404f, 0.71f}, {kPatch64, 64, 64, 5.37f, 0.00f, 0.303f, 0.134f, 1.64f},
    {kSplit16, 16, 16, 4.00f, 1.20f, 0.055f, 0.060f, 3.00f}, {kPatch64Deep, 64, 64, 5.30f, 1.53f, 0.142f, 0.161f, 1.62f}, {kPatch128x64Deep, 128, 64, 5.63f, 1.04f, 0.188f, 0.206f, 1.56f}};
const TileCost kSumsCost[] = {
    {0, 128, 128, 6.87f, 3.59f, 0.830f, 0.404f, 0.69f}, {1, 128, 64, 6.60f, 1.70f, 0.430f, 0.290f, 0.65f},
    {2, 64, 64, 6.41f, 0.85f, 0.364f, 0.188f, 0.53f}, {5, 128, 64, 3.36f, 5.47f, 0.295f, 0.010f, 0.64f},
    {12, 128, 128, 8.06f, 4.67f, 0.904f, 0.420f, 0.31f}, {13, 128, 64, 8.07f, 0.95f, 0.638f, 0.287f, 0.79f},
    {14, 64, 64, 7.33f, 0.10f, 0.585f, 0.210f, 1.13f}, {kSplit32, 32, 32, 6.35f, 0.00f, 0.134f, 0.099f, 4.42f},
    {kSplit32Deep, 32, 32, 5.72f, 1.24f, 0.180f, 0.109f, 0.25f}, {kSplit64x32, 64, 32, 6.71f, 0.26f, 0.213f, 0.150f, 2.36f},
    {kPipe64, 64, 64, 5.75f, 1.60f, 0.276f, 0.163f, 0.68f}, {kMix128x64, 128, 64, 4.52f, 4.11f, 0.256f, 0.316f, 0.74f},
    {kMix128, 128, 128, 3.63f, 5.89f, 0.446f, 0.382f, 0.83f}, {kPatch128, 128, 128, 6.01f, 0.52f, 0.473f, 0.473f, 0.65f},
    {kPatch64, 64, 64, 6.22f, 1.16f, 0.293f, 0.131f, 0.88f}, {kPatch64Deep, 64, 64, 5.70f, 2.80f, 0.066f, 0.155f, 0.80f},
    {kPatch128x64Deep, 128, 64, 5.98f, 3.45f, 0.170f, 0.194f, 1.03f}};
// fp32 where the output has fewer than one and a half 128 x 128 tiles per compute unit: the reduction is split inside the
// workgroup (igemm4_kernel), with smaller tiles as the grid shrinks.  fp32 takes at least eight times the multiplies of bf16, so it
// gains from spreading them over every SIMD (784 x 256 over 2304: 77.6 -> 14.8 us, with fp32 multiplies).  -1: none of them.
// The lines, with mean times over the layers of the three models in each class (244 launches, fp32 multiplies), the choice = 1:
//   up to one 32 x 32 tile per CU, K >= 1024 (53): eight wavefronts; four 1.11.  K < 1024 (25): four; eight 1.01
//   up to two, K < 1536 (38): 32 x 32 on four; eight 1.05, 64 x 32 1.05.  Two such tiles on a CU hide each other's
//     latencies until the reduction is long enough to do so alone: K >= 1536 (9) 64 x 32 on eight; 32 x 32 on eight 1.02, four 1.05
//   up to one 64 x 64 tile per CU, K >= 768 (19): kSplit64; 32 x 32 on eight 1.01 (0.89-1.17), kSplit64x32 1.08
//   up to two, K >= 512 (42): kSplit64x32; kSplit64Pair 1.01 (0.91-1.12), 32 x 32 1.03
//   beyond, K >= 256 (48): kSplit64Pair; igemm_kernel 64 x 64 0.97 (0.82-1.1), kSplit64x32 0.98: no line here is sharp
// From one and a half 128 x 128 tiles per CU on igemm_kernel takes 128 x 128 (33): 64 x 64 takes 0.91 of that on average
// (8192 x 768 over 3072: 383 us as 128 x 128, 294 as kSplit64Pair; 8192 x 3072 over 768: 287 and 330).
// (bf16 with channels that are no whole 64-element step: the two smallest forms only.)
int split_tile(int dtype, int gemm_m, int gemm_n, int gemm_k, int in_c, int taps) {
  if (!split_tile_fits(dtype, in_c, taps)) return -1;
  const int64_t t32 = tiles_for(gemm_m, gemm_n, 32, 32), t64 = tiles_for(gemm_m, gemm_n, 64, 64);
  if (t32 <= 256) return gemm_k >= 1024 ? kSplit32Deep : kSplit32;
  if (dtype == kBF16) return t32 <= 512 ? kSplit32 : -1;
  if (t32 <= 512) return gemm_k >= 1536 ? kSplit64x32Deep : kSplit32;
  if (t64 <= 256 && gemm_k >= 768) return kSplit64;
  if (t64 <= 512 && gemm_k >= 512) return kSplit64x32;
  return gemm_k >= 256 && tiles_for(gemm_m, gemm_n, 128, 128) < 384 ? kSplit64Pair : -1;
}

// The tiling the library takes by itself.  kAutoInOrder: one that adds up every reduction front to back, as all but the
// split ones do, so that a row's result is the same bits whatever the number of rows.  (The patch kernel, tiling 5, has
// an order of its own: never with kAutoInOrder.)
// kAutoLinear, kAutoLinearInOrder: for the linear layers of a transformer, the same two and igemm5_kernel, whose
// order of additions is front to back.
constexpr int kAutoInOrder = -2, kAutoLinear = -3, kAutoLinearInOrder = -4;
bool asks_in_order(int asked) { return asked == kAutoInOrder || asked == kAutoLinearInOrder; }
struct TileQuery {
  int dtype, gemm_m, gemm_n, gemm_k, in_c, taps;
  bool patch;   // the 3x3 patch kernel fits
  bool sums;    // data gradient with the BatchNorm sums in its epilogue
  bool dgrad;
  bool walk = false;   // igemm5_kernel takes it
  bool counted = false;   // a forward product whose row tiles leave sums: callers size those for row tiles of 32 at the least
};
// igemm5_kernel's tilings, priced as kPlainCost (r = tiles of a workgroup, one of them on a CU).  Fits to the linear layers of GPT-2 at 1024-
// 8192 tokens and of Swin-B at 4-32 images where they stand, 220 different ones with each tiling (mean error 5-8 %): first
// the forward ones, which add a bias and often a residual, then the data gradients.  Of 18.2 ms of forward launches with the tilings
// above 17.2 are left with this choice (17.1 with the fastest of every launch), of 20.8 ms of data gradients 19.3 (19.3).
const TileCost kWalkCost[2][3] = {
    {{kWalk128x192, 128, 192, 7.58f, 0.39f, 0.730f, 0.696f, 0.32f}, {kWalk128, 128, 128, 7.42f, 0.00f, 0.541f, 0.510f, 0.42f},
     {kWalk256x128, 256, 128, 7.44f, 0.42f, 0.734f, 0.734f, 0.46f}},
    {{kWalk128x192, 128, 192, 7.14f, 0.52f, 0.693f, 0.693f, 0.23f}, {kWalk128, 128, 128, 6.81f, 0.07f, 0.538f, 0.538f, 0.36f},
     {kWalk256x128, 256, 128, 6.97f, 0.47f, 0.733f, 0.733f, 0.43f}}};
int heuristic_tile(int asked, const TileQuery& q) {
  const bool linear = asked == kAutoLinear || asked == kAutoLinearInOrder;
  asked = asks_in_order(asked) ? kAutoInOrder : -1;
  if (!direct_tile_fits(q.dtype, q.in_c, q.taps)) {
    const int split = asked == kAutoInOrder ? -1 : split_tile(q.dtype, q.gemm_m, q.gemm_n, q.gemm_k, q.in_c, q.taps);
    return split >= 0 ? split : pick_tile(q.dtype, q.gemm_m, q.gemm_n, q.gemm_k);
  }
  const float steps = static_cast<float>(q.gemm_k) / 64.f, store = static_cast<float>(q.gemm_m) * q.gemm_n * 1e-6f;
  const bool large = q.gemm_n > 64 && tiles_for(q.gemm_m, q.gemm_n, 128, 128) >= 384;
  // what runs where the rules below leave nothing: data gradients on large grids over less than 1024, whose one tiling is 12,
  // with TCH_IGEMM_K32=0 (128 x 128 there too), and front-to-back products of up to 32 columns
  int best = large && !q.sums ? 0 : 2;
  float best_us = INFINITY;
  const TileCost* const costs = q.sums ? kSumsCost : kPlainCost;
  const size_t entries = q.sums ? std::size(kSumsCost) : std::size(kPlainCost);
  auto take = [&](const TileCost& t) {
    const float r = static_cast<float>((tiles_for(q.gemm_m, q.gemm_n, t.bm, t.bn) + 255) / 256);
    const float us = t.start + t.round * r + steps * fmaxf(t.alone, t.shared * r) + t.store * store;
    if (us < best_us) {
      best_us = us;
      best = t.cfg;
    }
  };
  for (size_t i = 0; i < entries; ++i) {
    const TileCost& t = costs[i];
    // From one and a half 128 x 128 tiles per compute unit on the table prices smaller tiles, which fetch more operand bytes per
    // flop, lower than they come out in a step.  GPT-2 8 x 1024 11.81 ms with this line, 11.91 without;
    // 1-6 x 1024, 3 x 777, Swin-B of 7-32 images, ResNet of 64 and requests of 24 and 64 the same.  From 256 tiles on 6 x 1024
    // takes 9.49 for 9.43 and 8 x 256 4.65 for 4.61; from 512 on 2 x 1024 5.26 for 5.16 and 8 x 256 4.71.  (384 tiles are
    // 8192 x 768 and 2048 x 3072, the products those sizes hang on; nothing measured lies closer on either side.)
    if (!q.sums && large && t.bm * t.bn < 128 * 128) continue;
    // 128 x 192 has a CU to itself: over a short reduction its epilogue and the next tile's first trip to memory are in
    // nobody's shadow, where the grid has several rounds, and the price knows rounds only as their number (8192 x 3072 over 768
    // alone 54.8 us, 47.5 as 128 x 128; 2048 x 3072 15.7 and 15.9; over 3072, 8192 x 768: 38.4 and 43.6).  In the steps: GPT-2 4 x
    // 1024 8.27 ms with this line, 8.35 without, 2 x 1024 5.16 and 5.28, 8 x 256 4.61 and 4.70, 3 x 1024 6.81 and 6.88; 8 x 1024 11.81
    // and 11.74, the one that it costs something.  Such grids were measured over 768 and from 2304 on; the line is in between.
    if (!q.sums && large && t.cfg == kMix128x192 && q.gemm_k < 1024) continue;
    // A transformer's data gradients run beside weight gradients that hold 64 KB of LDS and half of every SIMD's registers:
    // there the 128 x 128 tilings on eight wavefronts lose in the step (Swin-B of 32 images 9.85 ms without them, 9.91 with
    // both; of 24 images 8.30 and 8.38; GPT-2 2 x 512 3.70 and 3.75).  Not so over long reductions, where the table's next choice is
    // 64 x 64 at twice the operand bytes per flop: with three LDS tiles from 2048 on, GPT-2 takes 7.53 ms on 4 x 1024 (8.20
    // without), 8.46 on 5 x 1024 (8.88), 6.47 on 3 x 1024 (6.81), 5.85 on 12 x 256 (6.21); other GPT-2 sizes and Swin-B of 4-32
    // images, whose longest are 3072 and 4096, are the same.
    if (q.dgrad && !q.sums && (t.cfg == 0 || (t.cfg == kMix128 && q.gemm_k <= 2048))) continue;
    // more than half of the tile's columns lie in the output (56 x 56 x 256 -> 64, 20 images: 11.0 us as 128 x 128, 9.3 as 128 x 64)
    if (t.bn >= 2 * q.gemm_n && t.bn > 32) continue;
    if (t.cfg >= 12 && t.cfg <= 14 && !short_steps()) continue;
    if (patch_tile(t.cfg) && (!q.patch || asked == kAutoInOrder)) continue;
    if (t.bm * t.bn <= 64 * 32 && asked == kAutoInOrder) continue;   // igemm4_kernel's
    if (t.bm < 32 && (q.counted || q.gemm_k < 256)) continue;   // less than a reduction step for each of eight wavefronts
    take(t);
  }
  // Data gradients run beside weight gradients, whose LDS has no room on a compute unit that igemm5_kernel holds; from about 2560
  // rows on that costs less than it gains.  Step with igemm5_kernel for forward products only / for data gradients from 2560 rows on /
  // for all: GPT-2 of 8 x 256 4.60 / 4.60 / 4.63 ms, 3 x 777 5.33 / 5.33 / 5.42, 2 x 1024 5.16 / 5.16 / 5.20, 3 x 1024 6.25 / 6.20, 4 x 1024 7.37 /
  // 7.18, 5 x 1024 7.90 / 7.88, 8 x 1024 11.52 / 11.29, Swin-B of 24 images 8.26 / 8.22, of 28 9.00 / 8.98, of 12-20 the same.
  if (linear && q.walk && (!q.dgrad || q.gemm_m >= 2560))
    for (const TileCost& t : kWalkCost[q.dgrad])
      if (t.bn < 2 * q.gemm_n) take(t);
  return best;
}

int fill_common(IgemmArgs& a, const ConvShape& s, int dtype) {
  const int E = dtype == kBF16 ? 8 : 4;
  TCH_CHECK_ARG(dtype == kBF16 || dtype == kF32, "conv: dtype must be f32(0) or bf16(1)");
  TCH_CHECK_ARG(s.N > 0 && s.H > 0 && s.W > 0 && s.C > 0 && s.K > 0 && s.R > 0 && s.S > 0, "conv: non-positive dimension");
  TCH_CHECK_ARG(s.stride >= 1 && ilog2_exact(s.stride) >= 0, "conv: stride must be a power of two");
  TCH_CHECK_ARG(s.pad >= 0 && s.pad < s.R && s.pad < s.S, "conv: padding must be smaller than the filter");
  TCH_CHECK_ARG(s.C % E == 0 && s.K % E == 0, "conv: channel counts must be multiples of a 16-byte chunk");
  const int Ho = (s.H + 2 * s.pad - s.R) / s.stride + 1;
  const int Wo = (s.W + 2 * s.pad - s.S) / s.stride + 1;
  TCH_CHECK_ARG(Ho > 0 && Wo > 0, "conv: empty output");
  const int64_t in_elems = static_cast<int64_t>(s.N) * s.H * s.W * s.C;
  const int64_t out_elems = static_cast<int64_t>(s.N) * Ho * Wo * s.K;
  TCH_CHECK_ARG(in_elems < (1ll << 31) && out_elems < (1ll << 31), "conv: tensor exceeds 2^31 elements");
  TCH_CHECK_ARG(in_elems * (16 / E) < (1ll << 31) && out_elems * (16 / E) < (1ll << 31),
                "conv: tensor exceeds the 2 GiB reach of a buffer offset");
  TCH_CHECK_ARG(static_cast<int64_t>(s.K) * s.R * s.S * s.C < (1ll << 31), "conv: filter exceeds 2^31 elements");
  a.N = s.N;
  a.H = s.H;
  a.W = s.W;
  a.C = s.C;
  a.Ho = Ho;
  a.Wo = Wo;
  a.K = s.K;
  a.R = s.R;
  a.S = s.S;
  a.stride = s.stride;
  a.stride_log2 = ilog2_exact(s.stride);
  a.pad = s.pad;
  a.pointwise = (s.R == 1 && s.S == 1 && s.stride == 1 && s.pad == 0) ? 1 : 0;
  a.splits = 1;
  a.out_f32 = 0;
  a.accumulate = 0;
  a.add = nullptr;
  a.mask = nullptr;
  a.bias = nullptr;
  return 0;
}

}  // namespace

void conv_output_hw(const ConvShape& s, int* Ho, int* Wo) {
  *Ho = (s.H + 2 * s.pad - s.R) / s.stride + 1;
  *Wo = (s.W + 2 * s.pad - s.S) / s.stride + 1;
}

namespace {

bool check_finalize(const BnFinalize* f, bool forward) {
  return f->counters && f->gamma && f->out0 && f->out1 && f->coef && (!forward || f->beta) &&
         ((f->running_mean == nullptr) == (f->running_var == nullptr));
}

void bind_finalize(IgemmArgs& a, const BnFinalize* f) {
  a.fin_counters = f->counters;
  a.fin_gamma = f->gamma;
  a.fin_beta = f->beta;
  a.fin_running_mean = f->running_mean;
  a.fin_running_var = f->running_var;
  a.fin_out0 = f->out0;
  a.fin_out1 = f->out1;
  a.fin_coef = f->coef;
  a.fin_momentum = f->momentum;
  a.fin_eps = f->eps;
  a.fin_accumulate = f->accumulate;
}

}  // namespace

int conv2d_fwd(Context* ctx, int dtype, const ConvShape& s, const void* x, const void* w, void* y, const void* add,
               const void* mask, const float* bias, int out_f32, int tile_cfg, float* bn_partial,
               const BnFinalize* finalize, const float* scale, int relu_out, long long* bn_acc, int bn_acc_copies) {
  IgemmArgs a{};
  if (int rc = fill_common(a, s, dtype)) return rc;
  TCH_CHECK_ARG(!((scale || relu_out) && (bn_partial || bn_acc)), "conv2d_fwd: statistics are taken of the plain convolution output");
  TCH_CHECK_ARG(!(bn_acc && (bn_partial || finalize || out_f32)),
                "conv2d_fwd: accumulated statistics replace the per-tile ones and are taken of outputs stored in the compute type");
  TCH_CHECK_ARG(!bn_acc || (bn_acc_copies >= 1 && (bn_acc_copies & (bn_acc_copies - 1)) == 0),
                "conv2d_fwd: the number of accumulator copies must be a power of two");
  a.stat_acc = bn_acc;
  a.stat_acc_copies = bn_acc_copies;
  a.scale = scale;
  a.relu_out = relu_out ? 1 : 0;
  TCH_CHECK_ARG(x && w && y, "conv2d_fwd: null tensor");
  TCH_CHECK_ARG(!(bn_partial && out_f32), "conv2d_fwd: statistics are taken of outputs stored in the compute type");
  TCH_CHECK_ARG(!finalize || (bn_partial && check_finalize(finalize, true)), "conv2d_fwd: incomplete BatchNorm finalize operands");
  a.stats = bn_partial;
  const int eb = dtype == kBF16 ? 2 : 4;
  a.a_src = x;
  a.b_src = w;
  a.a_bytes = static_cast<uint32_t>(static_cast<int64_t>(s.N) * s.H * s.W * s.C * eb);
  a.b_bytes = static_cast<uint32_t>(static_cast<int64_t>(s.K) * s.R * s.S * s.C * eb);
  a.out = y;
  a.add = add;
  a.mask = mask;
  a.bias = bias;
  a.out_f32 = out_f32;
  a.gemm_m = s.N * a.Ho * a.Wo;
  a.gemm_n = s.K;
  a.gemm_k = s.R * s.S * s.C;
  a.k_per_split = (a.gemm_k + 31) / 32 * 32;
  a.div_plane = FastDiv(a.Ho * a.Wo);
  a.div_width = FastDiv(a.Wo);
  a.in_fp32 = asks_in_order(tile_cfg) ? 1 : 0;
  if (tile_cfg < 0) {
    tile_cfg = heuristic_tile(tile_cfg, {dtype, a.gemm_m, a.gemm_n, a.gemm_k, s.C, s.R * s.S, patch_kernel_fits(s, s.C), false, false, walk_tile_fits(a),
                                         bn_partial || bn_acc});
    // statistics are sized by the caller for the heuristic's row tiles: leave those launches alone
    if (!bn_partial && !bn_acc && wants_huge_tile(dtype, a.gemm_m, a.gemm_n, s.C, s.R * s.S)) tile_cfg = 10;
  }
  tile_cfg = effective_tile(tile_cfg, dtype, s.C, s.R * s.S);
  const int row_tiles = (a.gemm_m + tile_rows(tile_cfg) - 1) / tile_rows(tile_cfg);
  const bool in_kernel = finalize && row_tiles <= kBnFinalizeInKernelTiles && !narrow_tile(tile_cfg);
  if (in_kernel) bind_finalize(a, finalize);
  int rc = dtype == kBF16 ? launch_mode<bf16, kFwd>(ctx, a, tile_cfg, conv_flops(s, a.Ho, a.Wo))
                          : launch_mode<float, kFwd>(ctx, a, tile_cfg, conv_flops(s, a.Ho, a.Wo));
  if (rc || !finalize || in_kernel) return rc;
  return bn_fwd_finalize(ctx, bn_partial, row_tiles, s.K, a.gemm_m, finalize->gamma, finalize->beta,
                         finalize->running_mean, finalize->running_var, finalize->out0, finalize->out1, finalize->coef,
                         finalize->momentum, finalize->eps);
}

int conv2d_fwd_stat_rows(const ConvShape& s, int dtype, int tile_cfg) {
  int Ho, Wo;
  conv_output_hw(s, &Ho, &Wo);
  const int gemm_m = s.N * Ho * Wo;
  if (tile_cfg < 0) tile_cfg = heuristic_tile(tile_cfg, {dtype, gemm_m, s.K, s.R * s.S * s.C, s.C, s.R * s.S, patch_kernel_fits(s, s.C), false, false, false, true});
  tile_cfg = effective_tile(tile_cfg, dtype, s.C, s.R * s.S);
  const int bm = tile_rows(tile_cfg);
  return (gemm_m + bm - 1) / bm;
}

int conv2d_dgrad_stat_rows(const ConvShape& s, int dtype, int tile_cfg) {
  const int gemm_m = s.N * s.H * s.W;
  if (tile_cfg < 0) tile_cfg = heuristic_tile(tile_cfg, {dtype, gemm_m, s.C, s.R * s.S * s.K, s.K, s.R * s.S, patch_kernel_fits(s, s.K), true, true});
  tile_cfg = effective_tile(tile_cfg, dtype, s.K, s.R * s.S);
  const int bm = tile_rows(tile_cfg);
  return (gemm_m + bm - 1) / bm;
}

int conv2d_dgrad(Context* ctx, int dtype, const ConvShape& s, const void* dy, const void* wt, void* dx,
                 const void* add, const void* mask, int tile_cfg, const BnBwdSums* bn, int add_stride) {
  IgemmArgs a{};
  if (int rc = fill_common(a, s, dtype)) return rc;
  TCH_CHECK_ARG(dy && wt && dx, "conv2d_dgrad: null tensor");
  TCH_CHECK_ARG(add_stride == 1 || add_stride == 2, "conv2d_dgrad: the addend's grid is the output's or every second pixel of it");
  a.add_sub = (add && add_stride == 2) ? 1 : 0;
  if (bn) {
    TCH_CHECK_ARG(bn->x && bn->mean && bn->invstd && ((bn->partial != nullptr) != (bn->acc != nullptr)),
                  "conv2d_dgrad: incomplete BatchNorm operands");
    TCH_CHECK_ARG(!bn->finalize || (bn->partial && check_finalize(bn->finalize, false)),
                  "conv2d_dgrad: incomplete BatchNorm finalize operands");
    TCH_CHECK_ARG(!bn->acc || (bn->acc_copies >= 1 && (bn->acc_copies & (bn->acc_copies - 1)) == 0),
                  "conv2d_dgrad: the number of accumulator copies must be a power of two");
    a.stats = bn->partial;
    a.stat_acc = bn->acc;
    a.stat_acc_copies = bn->acc_copies;
    a.bn_mask = bn->mask;
    a.bn_x = bn->x;
    a.bn_mean = bn->mean;
    a.bn_invstd = bn->invstd;
  }
  const int eb = dtype == kBF16 ? 2 : 4;
  a.a_src = dy;
  a.b_src = wt;
  a.a_bytes = static_cast<uint32_t>(static_cast<int64_t>(s.N) * a.Ho * a.Wo * s.K * eb);
  a.b_bytes = static_cast<uint32_t>(static_cast<int64_t>(s.K) * s.R * s.S * s.C * eb);
  a.out = dx;
  a.add = add;
  a.mask = mask;
  a.gemm_m = s.N * s.H * s.W;
  a.gemm_n = s.C;
  a.gemm_k = s.R * s.S * s.K;
  a.k_per_split = (a.gemm_k + 31) / 32 * 32;
  // 1x1 stride 1: dy is a dense [pixels][K] matrix in the same pixel order as dx
  a.div_plane = FastDiv(s.H * s.W);
  a.div_width = FastDiv(s.W);
  a.in_fp32 = asks_in_order(tile_cfg) ? 1 : 0;
  if (tile_cfg < 0) {
    tile_cfg = heuristic_tile(tile_cfg, {dtype, a.gemm_m, a.gemm_n, a.gemm_k, s.K, s.R * s.S, patch_kernel_fits(s, s.K), bn != nullptr, true, walk_tile_fits(a)});
    if (!bn && wants_huge_tile(dtype, a.gemm_m, a.gemm_n, s.K, s.R * s.S)) tile_cfg = 10;
  }
  tile_cfg = effective_tile(tile_cfg, dtype, s.K, s.R * s.S);
  const BnFinalize* finalize = bn ? bn->finalize : nullptr;
  const int row_tiles = (a.gemm_m + tile_rows(tile_cfg) - 1) / tile_rows(tile_cfg);
  const bool in_kernel = finalize && row_tiles <= kBnFinalizeInKernelTiles && !narrow_tile(tile_cfg);
  if (in_kernel) bind_finalize(a, finalize);
  int rc = dtype == kBF16 ? launch_mode<bf16, kDgrad>(ctx, a, tile_cfg, conv_flops(s, a.Ho, a.Wo))
                          : launch_mode<float, kDgrad>(ctx, a, tile_cfg, conv_flops(s, a.Ho, a.Wo));
  if (rc || !finalize || in_kernel) return rc;
  return bn_bwd_finalize(ctx, bn->partial, row_tiles, s.C, a.gemm_m, finalize->gamma, bn->mean, bn->invstd,
                         finalize->out0, finalize->out1, finalize->coef, finalize->accumulate);
}

int64_t conv2d_wgrad_workspace_bytes(const ConvShape& s, int dtype, int splits) {
  if (splits <= 1) return 0;
  (void)dtype;
  // partial filters, then partial column sums of dy for callers that also want the bias gradient
  return static_cast<int64_t>(splits) * (static_cast<int64_t>(s.K) * s.R * s.S * s.C + s.K) * 4;
}

// tile of a weight gradient without a tiling from the caller: 128 x 128 where it leaves at least 128 workgroups, in fp32 1024
// (TCH_WGRAD_BIG_TILE_WGS: another count).  An fp32 gradient is bound by the matrix pipes: 144 workgroups of 128 x 128 use
// those of 144 compute units, and their 40 KB of LDS (64 x 64: 24; in parts 52 and 28) keep main-lane workgroups away.  In the step (fp32 multiplies), from 128 /
// 256 / 512 / 1024 / 2000 on / never: GPT-2 2 x 256 6.48 / 6.39 / 6.22 / 6.22 / 6.19 / 6.25 ms, 1 x 512 7.34 / 6.98 / 6.88 / 6.88 /
// 6.86 / 6.89, 8 x 512 31.48 / 31.50 / 31.56 / 31.50 / 31.94 / 31.88.
bool wgrad_big_tile(int dtype, int gemm_m, int gemm_n, int64_t splits) {
  static const int asked = [] {
    const char* e = getenv("TCH_WGRAD_BIG_TILE_WGS");
    return e && atoi(e) > 0 ? atoi(e) : 0;
  }();
  const int from = asked ? asked : dtype == kF32 ? 1024 : 128;
  return gemm_m >= 128 && gemm_n >= 128 && tiles_for(gemm_m, gemm_n, 128, 128) * splits >= from;
}

int conv2d_wgrad_pick_splits(const ConvShape& s, int dtype) {
  const int BK = dtype == kBF16 ? 32 : 16;
  int Ho, Wo;
  conv_output_hw(s, &Ho, &Wo);
  const int64_t pixels = static_cast<int64_t>(s.N) * Ho * Wo;
  const int gemm_m = s.K, gemm_n = s.R * s.S * s.C;
  int64_t most = pixels / (4 * BK);   // at least four reduction steps per split
  if (most > 512) most = 512;
  if (most < 1) most = 1;
  // TCH_WGRAD_WGS: a workgroup count to aim for instead
  static const int aim = [] {
    const char* e = getenv("TCH_WGRAD_WGS");
    return e && atoi(e) > 0 ? atoi(e) : 0;
  }();
  if (aim) {
    int64_t tiles = tiles_for(gemm_m, gemm_n, 128, 128);
    if (tiles < 8) tiles = tiles_for(gemm_m, gemm_n, 64, 64);
    return static_cast<int>(std::min((aim + tiles - 1) / tiles, most));
  }
  // The split count with the shortest start + steps * max(alone, shared * r) + store * (10^6 results written), r =
  // workgroups per compute unit, rounded up: least-squares fits (6-8 % mean error) to 1 500 launches of every split count
  // on the layers of the three models at 128-8192 rows and 1-64 images, per dtype for 128 x 128 and 64 x 64 tiles
  // (128 x 128 in bf16 alone on a CU measured again since: 0.249 -> 0.203, GPT-2 8 x 1024 11.20 -> 11.14 ms, ResNet of 32 images 8.94 ->
  // 8.73).  A partial filter is read again by the reduction that rides the next launch: kReread on top of what it
  // costs to write.  (Aiming at 192-384 workgroups instead split short reductions that were launch latency and
  // partial filters already: 1024 -> 3072 over 343 rows 17.8 us with two splits, 10.1 with one; 256 -> 768 over 5488
  // rows 15.6 with 16, 10.8 with 4.)
  struct Cost {
    float start, alone, shared, store;
  };
  static const Cost cost[2][2] = {{{3.39f, 0.229f, 0.383f, 1.55f}, {8.56f, 0.371f, 0.912f, 0.71f}},     // fp32: 64, 128
                                  {{3.08f, 0.109f, 0.089f, 2.33f}, {6.37f, 0.203f, 0.179f, 0.94f}}};   // bf16
  constexpr float kReread = 1.f;   // microseconds per 10^6 results; 0 - 2 in the steps: within 1 %, 1 the best of most
  int best = 1;
  float best_us = INFINITY;
  for (int64_t want = 1; want <= most; ++want) {
    const int64_t steps = ((pixels + want - 1) / want + BK - 1) / BK;
    const int64_t splits = (pixels + steps * BK - 1) / (steps * BK);
    if (splits != want) continue;   // the same as a smaller count
    const bool big = wgrad_big_tile(dtype, gemm_m, gemm_n, splits);
    const Cost& c = cost[dtype == kBF16][big];
    const int side = big ? 128 : 64;
    const float r = static_cast<float>((tiles_for(gemm_m, gemm_n, side, side) * splits + 255) / 256);
    const float results = static_cast<float>(gemm_m) * gemm_n * splits * 1e-6f;
    const float us = c.start + steps * fmaxf(c.alone, c.shared * r) + (c.store + (splits > 1 ? kReread : 0.f)) * results;
    if (us < best_us) {
      best_us = us;
      best = static_cast<int>(splits);
    }
  }
  return best;
}

int conv2d_wgrad_flush(Context* ctx) {
  if (int rc = col_sum_flush(ctx)) return rc;
  auto& tr = ctx->trailing_reduce;
  if (!tr.valid) return 0;
  tr.valid = false;
  return launch(ctx, splitk_reduce_kernel, dim3(tr.blocks), dim3(256), tr.args, "splitk_reduce_kernel", tr.bytes, 1);
}

int conv2d_wgrad(Context* ctx, int dtype, const ConvShape& s, const void* x, const void* dy, float* dw, float* workspace,
                 int splits, int accumulate, int tile_cfg, float* dbias, int trailing) {
  IgemmArgs a{};
  if (int rc = fill_common(a, s, dtype)) return rc;
  TCH_CHECK_ARG(x && dy && dw, "conv2d_wgrad: null tensor");
  const int eb = dtype == kBF16 ? 2 : 4;
  TCH_CHECK_ARG(splits >= 1, "conv2d_wgrad: splits must be >= 1");
  TCH_CHECK_ARG(splits == 1 || workspace, "conv2d_wgrad: split reduction needs a workspace");
  const int BK = dtype == kBF16 ? 32 : 16;
  a.a_src = dy;
  a.b_src = x;
  a.a_bytes = static_cast<uint32_t>(static_cast<int64_t>(s.N) * a.Ho * a.Wo * s.K * eb);
  a.b_bytes = static_cast<uint32_t>(static_cast<int64_t>(s.N) * s.H * s.W * s.C * eb);
  a.gemm_m = s.K;
  a.gemm_n = s.R * s.S * s.C;
  a.gemm_k = s.N * a.Ho * a.Wo;
  int per = (a.gemm_k + splits - 1) / splits;
  per = (per + BK - 1) / BK * BK;
  splits = (a.gemm_k + per - 1) / per;  // drop empty tail splits
  a.splits = splits;
  a.k_per_split = per;
  a.accumulate = accumulate;
  a.take_pending = trailing ? 1 : 0;
  a.out = splits > 1 ? static_cast<void*>(workspace) : static_cast<void*>(dw);
  float* dbias_partial = workspace ? workspace + static_cast<int64_t>(splits) * a.gemm_m * a.gemm_n : nullptr;
  a.dbias = !dbias ? nullptr : splits > 1 ? dbias_partial : dbias;
  a.div_plane = FastDiv(a.Ho * a.Wo);
  a.div_width = FastDiv(a.Wo);
  if (tile_cfg < 0) {
    tile_cfg = wgrad_big_tile(dtype, a.gemm_m, a.gemm_n, splits) ? 0 : 2;
  }
  int rc = dtype == kBF16 ? launch_wgrad<bf16>(ctx, a, tile_cfg, conv_flops(s, a.Ho, a.Wo))
                          : launch_wgrad<float>(ctx, a, tile_cfg, conv_flops(s, a.Ho, a.Wo));
  if (rc) return rc;
  if (splits > 1) {
    ReduceArgs r{workspace, dw, static_cast<int64_t>(a.gemm_m) * a.gemm_n, splits, accumulate, dbias_partial, dbias,
                 dbias ? a.gemm_m : 0, 0u};
    TCH_CHECK_ARG(r.n % 4 == 0, "conv2d_wgrad: filter size must be a multiple of 4");
    r.first_blocks = static_cast<unsigned>((r.n / 4 + 255) / 256);
    const unsigned blocks = r.first_blocks + static_cast<unsigned>((r.n2 + 255) / 256);
    const double red_bytes = 4.0 * r.n * (splits + 1 + (accumulate ? 1 : 0));
    if (trailing) {
      // not launched now: rides the next weight gradient of this context (which must use ANOTHER workspace), or
      // conv2d_wgrad_flush.  An earlier pending reduction was taken along by the launch above.
      auto& tr = ctx->trailing_reduce;
      tr.valid = true;
      tr.args = r;
      tr.blocks = blocks;
      tr.bytes = red_bytes;
      return 0;
    }
    return launch(ctx, splitk_reduce_kernel, dim3(blocks), dim3(256), r, "splitk_reduce_kernel", red_bytes, 1);
  }
  return 0;
}

// ---------------------------------------------------------------------------------------------------------------
// Grouped weight gradients: the weight gradients of several convolutions (a stage of a network, whose dy tensors
// are all at hand once the data-gradient chain has passed) as ONE launch over a table, plus one launch for the
// split reductions that are left.  Together the convolutions fill the chip, so each needs few splits or none:
// long reduction loops, little or nothing written as partial filters, two launches instead of two per layer.
// ---------------------------------------------------------------------------------------------------------------
namespace {

struct GroupLayout {
  int64_t args_off = 0, red_off = 0, map_off = 0, rmap_off = 0, bytes = 0;
  int64_t wgs = 0, reduce_blocks = 0, workspace_floats = 0;
};

int group_tile(int dtype, int n, const ConvShape* shapes, int tile_cfg) {
  if (tile_cfg == 0 || tile_cfg == 2) return tile_cfg;
  for (int i = 0; i < n; ++i)
    if (shapes[i].K < 128 || shapes[i].R * shapes[i].S * shapes[i].C < 128) return 2;
  return 0;
}

int64_t group_pixels(const ConvShape& s) {
  int Ho, Wo;
  conv_output_hw(s, &Ho, &Wo);
  return static_cast<int64_t>(s.N) * Ho * Wo;
}

// what conv2d_wgrad makes of a requested split count: whole reduction steps per split, no empty tail splits
void normalise_split(int64_t pixels, int BK, int want, int* splits, int* per) {
  if (want < 1) want = 1;
  int64_t p = (pixels + want - 1) / want;
  p = (p + BK - 1) / BK * BK;
  *per = static_cast<int>(p);
  *splits = static_cast<int>((pixels + p - 1) / p);
}

GroupLayout group_layout(int dtype, int n, const ConvShape* shapes, const int* splits, int tile) {
  const int BK = dtype == kBF16 ? 32 : 16;
  const int bm = tile == 0 ? 128 : 64;
  GroupLayout L;
  for (int i = 0; i < n; ++i) {
    const ConvShape& s = shapes[i];
    int sp, per;
    normalise_split(group_pixels(s), BK, splits[i], &sp, &per);
    const int64_t filt = static_cast<int64_t>(s.K) * s.R * s.S * s.C;
    L.wgs += tiles_for(s.K, s.R * s.S * s.C, bm, bm) * sp;
    if (sp > 1) {
      L.workspace_floats += sp * (filt + s.K);
      L.reduce_blocks += (filt / 4 + 255) / 256 + (s.K + 255) / 256;
    }
  }
  auto up = [](int64_t v) { return (v + 255) / 256 * 256; };
  L.args_off = 0;
  L.red_off = up(static_cast<int64_t>(n) * sizeof(IgemmArgs));
  L.map_off = L.red_off + up(static_cast<int64_t>(n) * sizeof(ReduceArgs));
  L.rmap_off = L.map_off + up(L.wgs * static_cast<int64_t>(sizeof(uint2)));
  L.bytes = L.rmap_off + up(L.reduce_blocks * static_cast<int64_t>(sizeof(uint2)));
  return L;
}

}  // namespace

int conv2d_wgrad_group_plan(int dtype, int n, const ConvShape* shapes, int target_wgs, int tile_cfg, int* splits,
                            int64_t* table_bytes, int64_t* workspace_bytes) {
  TCH_CHECK_ARG(n > 0 && shapes && splits, "conv2d_wgrad_group_plan: empty group");
  TCH_CHECK_ARG(dtype == kBF16 || dtype == kF32, "conv2d_wgrad_group_plan: dtype must be f32(0) or bf16(1)");
  const int BK = dtype == kBF16 ? 32 : 16;
  const int tile = group_tile(dtype, n, shapes, tile_cfg);
  const int bm = tile == 0 ? 128 : 64;
  if (target_wgs <= 0) target_wgs = 1024;
  constexpr int64_t kMinSteps = 16;   // a split is at least this many reduction steps long
  std::vector<int64_t> steps(n), tiles(n);
  int64_t longest = 1;
  for (int i = 0; i < n; ++i) {
    const ConvShape& s = shapes[i];
    TCH_CHECK_ARG(s.N > 0 && s.H > 0 && s.W > 0 && s.C > 0 && s.K > 0 && s.R > 0 && s.S > 0, "conv: non-positive dimension");
    steps[i] = (group_pixels(s) + BK - 1) / BK;
    tiles[i] = tiles_for(s.K, s.R * s.S * s.C, bm, bm);
    longest = std::max(longest, steps[i]);
  }
  // Every workgroup runs about `len` reduction steps: the largest `len` that still yields target_wgs workgroups
  // (none if the unsplit group already has that many).
  auto wgs_at = [&](int64_t len) {
    int64_t w = 0;
    for (int i = 0; i < n; ++i) w += tiles[i] * ((steps[i] + len - 1) / len);
    return w;
  };
  int64_t len = longest;
  if (wgs_at(len) < target_wgs) {
    int64_t lo = kMinSteps, hi = longest;   // wgs_at is non-increasing in len
    while (lo < hi) {
      const int64_t mid = (lo + hi + 1) / 2;
      if (wgs_at(mid) >= target_wgs) lo = mid; else hi = mid - 1;
    }
    len = lo;
  }
  for (int i = 0; i < n; ++i) {
    int sp, per;
    normalise_split(group_pixels(shapes[i]), BK, static_cast<int>(std::min<int64_t>((steps[i] + len - 1) / len, 512)), &sp, &per);
    splits[i] = sp;
  }
  const GroupLayout L = group_layout(dtype, n, shapes, splits, tile);
  if (table_bytes) *table_bytes = L.bytes;
  if (workspace_bytes) *workspace_bytes = std::max<int64_t>(L.workspace_floats * 4, 4);
  return tile;
}

int conv2d_wgrad_group(Context* ctx, int dtype, int n, const WgradGroupItem* items, int tile_cfg, int accumulate,
                       float* workspace, void* table, int max_wgs) {
  TCH_CHECK_ARG(n > 0 && items && table, "conv2d_wgrad_group: empty group or no table");
  const int eb = dtype == kBF16 ? 2 : 4;
  const int BK = dtype == kBF16 ? 32 : 16;
  std::vector<ConvShape> shapes(n);
  std::vector<int> splits(n);
  for (int i = 0; i < n; ++i) {
    shapes[i] = items[i].shape;
    splits[i] = items[i].splits;
  }
  const int tile = group_tile(dtype, n, shapes.data(), tile_cfg);
  const int bm = tile == 0 ? 128 : 64;
  const GroupLayout L = group_layout(dtype, n, shapes.data(), splits.data(), tile);
  TCH_CHECK_ARG(L.workspace_floats == 0 || workspace, "conv2d_wgrad_group: split reductions need a workspace");
  TCH_CHECK_ARG(L.wgs > 0 && L.wgs <= 0x7fffffff, "conv2d_wgrad_group: grid out of range");

  std::vector<unsigned char> host(static_cast<size_t>(L.bytes), 0);
  IgemmArgs* args = reinterpret_cast<IgemmArgs*>(host.data() + L.args_off);
  ReduceArgs* reds = reinterpret_cast<ReduceArgs*>(host.data() + L.red_off);
  uint2* map = reinterpret_cast<uint2*>(host.data() + L.map_off);
  uint2* rmap = reinterpret_cast<uint2*>(host.data() + L.rmap_off);
  double flops = 0.0, bytes = 0.0, red_bytes = 0.0;
  int64_t ws_off = 0;
  int n_red = 0;
  std::vector<int> order(n);
  for (int i = 0; i < n; ++i) order[i] = i;
  for (int i = 0; i < n; ++i) {
    IgemmArgs& a = args[i];
    const WgradGroupItem& it = items[i];
    if (int rc = fill_common(a, it.shape, dtype)) return rc;
    TCH_CHECK_ARG(it.x && it.dy && it.dw, "conv2d_wgrad_group: null tensor");
    const ConvShape& s = it.shape;
    a.a_src = it.dy;
    a.b_src = it.x;
    a.a_bytes = static_cast<uint32_t>(static_cast<int64_t>(s.N) * a.Ho * a.Wo * s.K * eb);
    a.b_bytes = static_cast<uint32_t>(static_cast<int64_t>(s.N) * s.H * s.W * s.C * eb);
    a.gemm_m = s.K;
    a.gemm_n = s.R * s.S * s.C;
    a.gemm_k = s.N * a.Ho * a.Wo;
    normalise_split(a.gemm_k, BK, it.splits, &a.splits, &a.k_per_split);
    a.accumulate = accumulate;
    a.tiles_m = (a.gemm_m + bm - 1) / bm;
    a.tiles_n = (a.gemm_n + bm - 1) / bm;
    bind_divisions(a, a.tiles_n);
    a.div_plane = FastDiv(a.Ho * a.Wo);
    a.div_width = FastDiv(a.Wo);
    const int64_t filt = static_cast<int64_t>(a.gemm_m) * a.gemm_n;
    if (a.splits > 1) {
      float* part = workspace + ws_off;
      float* bias_part = part + a.splits * filt;
      ws_off += a.splits * (filt + a.gemm_m);
      a.out = part;
      a.dbias = it.dbias ? bias_part : nullptr;
      TCH_CHECK_ARG(filt % 4 == 0, "conv2d_wgrad_group: filter size must be a multiple of 4");
      ReduceArgs& r = reds[n_red];
      r = ReduceArgs{part, it.dw, filt, a.splits, accumulate, bias_part, it.dbias, it.dbias ? a.gemm_m : 0, 0u};
      r.first_blocks = static_cast<unsigned>((filt / 4 + 255) / 256);
      red_bytes += 4.0 * filt * (a.splits + 1 + (accumulate ? 1 : 0));
      ++n_red;
    } else {
      a.out = it.dw;
      a.dbias = it.dbias;
    }
    flops += conv_flops(s, a.Ho, a.Wo);
    bytes += conv_bytes<kWgrad>(a, eb);
  }
  // long workgroups first: what is left for the tail of the launch is short
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return args[x].k_per_split > args[y].k_per_split; });
  int64_t w = 0;
  for (int oi = 0; oi < n; ++oi) {
    const int i = order[oi];
    const int64_t cnt = static_cast<int64_t>(args[i].tiles_m) * args[i].tiles_n * args[i].splits;
    for (int64_t j = 0; j < cnt; ++j) map[w++] = make_uint2(static_cast<unsigned>(i), static_cast<unsigned>(j));
  }
  TCH_CHECK_ARG(w == L.wgs, "conv2d_wgrad_group: workgroup count does not match the layout");
  int64_t rb = 0;
  for (int i = 0; i < n_red; ++i) {
    const unsigned cnt = reds[i].first_blocks + static_cast<unsigned>((reds[i].n2 + 255) / 256);
    for (unsigned j = 0; j < cnt; ++j) rmap[rb++] = make_uint2(static_cast<unsigned>(i), j);
  }
  TCH_CHECK_ARG(rb <= L.reduce_blocks, "conv2d_wgrad_group: reduction blocks do not match the layout");
  // The table is written once, here; the launches (recorded or not) read it whenever they run.
  hipError_t e = hipMemcpy(table, host.data(), host.size(), hipMemcpyHostToDevice);
  TCH_CHECK_ARG(e == hipSuccess, std::string("conv2d_wgrad_group: table upload: ") + hipGetErrorString(e));

  unsigned char* dev = static_cast<unsigned char*>(table);
  WgradGroupArgs g{reinterpret_cast<const IgemmArgs*>(dev + L.args_off), reinterpret_cast<const uint2*>(dev + L.map_off),
                   static_cast<uint32_t>(L.wgs)};
  const dim3 grid(static_cast<unsigned>(max_wgs > 0 && max_wgs < L.wgs ? max_wgs : L.wgs)), block(256);
  static const std::string names[2][2] = {{"wgrad_group_kernel<f32,128x128>", "wgrad_group_kernel<f32,64x64>"},
                                          {"wgrad_group_kernel<bf16,128x128>", "wgrad_group_kernel<bf16,64x64>"}};
  const char* name = names[dtype == kBF16 ? 1 : 0][tile == 0 ? 0 : 1].c_str();
  int rc;
  if (dtype == kBF16)
    rc = tile == 0 ? launch(ctx, wgrad_group_kernel<bf16, 2, 2, 2, 2>, grid, block, g, name, flops, 0, bytes)
                   : launch(ctx, wgrad_group_kernel<bf16, 2, 2, 1, 1>, grid, block, g, name, flops, 0, bytes);
  else
    rc = tile == 0 ? launch(ctx, wgrad_group_kernel<float, 2, 2, 2, 2>, grid, block, g, name, flops, 0, bytes)
                   : launch(ctx, wgrad_group_kernel<float, 2, 2, 1, 1>, grid, block, g, name, flops, 0, bytes);
  if (rc) return rc;
  if (rb > 0) {
    ReduceGroupArgs rg{reinterpret_cast<const ReduceArgs*>(dev + L.red_off), reinterpret_cast<const uint2*>(dev + L.rmap_off)};
    return launch(ctx, splitk_reduce_group_kernel, dim3(static_cast<unsigned>(rb)), dim3(256), rg,
                  "splitk_reduce_group_kernel", red_bytes, 1);
  }
  return 0;
}

// ---------------------------------------------------------------------------------------------------------------
// Weight gradient for callers that cannot allocate: the split-K partials go to a buffer that is part of the
// library's own device image, so that no workspace is passed in and none is made.
// ---------------------------------------------------------------------------------------------------------------
}  // namespace tch

// 64 MiB of fp32 partials per GPU, held from the moment the code object is loaded until the process ends.
// Host code never touches this name: it is a host-side stand-in for a device symbol.  The device address comes
// from hipGetSymbolAddress, once per device, and that pointer is what kernels and copies get.
static constexpr int64_t kStaticScratchFloats = 16ll << 20;
static __device__ __align__(256) float scratch[kStaticScratchFloats];

namespace tch {

namespace {
constexpr int kScratchDevices = 16;
std::mutex g_scratch_mu;
float* g_scratch_ptr[kScratchDevices] = {};
// who used the buffer last on each device: a call on another stream waits for that call's reduction first
hipEvent_t g_scratch_done[kScratchDevices] = {};
hipStream_t g_scratch_stream[kScratchDevices] = {};
bool g_scratch_used[kScratchDevices] = {};

// The device address of `scratch` on the current device (every GPU holds its own copy at its own address).
int static_scratch(float** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  TCH_CHECK_ARG(e == hipSuccess && dev >= 0 && dev < kScratchDevices,
                std::string("conv2d_wgrad_static: hipGetDevice: ") + hipGetErrorString(e));
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    TCH_CHECK_ARG(e == hipSuccess && ptr, std::string("conv2d_wgrad_static: hipGetSymbolAddress: ") + hipGetErrorString(e));
    g_scratch_ptr[dev] = static_cast<float*>(ptr);
    // set-up, once per device: the event that orders two streams' use of the buffer
    e = hipEventCreateWithFlags(&g_scratch_done[dev], hipEventDisableTiming);
    TCH_CHECK_ARG(e == hipSuccess, std::string("conv2d_wgrad_static: hipEventCreate: ") + hipGetErrorString(e));
  }
  *out = g_scratch_ptr[dev];
  return 0;
}

// Launches that go to a stream right now (not recorded into a program, not held in a launch queue, not captured
// into a graph) are ordered here: the buffer's previous user on ANOTHER stream must have finished its reduction
// before this call's partials overwrite it.  In the other three cases the launches run later, in an order only
// the caller knows: there the caller keeps two users of the buffer apart.
bool orders_itself(Context* ctx, hipStream_t stream) {
  if (ctx->recording || ctx->queue) return false;
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &st) != hipSuccess || st != hipStreamCaptureStatusNone) return false;
  return true;
}
}  // namespace

int64_t conv2d_wgrad_static_capacity_bytes() { return kStaticScratchFloats * 4; }

int conv2d_wgrad_static(Context* ctx, int dtype, const ConvShape& s, const void* x, const void* dy, float* dw, int splits,
                        int accumulate, int tile_cfg) {
  const int64_t cap = conv2d_wgrad_static_capacity_bytes();
  const int64_t per_split = conv2d_wgrad_workspace_bytes(s, dtype, 2) / 2;
  TCH_CHECK_ARG(per_split > 0, "conv2d_wgrad_static: empty filter");
  if (splits <= 0) {
    // the library's own choice, lowered to what the buffer holds (one split needs no partials at all)
    splits = conv2d_wgrad_pick_splits(s, dtype);
    if (splits > cap / per_split) splits = static_cast<int>(cap / per_split);
    if (splits < 2) splits = 1;
  } else if (splits > 1 && conv2d_wgrad_workspace_bytes(s, dtype, splits) > cap) {
    TCH_CHECK_ARG(false, "conv2d_wgrad_static: " + std::to_string(splits) + " splits of this filter need " +
                             std::to_string(conv2d_wgrad_workspace_bytes(s, dtype, splits)) +
                             " bytes of split-K partials, the static buffer holds " + std::to_string(cap));
  }
  float* ptr = nullptr;
  if (splits > 1)
    if (int rc = static_scratch(&ptr)) return rc;
  // Every partial element the reduction reads is written by the split kernels of the same call first, so
  // what an earlier call left in the buffer never shows; two calls that overlap on one GPU would race on it.
  if (splits <= 1) return conv2d_wgrad(ctx, dtype, s, x, dy, dw, ptr, splits, accumulate, tile_cfg);
  int dev = 0;
  (void)hipGetDevice(&dev);
  const hipStream_t stream = ctx->main_stream();
  const bool ordered = orders_itself(ctx, stream);
  std::lock_guard<std::mutex> lock(g_scratch_mu);   // two host threads do not interleave their launches either
  if (ordered && g_scratch_used[dev] && g_scratch_stream[dev] != stream)
    (void)hipStreamWaitEvent(stream, g_scratch_done[dev], 0);
  const int rc = conv2d_wgrad(ctx, dtype, s, x, dy, dw, ptr, splits, accumulate, tile_cfg);
  if (ordered && rc == 0 && hipEventRecord(g_scratch_done[dev], stream) == hipSuccess) {
    g_scratch_stream[dev] = stream;
    g_scratch_used[dev] = true;
  }
  return rc;
}

}  // namespace tch
