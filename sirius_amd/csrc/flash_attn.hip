// Fused attention for the GPT-2 step (bf16, head width 64): softmax(scale * Q K^T [+ causal mask]) V and its
// backward without ever writing the [T, T] score matrix.  What the reference runs here is transformers'
// GPT2Attention inside train/gpt2.py:26 (scores, mask, softmax, dropout p = 0 in the benchmark, context).
//
// Three kernels, all built from the same two MFMA products per step.  In each of them the workgroup keeps one
// side of the problem fixed (128 rows, 32 per wavefront, fragments in registers for the whole kernel) and walks
// over the other side in tiles of 64 rows staged in LDS:
//
//   forward   fixed: 32 queries / wave     walks keys     S^T = K Q^T,  O^T += V^T P^T
//   dQ        fixed: 32 queries / wave     walks keys     S^T, dP^T = V dO^T,  dQ^T += K^T dS^T
//   dK, dV    fixed: 32 keys / wave        walks queries  S = Q K^T, dP = dO V^T,  dV^T += dO^T P,  dK^T += Q^T dS
//
// The products are oriented so that the fixed side is the lane dimension of the 32x32 accumulator (lane % 32 =
// the fixed row, registers = the walked rows).  A row statistic of the fixed side (running maximum, sum, the
// saved log-sum-exp, delta = sum_d dO*O) is then one scalar per lane, a reduction over the walked rows runs over
// the lane's own registers plus one exchange with lane ^ 32, and the probabilities are already laid out as the
// second operand of the next product: the accumulator's registers 8s .. 8s+7 of a lane are 8 walked rows
// {16s + 8t + 4(lane/32) + i}, which is a permutation of the 16 reduction indices of one MFMA step; the other
// operand is read from LDS with the same permutation (transposing reads, ds_read_b64_tr_b16).
//
// A step stores its tiles to one of two buffers, so that one barrier a step is enough; a mask is applied behind a branch of the
// whole wavefront instead of in every score.  The key kernel has KG = 1 or 2 walk groups of four wavefronts: group g walks the
// tiles g, g + KG, .. for the same fixed rows, staged in LDS of its own, and the groups' accumulators are added at the end.
// What bounds them: with several workgroups on a CU the exponentials and what surrounds them, 960 of the 1470 cycles that a
// forward step's instructions take (96 heads of 1024: forward 32.9 -> 29.3 us, backward 82 -> 76); with one, the chain of steps (36
// heads of 777: 20.8 -> 15.7 and 46.8 -> 38.2).
//
// RAGGED (a sequence length that is no multiple of 128): the last fixed block and the last walked tile reach past the
// sequence.  Loads of rows beyond it fetch the last row again (no branch, always a finite value), and nothing is
// stored for them.  A walked key beyond the end is masked like a future key (a causal mask covers it already); a walked
// query beyond the end gets a log-sum-exp of +inf, so that its probabilities are exp2(-inf) = 0: the inner loops
// are those of the whole-tile form.  The whole-tile form keeps its own instantiation (no clamps in its address path).
// Against the three-launch chain over materialised scores that such lengths took before: 12 layers of 3 x 777
// tokens, forward + backward, 5.36 -> 0.7 ms (the step 10.7 -> 6.1 ms).
//
// Numerics: scores and statistics in fp32 from the bf16 products, exponentials as exp2 of pre-scaled values,
// probabilities rounded to bf16 for the second product (as the unfused path stores them).  The backward
// recomputes the probabilities from the saved log-sum-exp; dQ and (dK, dV) are two launches so that nothing is
// accumulated atomically and results do not depend on scheduling.
#include "attn_frag.h"
#include "kernels.h"
#include "ops.h"

namespace tch {
namespace {

constexpr int kHd = 64;          // head width
constexpr int kFixed = 128;      // rows of the fixed side per workgroup
constexpr int kWalk = 64;        // rows of the walked side per step
constexpr int kRowB = 144;       // LDS bytes per tile row: 64 bf16 + 16 bytes, so that 16 rows at one column
                                 // offset and the 4 x 32-byte patches of a transposing read spread over the banks
constexpr int kTileB = kWalk * kRowB;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

struct FlashArgs {
  const bf16* q;
  const bf16* k;
  const bf16* v;
  const bf16* o;      // backward
  const bf16* dout;   // backward
  bf16* out;          // forward: o; dQ kernel: dq
  bf16* dk;
  bf16* dv;
  float* lse;         // [B * H][T], natural logarithm
  float* delta;       // [B * H][T]
  int64_t qkv_rs, qkv_bs;   // row / sample strides of q, k, v, dq, dk, dv (elements); head h starts at column 64 h
  int64_t o_rs, o_bs;       // the same for o and dout
  int H, T;
  float scale;
};

// a [64][64] bf16 tile: global -> registers (two 16-byte chunks per thread) -> LDS rows of kRowB bytes
struct TileRegs {
  uint4 lo, hi;   // rows tid / 8 and 32 + tid / 8, slot tid % 8 (plain members: an array here ends up in scratch)
};
__device__ inline TileRegs tile_load(const bf16* base, int64_t rs, int tid) {
  const bf16* src = base + static_cast<int64_t>(tid >> 3) * rs + (tid & 7) * 8;
  TileRegs r;
  r.lo = *reinterpret_cast<const uint4*>(src);
  r.hi = *reinterpret_cast<const uint4*>(src + 32 * rs);
  return r;
}
// rows `first` .. `first` + 63 of a sequence of T rows; rows beyond it repeat the last one
template <bool RAGGED>
__device__ inline TileRegs tile_load_at(const bf16* base, int64_t rs, int first, int T, int tid) {
  if (!RAGGED) return tile_load(base + first * rs, rs, tid);
  const int r0 = first + (tid >> 3), r1 = r0 + 32;
  TileRegs r;
  r.lo = *reinterpret_cast<const uint4*>(base + (r0 < T ? r0 : T - 1) * rs + (tid & 7) * 8);
  r.hi = *reinterpret_cast<const uint4*>(base + (r1 < T ? r1 : T - 1) * rs + (tid & 7) * 8);
  return r;
}
__device__ inline void tile_store(unsigned char* lds, int tid, const TileRegs& r) {
  unsigned char* dst = lds + (tid >> 3) * kRowB + (tid & 7) * 16;
  *reinterpret_cast<uint4*>(dst) = r.lo;
  *reinterpret_cast<uint4*>(dst + 32 * kRowB) = r.hi;
}

// this wave's fragments of 32 fixed rows (row = first + lane % 32): 4 chunks cover the lane half's 32 columns
template <bool RAGGED>
__device__ inline void load_fixed(const bf16* base, int64_t rs, int first, int T, int lane, Chunk (&f)[4]) {
  int r = first + (lane & 31);
  if (RAGGED && r >= T) r = T - 1;
  const bf16* row = base + static_cast<int64_t>(r) * rs + 8 * (lane >> 5);
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) f[ks].u = *reinterpret_cast<const uint4*>(row + ks * 16);
}

// acc[ct] holds the transposed result: column 32 ct + 8 (r / 4) + 4 (lane / 32) + r % 4 of fixed row lane % 32.
// Goes through this wave's LDS patch so that a row leaves as 16-byte pieces.  T = 0: a wave that stores nothing.
__device__ inline void store_fixed(f32x16_t (&acc)[2], float mul, unsigned char* patch, bf16* base, int64_t rs, int first,
                                   int T, int lane) {
#pragma unroll
  for (int ct = 0; ct < 2; ++ct)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint2 w;
      w.x = pack_bf16(acc[ct][4 * j] * mul, acc[ct][4 * j + 1] * mul);
      w.y = pack_bf16(acc[ct][4 * j + 2] * mul, acc[ct][4 * j + 3] * mul);
      *reinterpret_cast<uint2*>(patch + (lane & 31) * kRowB + (32 * ct + 8 * j + 4 * (lane >> 5)) * 2) = w;
    }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int q = lane + 64 * i;
    const uint4 v = *reinterpret_cast<const uint4*>(patch + (q >> 3) * kRowB + (q & 7) * 16);
    if (first + (q >> 3) < T)
      *reinterpret_cast<uint4*>(base + static_cast<int64_t>(first + (q >> 3)) * rs + (q & 7) * 8) = v;
  }
}

// the workgroup's tiles: two buffers of one pair of tiles per walk group, later what join_groups hands over (32 KB)
template <int KG>
constexpr int flash_lds() {
  return 2 * KG * 2 * kTileB;
}

// ---------------------------------------------------------------------------------------------------------
// forward (DQ = false) and the dQ half of the backward (DQ = true): fixed queries, walked keys
// ---------------------------------------------------------------------------------------------------------
template <bool CAUSAL, bool DQ, bool RAGGED>
__global__ __launch_bounds__(256, 3) void flash_query_kernel(FlashArgs p) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[flash_lds<1>()];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, half = lane >> 5;
  // Workgroup ids go to the XCDs round-robin and most of them are resident at once, so the order is the
  // placement: the blocks of one head keep one residue of the id modulo 8 (one XCD, one L2 for its keys and
  // values), and the long blocks of a causal problem come first, so that the short ones fill what they leave.
  const int blocks = RAGGED ? (p.T + kFixed - 1) / kFixed : p.T / kFixed;
  const int nbh = gridDim.x / blocks;
  const int qb = blocks - 1 - blockIdx.x / nbh;
  const int bh = blockIdx.x % nbh;
  const int b = bh / p.H, h = bh - b * p.H;
  const int64_t qkv_off = b * p.qkv_bs + h * kHd, o_off = b * p.o_bs + h * kHd;
  const int q0 = qb * kFixed, qw0 = q0 + 32 * wave;
  const int query = qw0 + (lane & 31);
  const bool real = !RAGGED || query < p.T;
  const int64_t stat_at = static_cast<int64_t>(bh) * p.T + (real ? query : p.T - 1);

  const int tiles = RAGGED ? (p.T + kWalk - 1) / kWalk : p.T / kWalk;
  const int seen = (q0 + kFixed) / kWalk;   // tiles a causal block of queries sees
  const int steps = CAUSAL ? (RAGGED && seen > tiles ? tiles : seen) : tiles;
  const bf16* kbase = p.k + qkv_off;
  const bf16* vbase = p.v + qkv_off;
  TileRegs rk, rv;
  auto fetch = [&](int kb) {   // behind the last tile the last one again: no branch around the loads
    const int row = (kb < steps ? kb : steps - 1) * kWalk;
    rk = tile_load_at<RAGGED>(kbase, p.qkv_rs, row, p.T, tid);
    rv = tile_load_at<RAGGED>(vbase, p.qkv_rs, row, p.T, tid);
  };
  fetch(0);

  Chunk qf[4], dof[4];
  load_fixed<RAGGED>(p.q + qkv_off, p.qkv_rs, qw0, p.T, lane, qf);
  float lse2 = 0.f, delta = 0.f;
  if (DQ) {
    load_fixed<RAGGED>(p.dout + o_off, p.o_rs, qw0, p.T, lane, dof);
    Chunk of[4];
    load_fixed<RAGGED>(p.o + o_off, p.o_rs, qw0, p.T, lane, of);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      float a[8], g[8];
      chunk_to_float<bf16>(of[ks], a);
      chunk_to_float<bf16>(dof[ks], g);
#pragma unroll
      for (int e = 0; e < 8; ++e) delta += a[e] * g[e];
    }
    delta += __shfl_xor(delta, 32, 64);
    if (half == 0 && real) p.delta[stat_at] = delta;
    lse2 = p.lse[stat_at] * kLog2e;
  }

  f32x16_t acc[2];
  zero_acc(acc[0]);
  zero_acc(acc[1]);
  const float c = p.scale * kLog2e;
  float m = -INFINITY, l = 0.f;

  for (int kb = 0; kb < steps; ++kb) {
    unsigned char* kt = lds + (kb & 1) * 2 * kTileB;
    unsigned char* vt = kt + kTileB;
    tile_store(kt, tid, rk);
    tile_store(vt, tid, rv);
    // the one barrier of a step: whoever stores to the other buffer next has seen everyone through the step that read it
    __syncthreads();
    fetch(kb + 1);
    const int k0 = kb * kWalk;
    if (CAUSAL && k0 > qw0 + 31) continue;   // nothing of this tile is visible to this wave's queries

    // some key of the tile lies beyond some query, or beyond the sequence
    const bool diagonal = CAUSAL ? k0 + kWalk - 1 > qw0 : RAGGED && k0 + kWalk > p.T;
    const int last = (CAUSAL ? query : p.T - 1) - k0 - 4 * half;   // the last key this lane's query sees, from the lane's first
    if constexpr (!DQ) {
      f32x16_t s[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        zero_acc(s[t]);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) s[t] = mma16(frag_rows<kRowB>(kt, 32 * t, ks, lane), qf[ks], s[t]);
      }
      if (diagonal) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (32 * t + 8 * (r >> 2) + (r & 3) > last) s[t][r] = -INFINITY;
      }
      // running maximum on the raw scores (the scale is positive), then exp2(s * c - m * c) as one fused
      // multiply-add and one exponential per score
      float bmax = -INFINITY;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) bmax = fmaxf(bmax, s[t][r]);
      bmax = fmaxf(bmax, __shfl_xor(bmax, 32, 64));
      const float m_new = fmaxf(m, bmax);
      const bool moved = m_new != m;
      const float alpha = __builtin_amdgcn_exp2f((m - m_new) * c);
      m = m_new;
      const float mc = m_new * c;
      float sum = 0.f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          s[t][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][r], c, -mc));
          sum += s[t][r];
        }
      l = l * alpha + sum;
      // after the first tiles the maxima seldom move: the accumulators are rescaled only when one in the wave did
      if (__any(moved)) {
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[ct][e] *= alpha;
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int sl = 0; sl < 2; ++sl) {
          const Chunk pc = pack_half(s[t], sl);
#pragma unroll
          for (int ct = 0; ct < 2; ++ct) acc[ct] = mma16(frag_cols<kRowB>(vt, 32 * t + 16 * sl, ct, lane), pc, acc[ct]);
        }
    } else {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        f32x16_t s, dp;
        zero_acc(s);
        zero_acc(dp);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          s = mma16(frag_rows<kRowB>(kt, 32 * t, ks, lane), qf[ks], s);
          dp = mma16(frag_rows<kRowB>(vt, 32 * t, ks, lane), dof[ks], dp);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = __builtin_amdgcn_exp2f(s[r] * c - lse2);
        if (diagonal) {
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (32 * t + 8 * (r >> 2) + (r & 3) > last) s[r] = 0.f;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] *= dp[r] - delta;
#pragma unroll
        for (int sl = 0; sl < 2; ++sl) {
          const Chunk pc = pack_half(s, sl);
#pragma unroll
          for (int ct = 0; ct < 2; ++ct) acc[ct] = mma16(frag_cols<kRowB>(kt, 32 * t + 16 * sl, ct, lane), pc, acc[ct]);
        }
      }
    }
  }

  float mul = p.scale;
  if (!DQ) {
    l += __shfl_xor(l, 32, 64);
    mul = 1.f / l;
    if (half == 0 && real) p.lse[stat_at] = m * p.scale + __builtin_amdgcn_logf(l) * kLn2;
  }
  __syncthreads();   // every wave is done with the space: it becomes four output patches
  store_fixed(acc, mul, lds + wave * 32 * kRowB, p.out + (DQ ? qkv_off : o_off), DQ ? p.qkv_rs : p.o_rs, qw0, p.T,
                      lane);
}

// ---------------------------------------------------------------------------------------------------------
// dK and dV: fixed keys, walked queries
// ---------------------------------------------------------------------------------------------------------
// Adds the accumulators of walk group 1 to those of group 0.  Uses the LDS of the tiles; every wave calls it.
__device__ inline void join_groups(f32x16_t (&acc)[2], unsigned char* lds, int group, int wave, int lane) {
  float4* place = reinterpret_cast<float4*>(lds) + wave * 512 + lane;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const f32x16_t& v = acc[j >> 2];
    const int e = 4 * (j & 3);
    if (group == 1) place[64 * j] = make_float4(v[e], v[e + 1], v[e + 2], v[e + 3]);
  }
  __syncthreads();
  if (group == 1) return;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float4 v = place[64 * j];
    f32x16_t& to = acc[j >> 2];
    const int e = 4 * (j & 3);
    to[e] += v.x;
    to[e + 1] += v.y;
    to[e + 2] += v.z;
    to[e + 3] += v.w;
  }
}

template <bool CAUSAL, bool RAGGED, int KG>
__global__ __launch_bounds__(256 * KG, 2) void flash_key_kernel(FlashArgs p) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[flash_lds<KG>()];
  __shared__ __attribute__((aligned(16))) float stat[2][KG][2][kWalk];   // log-sum-exp (base 2) and delta of the staged queries
  const int lane = threadIdx.x & 63, tid = threadIdx.x & 255, wave = tid >> 6, half = lane >> 5;
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int nbh = gridDim.x / (RAGGED ? (p.T + kFixed - 1) / kFixed : p.T / kFixed);   // placement as in flash_query_kernel: early keys see most queries
  const int kblk = blockIdx.x / nbh;
  const int bh = blockIdx.x % nbh;
  const int b = bh / p.H, h = bh - b * p.H;
  const int64_t qkv_off = b * p.qkv_bs + h * kHd, o_off = b * p.o_bs + h * kHd;
  const int k0 = kblk * kFixed, kw0 = k0 + 32 * wave;
  const int key = kw0 + (lane & 31);

  const int first = CAUSAL ? k0 / kWalk : 0;   // queries before the first key see none of these keys
  const int steps = RAGGED ? (p.T + kWalk - 1) / kWalk : p.T / kWalk;
  const bf16* qbase = p.q + qkv_off;
  const bf16* dobase = p.dout + o_off;
  const float* lse = p.lse + static_cast<int64_t>(bh) * p.T;
  const float* dlt = p.delta + static_cast<int64_t>(bh) * p.T;
  TileRegs rq, rd;
  float rstat = 0.f;
  auto fetch = [&](int at_tile) {   // behind the last tile the last one again: no branch around the loads
    const int qb = at_tile < steps ? at_tile : steps - 1;
    rq = tile_load_at<RAGGED>(qbase, p.qkv_rs, qb * kWalk, p.T, tid);
    rd = tile_load_at<RAGGED>(dobase, p.o_rs, qb * kWalk, p.T, tid);
    const int row = qb * kWalk + (tid & (kWalk - 1));
    const bool real = !RAGGED || row < p.T;
    const int at = real ? row : p.T - 1;
    if (tid < kWalk) rstat = real ? lse[at] * kLog2e : INFINITY;
    else if (tid < 2 * kWalk) rstat = dlt[at];
  };
  fetch(first + group);

  Chunk kf[4], vf[4];
  load_fixed<RAGGED>(p.k + qkv_off, p.qkv_rs, kw0, p.T, lane, kf);
  load_fixed<RAGGED>(p.v + qkv_off, p.qkv_rs, kw0, p.T, lane, vf);

  f32x16_t dk[2], dv[2];
  zero_acc(dk[0]);
  zero_acc(dk[1]);
  zero_acc(dv[0]);
  zero_acc(dv[1]);
  const float c = p.scale * kLog2e;

  for (int qb0 = first, turn = 0; qb0 < steps; qb0 += KG, turn ^= 1) {
    const int qb = qb0 + group;
    unsigned char* qt = lds + (turn * KG + group) * 2 * kTileB;
    unsigned char* dot = qt + kTileB;
    float(&st)[2][kWalk] = stat[turn][group];
    tile_store(qt, tid, rq);
    tile_store(dot, tid, rd);
    if (tid < 2 * kWalk) st[tid >> 6][tid & 63] = rstat;
    __syncthreads();   // the one of a step, as in flash_query_kernel
    fetch(qb + KG);
    const int q0 = qb * kWalk;
    if (qb >= steps || (CAUSAL && q0 + kWalk - 1 < kw0)) continue;   // no (more) staged query sees this wave's keys

    const bool diagonal = CAUSAL && q0 < kw0 + 31;   // some staged query lies before some key of this wave
    const int before = key - q0 - 4 * half;          // the lane's queries below this one lie before its key
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      f32x16_t s, dp;
      zero_acc(s);
      zero_acc(dp);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        s = mma16(frag_rows<kRowB>(qt, 32 * t, ks, lane), kf[ks], s);
        dp = mma16(frag_rows<kRowB>(dot, 32 * t, ks, lane), vf[ks], dp);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float4 l4 = *reinterpret_cast<const float4*>(&st[0][32 * t + 8 * j + 4 * half]);
        const float ls[4] = {l4.x, l4.y, l4.z, l4.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) s[4 * j + i] = __builtin_amdgcn_exp2f(s[4 * j + i] * c - ls[i]);
      }
      if (diagonal) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (32 * t + 8 * (r >> 2) + (r & 3) < before) s[r] = 0.f;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float4 d4 = *reinterpret_cast<const float4*>(&st[1][32 * t + 8 * j + 4 * half]);
        const float dl[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) dp[4 * j + i] = s[4 * j + i] * (dp[4 * j + i] - dl[i]);
      }
#pragma unroll
      for (int sl = 0; sl < 2; ++sl) {
        const Chunk pc = pack_half(s, sl);
        const Chunk dc = pack_half(dp, sl);
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
          dv[ct] = mma16(frag_cols<kRowB>(dot, 32 * t + 16 * sl, ct, lane), pc, dv[ct]);
          dk[ct] = mma16(frag_cols<kRowB>(qt, 32 * t + 16 * sl, ct, lane), dc, dk[ct]);
        }
      }
    }
  }
  if (KG == 2) {
    join_groups(dv, lds, group, wave, lane);
    join_groups(dk, lds, group, wave, lane);
  }
  __syncthreads();
  unsigned char* patch = lds + (4 * group + wave) * 32 * kRowB;
  const int rows = group == 0 ? p.T : 0;
  store_fixed(dv, 1.f, patch, p.dv + qkv_off, p.qkv_rs, kw0, rows, lane);
  __syncthreads();
  store_fixed(dk, p.scale, patch, p.dk + qkv_off, p.qkv_rs, kw0, rows, lane);
}

int check_geometry(const char* who, int dtype, int B, int H, int T, int64_t qkv_rs, int64_t qkv_bs, int64_t o_rs,
                   int64_t o_bs, int any_length) {
  const std::string w(who);
  TCH_CHECK_ARG(dtype == kBF16, w + ": bf16 only");
  TCH_CHECK_ARG(B >= 1 && H >= 1 && T >= 1 && (any_length || T % kFixed == 0),
                w + ": the sequence length must be a multiple of 128");
  TCH_CHECK_ARG(T <= (1 << 30) && static_cast<int64_t>(B) * H * ((T + kFixed - 1) / kFixed) < (1ll << 31),
                w + ": too many blocks for one grid");
  TCH_CHECK_ARG(qkv_rs >= static_cast<int64_t>(H) * kHd && o_rs >= static_cast<int64_t>(H) * kHd,
                w + ": row strides shorter than the heads");
  TCH_CHECK_ARG(qkv_rs % 8 == 0 && qkv_bs % 8 == 0 && o_rs % 8 == 0 && o_bs % 8 == 0,
                w + ": strides must keep 16-byte alignment");
  return 0;
}

// Workgroups that share one CU hide each other's latencies; one that is alone on it lives off its own wavefronts, and two groups
// halve its chain of steps.  dK and dV with one group / two, in us more or less than one: 36 heads of 777 (252 workgroups) -4, 12
// of 1024 (96) -5, 24 of 512 (96) -2, 96 of 256 (192) 0; 96 of 512 (384) +5, 96 of 1024 (768) +6.  (The two query kernels gain less:
// groups of 36 heads of 777 dQ -1.3, forward -2 with three of them; and with one their results are those they always were.)
bool split_walk(const dim3& grid, int T) { return grid.x <= 256 && T > 5 * kWalk; }

template <bool DQ>
void (*query_kernel(bool causal, bool ragged))(FlashArgs) {
  return causal ? (ragged ? flash_query_kernel<true, DQ, true> : flash_query_kernel<true, DQ, false>)
                : (ragged ? flash_query_kernel<false, DQ, true> : flash_query_kernel<false, DQ, false>);
}
template <int KG>
void (*key_kernel(bool causal, bool ragged))(FlashArgs) {
  return causal ? (ragged ? flash_key_kernel<true, true, KG> : flash_key_kernel<true, false, KG>)
                : (ragged ? flash_key_kernel<false, true, KG> : flash_key_kernel<false, false, KG>);
}

bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }

}  // namespace

int flash_attn_fwd(Context* ctx, int dtype, const void* q, const void* k, const void* v, void* o, float* lse, int B,
                   int H, int T, int64_t qkv_rs, int64_t qkv_bs, int64_t o_rs, int64_t o_bs, float scale, int causal,
                   int any_length) {
  if (int rc = check_geometry("flash_attn_fwd", dtype, B, H, T, qkv_rs, qkv_bs, o_rs, o_bs, any_length)) return rc;
  TCH_CHECK_ARG(q && k && v && o && lse, "flash_attn_fwd: null tensor");
  TCH_CHECK_ARG(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(o), "flash_attn_fwd: tensors must be 16-byte aligned");
  FlashArgs a{};
  a.q = static_cast<const bf16*>(q);
  a.k = static_cast<const bf16*>(k);
  a.v = static_cast<const bf16*>(v);
  a.out = static_cast<bf16*>(o);
  a.lse = lse;
  a.qkv_rs = qkv_rs;
  a.qkv_bs = qkv_bs;
  a.o_rs = o_rs;
  a.o_bs = o_bs;
  a.H = H;
  a.T = T;
  a.scale = scale;
  const dim3 grid(static_cast<unsigned>((T + kFixed - 1) / kFixed) * B * H);
  const double flops = 4.0 * B * H * static_cast<double>(T) * T * kHd * (causal ? 0.5 : 1.0);
  const bool ragged = T % kFixed != 0;
  return launch(ctx, query_kernel<false>(causal, ragged), grid, dim3(256), a, causal ? "flash_attn_fwd<causal>" : "flash_attn_fwd<full>",
                flops, 0);
}

int flash_attn_bwd(Context* ctx, int dtype, const void* q, const void* k, const void* v, const void* o, const void* dout,
                   const float* lse, float* delta, void* dq, void* dk, void* dv, int B, int H, int T, int64_t qkv_rs,
                   int64_t qkv_bs, int64_t o_rs, int64_t o_bs, float scale, int causal, int any_length) {
  if (int rc = check_geometry("flash_attn_bwd", dtype, B, H, T, qkv_rs, qkv_bs, o_rs, o_bs, any_length)) return rc;
  TCH_CHECK_ARG(q && k && v && o && dout && lse && delta && dq && dk && dv, "flash_attn_bwd: null tensor");
  TCH_CHECK_ARG(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(o) && aligned16(dout) && aligned16(dq) &&
                    aligned16(dk) && aligned16(dv),
                "flash_attn_bwd: tensors must be 16-byte aligned");
  FlashArgs a{};
  a.q = static_cast<const bf16*>(q);
  a.k = static_cast<const bf16*>(k);
  a.v = static_cast<const bf16*>(v);
  a.o = static_cast<const bf16*>(o);
  a.dout = static_cast<const bf16*>(dout);
  a.out = static_cast<bf16*>(dq);
  a.dk = static_cast<bf16*>(dk);
  a.dv = static_cast<bf16*>(dv);
  a.lse = const_cast<float*>(lse);
  a.delta = delta;
  a.qkv_rs = qkv_rs;
  a.qkv_bs = qkv_bs;
  a.o_rs = o_rs;
  a.o_bs = o_bs;
  a.H = H;
  a.T = T;
  a.scale = scale;
  const dim3 grid(static_cast<unsigned>((T + kFixed - 1) / kFixed) * B * H);
  const double pair = 2.0 * B * H * static_cast<double>(T) * T * kHd * (causal ? 0.5 : 1.0);   // one T x T x 64 product
  // the dQ launch leaves delta for the dK / dV launch
  const bool ragged = T % kFixed != 0;
  const bool split = split_walk(grid, T);
  if (int rc = launch(ctx, query_kernel<true>(causal, ragged), grid, dim3(256), a,
                      causal ? "flash_attn_dq<causal>" : "flash_attn_dq<full>", 3.0 * pair, 0))
    return rc;
  return launch(ctx, split ? key_kernel<2>(causal, ragged) : key_kernel<1>(causal, ragged), grid, dim3(split ? 512 : 256), a,
                causal ? "flash_attn_dkv<causal>" : "flash_attn_dkv<full>", 4.0 * pair, 0);
}

}  // namespace tch
