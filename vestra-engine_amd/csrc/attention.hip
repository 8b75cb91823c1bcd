// Scaled dot-product attention for gfx950, F32 in / F32 accumulate:
// out = softmax(Q K^T / sqrt(64)) V over independent head-major sequences
// [n, 64] (a head of one view for local layers, a head of the whole flattened
// multi-view sequence for global layers), with an online (one-pass) softmax.
//
// Both products run on the f16 matrix cores as three products of two-part
// splits (split_f16.h), scaled so that the remainders stay normal numbers:
// one accumulator, the small products first.
//
// A workgroup of eight waves (or four, attention_plan) owns 32 queries a wave of
// one sequence.  Grids of few tiles split the key blocks of each tile over
// several workgroups and merge the partial results in a second pass
// (attention_kernel<true, *>, attention_merge_kernel).  Keys and values stream
// through LDS in blocks of 64 as f16 parts, split once per workgroup by the
// thread that loaded them: K as [key][part][d] rows, V transposed as
// [d][part][key] rows, both with a pitch of 272 bytes (16 x odd: fragment
// reads of consecutive rows are bank-conflict free).  Two buffers, loads a
// block ahead in registers, one barrier a block.
//
// Per key block a wave runs 48 v_mfma_f32_32x32x16_f16:
//  * S^T = K Q^T (A = K, B = Q^T).  The transposed product leaves, in lane l,
//    the scores of query l%32 for keys 32t + 8(r/4) + 4(l/32) + r%4 of key
//    tile t; the row max and sum of a query are in-register plus one exchange
//    with lane l ^ 32.
//  * O^T += V^T P^T (A = V^T, B = P^T).  Key slots of a 16-key chunk are
//    numbered so that lane l's eight slots are the eight keys whose weights it
//    already holds: P never leaves registers, and V^T is stored in that order.
//    O^T's columns are the lane's own query: rescales and the final division
//    need no exchange.
// Scores are kept in the base-2 domain: Q is pre-scaled by log2(e)/sqrt(64), so
// every softmax weight is one v_exp_f32 (2^x) of an FMA of the score.  The
// running maximum is only moved when a score passes it by more than 2^kSlack;
// the weights carry 2^kPBits so that small ones keep both parts.
// Keys past n are masked to -inf (last block only); queries past n are
// computed on a clamped row and not stored.
//
// What bounds it: per block and wave 1,536 cycles of MFMA against about 1,300
// of VALU (32 weights a lane: FMA, exp, sum, split; the staging's conversions)
// and, per CU, 2 x 34 KiB of fragment reads a wave pair from LDS.  12 x 10,392
// rows: 920 us, 361 TFLOP/s of the product's own FLOP = 1,082 of f16 MFMA, 87%
// of what a large f16 library product reaches on the card; with F32 matrix
// instructions 2,478 us.  128-query workgroups there stage twice as often:
// 1,064 us.
//
// A query that the split does not hold (a result that is not finite, or one
// that is small beside V's columns, kHeldSum) is computed again with F32 matrix
// instructions by its workgroup, alone: a query's bits depend on its own row and
// its sequence's K and V only (attention_tile_f32).
// V of any scale runs at full speed (12 x 866, V x 1e-4: 25 us; judged by one
// fixed scale 55).  A launch that takes every query again: 12 x 10,392 3.3 ms
// where K does not fit from the first block on, 3.9 ms where one late value of K
// or V does not (F32 matrix instructions alone 2.5); 12 x 866 50-53 us (35).
// What an output may then be off beside F32's rounding: 2^-34 of its V column's
// largest value in the run's first key block, and 2^-23 of the largest of its
// query's 64 (each measured against its column).
#include <cmath>

#include "common.h"
#include "split_f16.h"

namespace {

using vks::f32x16;
using vks::f32x4;
using vks::u32x4;

constexpr int HD = vk::kHeadDim;
constexpr int KB = vk::kKeyBlock;  // keys per block
constexpr int PITCH = 68;
constexpr int kSlots = KB * HD / 4;  // float4 of one K (or V) block: 1024
constexpr float kQScale = 0.125f * 1.44269504088896341f;  // log2(e) / sqrt(64)
// Scales of the f16 parts (powers of two): K by 2^8, Q (with kQScale) by 2^10,
// the weights by 2^11 with room for a factor 2^2 above the running max (2^4 saves
// a few rescales, 0.5% at 12 x 10,392, but leaves more weights where the exponent's
// argument is rounded at 2^-21: 3.95e-7 of the 64-bit result at 12 x 866 against
// 3.88e-7; f16 holds 2^4).  |k| of
// 256 and |q| of 354 no longer fit (queries that meet them run in F32).  A
// column of V is brought to [2^kVBits, 2 x that) by the largest value of the
// run's first key block; one of 64 to 128 times that no longer fits.
constexpr float kKUp = 256.0f, kQUp = 1024.0f, kSDown = 1.0f / 262144.0f;
constexpr float kPBits = 11.0f, kPDown = 1.0f / 2048.0f, kSlack = 2.0f;
constexpr int kVBits = 9;
// A query is held whose largest sum m (of 64, over scaled V and weights of sum l)
// has m >= kHeldSum and m^2 >= kHeldSquare l.  The floors are 2^-25 of every scaled
// value of V and of every weight, of random sign: V's add up to 2^-25 sqrt(sum
// p^2) <= 2^-25 sqrt(2^13 l), the largest weight being at most 2^13, which the
// second keeps below 2^-24 m; the weights' to 2^-25 sqrt(n) of V's usual size
// (2^8), below 2^-24 m for n = 4,096 by the first.  (l / 2 in place of its root took
// queries again that attend evenly to 10,000 keys beside a few with larger V.)
constexpr float kHeldSquare = 2048.0f, kHeldSum = 8192.0f;
constexpr int kFlush = 8;       // blocks between additions to the running total
constexpr int kRowBytes = 272;  // LDS pitch of 64 values: 2 parts x 128 bytes + 16
constexpr int kBufBytes = 2 * KB * kRowBytes;  // a block of K and of V
static_assert(PITCH % 4 == 0 && (PITCH / 4) % 2 == 1, "pitch 4 x odd");
static_assert(PITCH % 16 == 4, "transposed V stores: 16 (l >> 4) + (l & 15) covers 64 banks");

// Max and sum over the lanes l, l ^ 16, l ^ 32, l ^ 48 (the four lane groups
// of one query column).  v_permlane16_swap / v_permlane32_swap with both
// operands v leave each lane its own value and that of lane l ^ 16 (l ^ 32)
// in the two results: a VALU exchange, with no LDS round trip.  Both
// operations are commutative, so the result has the bits of the butterfly
// v op shfl_xor(v, 16), then op shfl_xor(., 32).
__device__ __forceinline__ float xor16_pair(float v, float* other) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v),
                                                  false, false);
  *other = __uint_as_float(r[1]);
  return __uint_as_float(r[0]);
}

__device__ __forceinline__ float xor32_pair(float v, float* other) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v),
                                                  false, false);
  *other = __uint_as_float(r[1]);
  return __uint_as_float(r[0]);
}

__device__ __forceinline__ float group_max(float v) {
  float o;
  v = xor16_pair(v, &o);
  v = fmaxf(v, o);
  v = xor32_pair(v, &o);
  return fmaxf(v, o);
}

__device__ __forceinline__ float group_sum(float v) {
  float o;
  v = xor16_pair(v, &o);
  v = v + o;
  v = xor32_pair(v, &o);
  return v + o;
}

// Largest |value| over a thread's four and over its row of 16 lanes.
__device__ __forceinline__ float row16_max(float v) {
#define VK_ROR(n)                                                                             \
  v = fmaxf(v, __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(v), 0x120 | n, 0xf, \
                                                        0xf, true)));
  VK_ROR(8) VK_ROR(4) VK_ROR(2) VK_ROR(1)
#undef VK_ROR
  return v;
}

__device__ __forceinline__ float column_max(float a, float b, float c, float d) {
  return row16_max(fmaxf(fmaxf(fabsf(a), fabsf(b)), fmaxf(fabsf(c), fabsf(d))));
}

__device__ __forceinline__ void split8_plain(const f32x4& x, const f32x4& y, u32x4* p0, u32x4* p1) {
  uint32_t h[4], l[4];
  vks::split2_plain(x[0], x[1], &h[0], &l[0]);
  vks::split2_plain(x[2], x[3], &h[1], &l[1]);
  vks::split2_plain(y[0], y[1], &h[2], &l[2]);
  vks::split2_plain(y[2], y[3], &h[3], &l[3]);
  *p0 = u32x4{h[0], h[1], h[2], h[3]};
  *p1 = u32x4{l[0], l[1], l[2], l[3]};
}

// 16 queries a wave with F32 matrix instructions, for those that the split does
// not hold: bit i of `mask` says whether the wave's query i is stored (a wave
// without any only helps to stage).  In the k-permuted fragment order (lane
// group g holds k = 16 b + 4 g + j in component j, MFMA step j takes component
// j) the A operand of key tile t is the lane's four probabilities of that
// tile; K is staged as [key][d] and V as [d][key] rows of 68 floats.
template <bool PART, int kThreads>
__device__ __forceinline__ void attention_tile_f32(
    float* smem, const float* __restrict__ q, const float* __restrict__ k,
    const float* __restrict__ v, float* __restrict__ out, int sequences, int n, int seq, int qb,
    int kb_begin, int kb_end, int split, int splits, float* __restrict__ part, uint32_t mask) {
  constexpr int kPer = kSlots / kThreads;  // staged float4 of K (and of V) per thread
  constexpr int QG = kThreads / 64;

  const int tid = threadIdx.x;
  __builtin_assume(tid < kThreads);
  const int wave = tid >> 6, lane = tid & 63;
  const int wq = wave;  // query group
  const int g = lane >> 4, c16 = lane & 15;
  float* Ks = smem;
  float* Vt = Ks + KB * PITCH;
  const int q0 = qb + wq * 16;
  const bool live = mask != 0 && q0 < n;  // uniform over the wave
  const size_t base = static_cast<size_t>(seq) * n * HD;

  // Q^T fragments (B operand): query q0 + c16, d = 16 bd + 4 g + j
  f32x4 qf[4];
  {
    const int qi = q0 + c16 < n ? q0 + c16 : n - 1;
    const float* qrow = q + base + static_cast<size_t>(qi) * HD + 4 * g;
#pragma unroll
    for (int bd = 0; bd < 4; ++bd) {
      const f32x4 t = *reinterpret_cast<const f32x4*>(qrow + 16 * bd);
      qf[bd] = t * kQScale;
    }
  }

  f32x4 o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.0f;  // statistics of query q0 + c16

  // K staging: slot f = tid + 256 i is key f/16, float4 f%16 (16 lanes fill
  // one key row).  V staging: slot f -> w' = f/64, key 16 (w' % 4) + (l & 15),
  // float4 column (l >> 4) + 4 (w' / 4); one wave instruction covers 16 keys
  // x 4 columns.
  const int skey = tid >> 4, sd = 4 * (tid & 15);
  const float* karow = Ks + c16 * PITCH + 4 * g;
  const float* vtrow = Vt + c16 * PITCH + 4 * g;
  // Whole key blocks load through buffer resources: the lane's byte offset
  // inside a block is fixed, the block's offset is uniform, so the loads
  // carry no per-block vector address arithmetic.  (The kernel's tensors
  // are under 4 GiB, checked at launch.)
  const uint32_t bytes = 4u * static_cast<uint32_t>(sequences) * static_cast<uint32_t>(n) * HD;
  const __amdgpu_buffer_rsrc_t k_rsrc = vkd::buffer_rsrc(k, bytes);
  const __amdgpu_buffer_rsrc_t v_rsrc = vkd::buffer_rsrc(v, bytes);
  uint32_t k_off[kPer], v_off[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    k_off[i] = 4u * static_cast<uint32_t>((skey + (kThreads / 16) * i) * HD + sd);
    const int w2 = wq + QG * i;
    v_off[i] = 4u * static_cast<uint32_t>((16 * (w2 & 3) + (lane & 15)) * HD +
                                          4 * ((lane >> 4) + 4 * (w2 >> 2)));
  }

  for (int kb = kb_begin; kb < kb_end; ++kb) {
    const int k0 = kb * KB;
    f32x4 kr[kPer], vr[kPer];
    if (k0 + KB <= n) {
      const uint32_t blk = 4u * (static_cast<uint32_t>(seq) * static_cast<uint32_t>(n) +
                                 static_cast<uint32_t>(k0)) * HD;
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const float4 a = vkd::buffer_load4(k_rsrc, k_off[i], blk);
        const float4 b = vkd::buffer_load4(v_rsrc, v_off[i], blk);
        kr[i] = f32x4{a.x, a.y, a.z, a.w};
        vr[i] = f32x4{b.x, b.y, b.z, b.w};
      }
    } else {  // the last, partial block: keys past n read key n - 1
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int key = k0 + skey + (kThreads / 16) * i;
        const int ck = key < n ? key : n - 1;
        kr[i] = *reinterpret_cast<const f32x4*>(k + base + static_cast<size_t>(ck) * HD + sd);
        const int w2 = wq + QG * i;
        const int vkey = k0 + 16 * (w2 & 3) + (lane & 15);
        const int cv = vkey < n ? vkey : n - 1;
        vr[i] = *reinterpret_cast<const f32x4*>(v + base + static_cast<size_t>(cv) * HD +
                                                4 * ((lane >> 4) + 4 * (w2 >> 2)));
      }
    }
    __syncthreads();  // the previous block is consumed
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      *reinterpret_cast<f32x4*>(Ks + (skey + (kThreads / 16) * i) * PITCH + sd) = kr[i];
      const int w2 = wq + QG * i;
      const int key = 16 * (w2 & 3) + (lane & 15);
      const int d = 4 * ((lane >> 4) + 4 * (w2 >> 2));
#pragma unroll
      for (int c = 0; c < 4; ++c) Vt[(d + c) * PITCH + key] = vr[i][c];
    }
    __syncthreads();
    if (!live) continue;

    // S^T tiles: s[t][r] = score of query q0 + c16 with key k0 + 16t + 4g + r
    // (K fragments of tile t + 1 are read while tile t's 16 MFMAs run)
    f32x4 s[4], ka[2][4];
#pragma unroll
    for (int bd = 0; bd < 4; ++bd)
      ka[0][bd] = *reinterpret_cast<const f32x4*>(karow + 16 * bd);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (t < 3) {
#pragma unroll
        for (int bd = 0; bd < 4; ++bd)
          ka[(t + 1) & 1][bd] =
              *reinterpret_cast<const f32x4*>(karow + (t + 1) * 16 * PITCH + 16 * bd);
      }
      __builtin_amdgcn_sched_barrier(0);
      s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int bd = 0; bd < 4; ++bd)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[t & 1][bd][j], qf[bd][j], s[t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (k0 + KB > n) {  // the last, partial block
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (k0 + 16 * t + 4 * g + r >= n) s[t][r] = -INFINITY;
    }
    float mb = -INFINITY;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) mb = fmaxf(mb, s[t][r]);
    const float m_new = fmaxf(m_run, group_max(mb));
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);  // 0 on the first block
    float ps = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[t][r] = __builtin_amdgcn_exp2f(s[t][r] - m_new);
        ps += s[t][r];
      }
    l_run = l_run * alpha + group_sum(ps);
    m_run = m_new;

    // rescale O: row 4g + r belongs to query q0 + 4g + r, whose factor sits
    // in lane 4g + r.  Skipped when every factor of the wave is exactly 1 (no
    // row maximum grew): multiplying by 1 changes no bits.
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float ar = __shfl(alpha, 4 * g + r, 64);
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) o[dt][r] *= ar;
      }
    }
    // O += P V: A = the lane's probabilities of key tile t, B = V^T rows
    // (V^T fragments of column tile dt + 1 are read while dt's MFMAs run)
    f32x4 vb[2][4];
#pragma unroll
    for (int t = 0; t < 4; ++t) vb[0][t] = *reinterpret_cast<const f32x4*>(vtrow + 16 * t);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      if (dt < 3) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
          vb[(dt + 1) & 1][t] =
              *reinterpret_cast<const f32x4*>(vtrow + (dt + 1) * 16 * PITCH + 16 * t);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(s[t][j], vb[dt & 1][t][j], o[dt], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  if (!live) return;
  if constexpr (PART) {
    // this split's O (rescaled to its own running max), max and sum
    const size_t rows = static_cast<size_t>(sequences) * n;
    float* po = part + (static_cast<size_t>(split) * rows + static_cast<size_t>(seq) * n) * HD;
    float* pml = part + static_cast<size_t>(splits) * rows * HD +
                 (static_cast<size_t>(split) * rows + static_cast<size_t>(seq) * n) * 2;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int qi = q0 + 4 * g + r;
      if (qi < n && ((mask >> (4 * g + r)) & 1)) {
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) po[static_cast<size_t>(qi) * HD + 16 * dt + c16] = o[dt][r];
      }
    }
    if (g == 0 && q0 + c16 < n && ((mask >> c16) & 1))
      *reinterpret_cast<float2*>(pml + 2 * static_cast<size_t>(q0 + c16)) =
          make_float2(m_run, l_run);
    return;
  }

  // out[query][d] = O / l, O row 4g + r, column 16 dt + c16
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float lr = __shfl(l_run, 4 * g + r, 64);
    const int qi = q0 + 4 * g + r;
    if (qi < n && ((mask >> (4 * g + r)) & 1)) {
      float* orow = out + base + static_cast<size_t>(qi) * HD + c16;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) orow[16 * dt] = o[dt][r] / lr;
    }
  }
}


// A workgroup of QW waves, 32 queries each, over every key block.  PART: the
// key blocks of each query tile are split into `splits` contiguous runs, one
// workgroup each; a run writes its O (scaled to its own running max), the max
// and the sum to `part` ([splits][rows][64], then [splits][rows][2]) and
// attention_merge_kernel combines them in split order.
template <bool PART, int QW>
__global__ __launch_bounds__(64 * QW, 2) void attention_kernel(const float* __restrict__ q,
                                                               const float* __restrict__ k,
                                                               const float* __restrict__ v,
                                                               float* __restrict__ out,
                                                               int sequences, int n, int splits,
                                                               float* __restrict__ part) {
  constexpr int kThreads = 64 * QW;
  constexpr int QB = 32 * QW;  // queries per workgroup
  static_assert(QW == 4 || QW == 8, "four or eight waves");
  // with eight waves the first four stage V and the others K
  constexpr bool kShared = QW == 8;
  __shared__ __align__(16) char smem[2 * kBufBytes];
  __shared__ __align__(16) float vdown[HD];
  __shared__ uint32_t flags[QW];  // per wave: its queries to compute again

  const int tid = threadIdx.x;
  __builtin_assume(tid < kThreads);
  const int wave = tid >> 6, lane = tid & 63;
  const int half = lane >> 5, c32 = lane & 31;
  const int nqb = (n + QB - 1) / QB;
  // XCD-major numbering: the query blocks of one sequence share an XCD's L2
  const int tile_all = vkd::xcd_tile(blockIdx.x, gridDim.x);
  const int split = PART ? tile_all % splits : 0;
  const int tile = PART ? tile_all / splits : tile_all;
  const int seq = tile / nqb, qb = (tile % nqb) * QB;
  const int q0 = qb + 32 * wave;
  const bool live = q0 < n;  // uniform over the wave
  const size_t base = static_cast<size_t>(seq) * n * HD;
  const int nkb = (n + KB - 1) / KB;
  const int kb_begin = PART ? static_cast<int>(static_cast<long long>(split) * nkb / splits) : 0;
  const int kb_end =
      PART ? static_cast<int>(static_cast<long long>(split + 1) * nkb / splits) : nkb;

  // O^T: d = 32 dt + 8 (r / 4) + 4 half + r % 4 of query q0 + c32.  Blocks add
  // to `o`, which moves to `total` every kFlush of them: a value is rounded 12
  // times a block at the size of a few blocks, and then once per kFlush at
  // that of the whole sum.
  f32x16 o[2], total[2];
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = total[dt][r] = 0.0f;
  float m_run = -INFINITY;  // running max of query q0 + c32 (both halves alike)
  float l_run = 0.0f;       // sum over the keys that this lane holds

  // Staging, one block ahead through registers.  K: piece s = 8 floats, key
  // s / 8, d 8 (s % 8).. ; V: 4 keys x 4 d per thread (its lanes in key order:
  // a transposed 8-byte store of 16 lanes fills one 128-byte row).  Keys past
  // n read past the sequence's buffer, which gives zeros (the block's offset
  // is part of the lane's: the uniform offset is left out of bounds checks).
  const int st = kShared ? tid & 255 : tid;
  const bool upper = kShared && __builtin_amdgcn_readfirstlane(wave) >= 4;
  const uint32_t bytes = 4u * static_cast<uint32_t>(n) * HD;
  const int quad = st & 15, d4 = st >> 4;
  // byte offsets of piece st, float4 i, in a block of K and of V
  auto k_off = [&](int i) {
    return 4u * static_cast<uint32_t>(((st >> 3) + 32 * (i >> 1)) * HD + 8 * (st & 7) + 4 * (i & 1));
  };
  auto v_off = [&](int i) { return 4u * static_cast<uint32_t>((4 * quad + i) * HD + 4 * d4); };
  const __amdgpu_buffer_rsrc_t rsrc0 = vkd::buffer_rsrc((upper ? k : v) + base, bytes);
  const __amdgpu_buffer_rsrc_t rsrc1 = vkd::buffer_rsrc(k + base, bytes);
  uint32_t off0[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) off0[i] = upper ? k_off(i) : v_off(i);
  float4 r0[4], r1[4];  // V (the upper waves: K), and K where a thread stages both
  auto load_block = [&](int kb) {
    const uint32_t blk = static_cast<uint32_t>(kb) * KB * HD * 4u;
#pragma unroll
    for (int i = 0; i < 4; ++i) r0[i] = vkd::buffer_load4(rsrc0, blk + off0[i], 0);
    if constexpr (!kShared) {
#pragma unroll
      for (int i = 0; i < 4; ++i) r1[i] = vkd::buffer_load4(rsrc1, blk + k_off(i), 0);
    }
  };
  load_block(kb_begin);

  // The scale of V's columns 4 d4 .. + 3: the block's largest values (a thread
  // holds four keys of them, its row of 16 lanes all 64), to the queries' waves
  // through LDS as 1 / scale.  A column of zeros takes the largest scale: any
  // value met later is beyond f16, or else too small for any other scale.
  uint32_t vup = 0;  // the four scales' exponent fields, a byte each
  if (!upper) {
    const float m4[4] = {column_max(r0[0].x, r0[1].x, r0[2].x, r0[3].x),
                         column_max(r0[0].y, r0[1].y, r0[2].y, r0[3].y),
                         column_max(r0[0].z, r0[1].z, r0[2].z, r0[3].z),
                         column_max(r0[0].w, r0[1].w, r0[2].w, r0[3].w)};
    float down[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int b = static_cast<int>(__float_as_uint(m4[c]) >> 23);
      int e = kVBits + 127 - b;
      e = b == 255 ? 0 : (m4[c] == 0.0f || e > 126 ? 126 : e);
      vup |= static_cast<uint32_t>(127 + e) << (8 * c);
      down[c] = __uint_as_float(static_cast<uint32_t>(127 - e) << 23);
    }
    if (quad == 0) *reinterpret_cast<float4*>(vdown + 4 * d4) =
        make_float4(down[0], down[1], down[2], down[3]);
  }

  // Q^T fragments (B operand): query q0 + c32, d = 16 ks + 8 half + j
  u32x4 qf[4][2];
  {
    const int qi = q0 + c32 < n ? q0 + c32 : n - 1;
    const float* qrow = q + base + static_cast<size_t>(qi) * HD + 8 * half;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(qrow + 16 * ks) * kQScale * kQUp;
      const f32x4 b = *reinterpret_cast<const f32x4*>(qrow + 16 * ks + 4) * kQScale * kQUp;
      split8_plain(a, b, &qf[ks][0], &qf[ks][1]);
    }
  }

  char* k_dst = smem + (st >> 3) * kRowBytes + 16 * (st & 7);
  // V^T row d: [part][4 chunks of 16 keys], quad order 0 2 1 3 in a chunk
  char* v_dst = smem + KB * kRowBytes + 4 * d4 * kRowBytes + 32 * (quad >> 2) +
                16 * (quad & 1) + 8 * ((quad >> 1) & 1);
  auto store_k = [&](int buf, const float4 (&kr)[4]) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float4 x = kr[2 * i], y = kr[2 * i + 1];
      u32x4 p0, p1;
      split8_plain(f32x4{x.x, x.y, x.z, x.w} * kKUp, f32x4{y.x, y.y, y.z, y.w} * kKUp, &p0, &p1);
      char* d = k_dst + buf * kBufBytes + 32 * i * kRowBytes;
      *reinterpret_cast<u32x4*>(d) = p0;
      *reinterpret_cast<u32x4*>(d + 128) = p1;
    }
  };
  auto store_v4 = [&](char* d, float up, float a, float b, float e, float f) {
    uint32_t p0[2], p1[2];
    vks::split2_plain(a * up, b * up, &p0[0], &p1[0]);
    vks::split2_plain(e * up, f * up, &p0[1], &p1[1]);
    *reinterpret_cast<uint2*>(d) = make_uint2(p0[0], p0[1]);
    *reinterpret_cast<uint2*>(d + 128) = make_uint2(p1[0], p1[1]);
  };
  auto store_v = [&](int buf, const float4 (&vr)[4]) {
    char* d = v_dst + buf * kBufBytes;
    auto up = [&](int c) { return __uint_as_float(((vup >> (8 * c)) & 0xffu) << 23); };
    store_v4(d, up(0), vr[0].x, vr[1].x, vr[2].x, vr[3].x);
    store_v4(d + kRowBytes, up(1), vr[0].y, vr[1].y, vr[2].y, vr[3].y);
    store_v4(d + 2 * kRowBytes, up(2), vr[0].z, vr[1].z, vr[2].z, vr[3].z);
    store_v4(d + 3 * kRowBytes, up(3), vr[0].w, vr[1].w, vr[2].w, vr[3].w);
  };
  auto store_block = [&](int buf) {
    if (upper) {
      store_k(buf, r0);
    } else {
      store_v(buf, r0);
      if constexpr (!kShared) store_k(buf, r1);
    }
  };

  const char* kfrag = smem + c32 * kRowBytes + 16 * half;
  const char* vfrag = kfrag + KB * kRowBytes;
  auto compute = [&](int kb, int buf) {
    // S^T: s[t][r] = score of query q0 + c32 with key 32 t + 8 (r / 4) +
    // 4 half + r % 4 of the block; small products first
    f32x16 s[2];
    u32x4 k0f[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[t][r] = 0.0f;
    const char* kf = kfrag + buf * kBufBytes;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const char* f = kf + 32 * t * kRowBytes + 32 * ks;
        k0f[t][ks] = *reinterpret_cast<const u32x4*>(f);
        const u32x4 k1 = *reinterpret_cast<const u32x4*>(f + 128);
        s[t] = vks::mfma32(k1, qf[ks][0], s[t]);
        s[t] = vks::mfma32(k0f[t][ks], qf[ks][1], s[t]);
      }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int t = 0; t < 2; ++t) s[t] = vks::mfma32(k0f[t][ks], qf[ks][0], s[t]);
    const int left = n - kb * KB;
    if (left < KB) {  // the last, partial block
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (32 * t + 8 * (r / 4) + 4 * half + r % 4 >= left) s[t][r] = -INFINITY;
    }
    float mb = s[0][0];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) mb = fmaxf(mb, s[t][r]);
    mb *= kSDown;
    // A query's running max follows only where one of its scores passes it by
    // more than kSlack (the weights keep that much room below f16's largest).
    if (__builtin_amdgcn_ballot_w64(mb > m_run + kSlack) != 0) {
      float other;
      mb = xor32_pair(mb, &other);
      mb = fmaxf(mb, other);
      const bool moves = mb > m_run + kSlack;
      const float m_new = moves ? mb : m_run;
      const float alpha = moves ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.0f;  // 0 at first
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          o[dt][r] *= alpha;
          total[dt][r] *= alpha;
        }
      l_run *= alpha;
      m_run = m_new;
    }
    const float c = kPBits - m_run;
    float ps = 0.0f;  // this block's weights (one addition to l_run a block)
    const char* vf = vfrag + buf * kBufBytes;
#pragma unroll
    for (int ch = 0; ch < 4; ++ch) {
      const int t = ch >> 1, r0 = 8 * (ch & 1);
      u32x4 vv[2][2];
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int p = 0; p < 2; ++p)
          vv[dt][p] = *reinterpret_cast<const u32x4*>(vf + 32 * dt * kRowBytes + 128 * p + 32 * ch);
      u32x4 p0, p1;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float a = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][r0 + 2 * j], kSDown, c));
        const float b = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][r0 + 2 * j + 1], kSDown, c));
        ps += a;
        ps += b;
        uint32_t x, y;
        vks::split2_plain(a, b, &x, &y);
        p0[j] = x;
        p1[j] = y;
      }
#pragma unroll
      for (int dt = 0; dt < 2; ++dt) o[dt] = vks::mfma32(vv[dt][1], p0, o[dt]);
#pragma unroll
      for (int dt = 0; dt < 2; ++dt) o[dt] = vks::mfma32(vv[dt][0], p1, o[dt]);
#pragma unroll
      for (int dt = 0; dt < 2; ++dt) o[dt] = vks::mfma32(vv[dt][0], p0, o[dt]);
    }
    l_run += ps;
  };

  auto flush = [&]() {
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        total[dt][r] += o[dt][r];
        o[dt][r] = 0.0f;
      }
  };
  store_block(0);
  __syncthreads();
  for (int kb = kb_begin; kb < kb_end; ++kb) {
    const int buf = (kb - kb_begin) & 1;
    const bool more = kb + 1 < kb_end;
    if (more) load_block(kb + 1);
    __builtin_amdgcn_sched_barrier(0);
    // a wave whose queries are all to be taken again only stages
    if (live && __builtin_amdgcn_ballot_w64(vks::is_finite(l_run)) != 0) {
      if ((kb - kb_begin) % kFlush == kFlush - 1) flush();
      compute(kb, buf);
    }
    if (more) store_block(buf ^ 1);
    __syncthreads();
  }

  flush();

  // Which queries did the split hold?  Any value of Q, K or V beyond f16, an
  // infinity or a NaN makes the sums that it enters NaN or infinite; sums that
  // are all small beside V's columns may show the floors (kHeldSum, kHeldSquare).
  const int qi = q0 + c32;
  const bool mine = live && qi < n;
  {
    float other;
    const float l = xor32_pair(l_run, &other);
    l_run = l + other;
  }
  bool odd = !vks::is_finite(l_run);
  float most = 0.0f;
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      odd |= !vks::is_finite(total[dt][r]);
      most = fmaxf(most, fabsf(total[dt][r]));
    }
  {
    float other;
    const float m = xor32_pair(most, &other);
    most = fmaxf(m, other);
  }
  const bool small = !(most >= kHeldSum && most * most >= kHeldSquare * l_run);
  auto queries = [&](bool x) {  // one bit per query of the wave, from either half
    const uint64_t b = __builtin_amdgcn_ballot_w64(mine && x);
    return static_cast<uint32_t>(b) | static_cast<uint32_t>(b >> 32);
  };
  const uint32_t odd_q = queries(odd), small_q = queries(small);
  // With every column at the largest scale, V of the run is zeros or has no floor
  // (2^-25 is then 2^-151 of a value).
  const bool some =
      __builtin_amdgcn_ballot_w64(vdown[lane] != __uint_as_float(1u << 23)) != 0;
  if (lane == 0) flags[wave] = odd_q | (some ? small_q : 0u);
  __syncthreads();
  
  uint32_t any = 0;
#pragma unroll
  for (int w = 0; w < QW; ++w) any |= flags[w];
  if (mine && ((flags[wave] >> c32) & 1) == 0) {
    const float* dn = vdown + 4 * half;
    if constexpr (PART) {
      // this split's O (rescaled to its own running max), max and sum
      const size_t rows = static_cast<size_t>(sequences) * n;
      const size_t row = static_cast<size_t>(split) * rows + static_cast<size_t>(seq) * n + qi;
      float* po = part + row * HD + 4 * half;
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const f32x4 d = *reinterpret_cast<const f32x4*>(dn + 32 * dt + 8 * r);
          const f32x4 t = {total[dt][4 * r], total[dt][4 * r + 1], total[dt][4 * r + 2],
                           total[dt][4 * r + 3]};
          *reinterpret_cast<f32x4*>(po + 32 * dt + 8 * r) = t * kPDown * d;
        }
      if (half == 0)
        *reinterpret_cast<float2*>(part + static_cast<size_t>(splits) * rows * HD + 2 * row) =
            make_float2(m_run, l_run * kPDown);
    } else {
      // out[query][d] = O / l; both carry the weights' scale, O also V's
      float* orow = out + base + static_cast<size_t>(qi) * HD + 4 * half;
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const f32x4 d = *reinterpret_cast<const f32x4*>(dn + 32 * dt + 8 * r);
          const f32x4 t = {total[dt][4 * r] / l_run, total[dt][4 * r + 1] / l_run,
                           total[dt][4 * r + 2] / l_run, total[dt][4 * r + 3] / l_run};
          *reinterpret_cast<f32x4*>(orow + 32 * dt + 8 * r) = t * d;
        }
    }
  }
  if (__builtin_expect(any != 0, 0)) {
    // 16 queries a wave and pass; the stores are those of the flagged ones
#pragma unroll 1
    for (int h = 0; h < 2; ++h) {
      const int first = 16 * QW * h;  // of the workgroup's queries
      uint32_t pass = 0;
      for (int w = first / 32; w < (first + 16 * QW) / 32; ++w) pass |= flags[w];
      if (pass == 0) continue;
      const uint32_t mask =
          (flags[(first + 16 * wave) / 32] >> (16 * (wave & 1))) & 0xffffu;
      __syncthreads();
      attention_tile_f32<PART, kThreads>(reinterpret_cast<float*>(smem), q, k, v, out, sequences,
                                         n, seq, qb + first, kb_begin, kb_end, split, splits, part,
                                         mask);
    }
  }
}

// Sequences of at most one key block: a workgroup per sequence with F32
// matrix instructions.  There is one short chain of loads, products and
// stores, and nothing for the split to save: 12 x 38 5.5 us, 192 x 60 6.2 (the
// kernel above: 6.1 and 6.8; from 65 rows on it is the faster, 8.1 to 11.7).
__global__ __launch_bounds__(256) void attention_short_kernel(const float* __restrict__ q,
                                                              const float* __restrict__ k,
                                                              const float* __restrict__ v,
                                                              float* __restrict__ out,
                                                              int sequences, int n) {
  __shared__ __align__(16) float smem[2 * KB * PITCH];
  attention_tile_f32<false, 256>(smem, q, k, v, out, sequences, n, blockIdx.x, 0, 0, 1, 0, 1,
                                 nullptr, 0xffffu);
}

// Combines the key splits of the PART form: 16 threads per query row, one
// float4 of O each; the splits' weights 2^(m_s - m) and sums are taken in
// split order.  SP (the split count) is a template parameter so that every
// load of a row is issued before the first is used: with a run-time count
// each loop iteration waited for its own loads.
template <int SP>
__global__ __launch_bounds__(256) void attention_merge_kernel(const float* __restrict__ part,
                                                              float* __restrict__ out,
                                                              long long rows) {
  const long long idx = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  const long long row = idx >> 4;
  const int c4 = static_cast<int>(idx & 15);
  if (row >= rows) return;
  const float* ml = part + static_cast<size_t>(SP) * rows * HD;
  float2 st[SP];
  f32x4 po[SP];
#pragma unroll
  for (int sp = 0; sp < SP; ++sp) {
    st[sp] = *reinterpret_cast<const float2*>(ml + 2 * (sp * rows + row));
    po[sp] = *reinterpret_cast<const f32x4*>(part + (sp * rows + row) * HD + 4 * c4);
  }
  float m = -INFINITY;
#pragma unroll
  for (int sp = 0; sp < SP; ++sp) m = fmaxf(m, st[sp].x);
  float l = 0.0f;
  f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int sp = 0; sp < SP; ++sp) {
    const float w = __builtin_amdgcn_exp2f(st[sp].x - m);
    l = l + st[sp].y * w;
    o = o + po[sp] * w;
  }
  *reinterpret_cast<f32x4*>(out + row * HD + 4 * c4) =
      f32x4{o[0] / l, o[1] / l, o[2] / l, o[3] / l};
}

int check_qkv(const vk_tensor* t, size_t len, const char* what) {
  VK_REQUIRE(t && t->dtype == VK_F32 && t->len == len, "attention: %s must be f32 [%zu] (holds %zu)",
             what, len, t ? t->len : 0);
  VK_REQUIRE(reinterpret_cast<uintptr_t>(t->ptr) % 16 == 0, "attention: %s must be 16-byte aligned",
             what);
  return VK_OK;
}

}  // namespace

extern "C" {

int vk_attention_into_f32(vk_runtime* rt, const vk_tensor* q, const vk_tensor* k,
                          const vk_tensor* v, size_t sequences, size_t n, size_t head_dim,
                          vk_tensor* out) {
  VK_TRY(vk::bind(rt));
  VK_REQUIRE(q && k && v && out, "null argument");
  VK_UNSUPPORTED_IF(head_dim != HD, "attention: head_dim=%zu (qualified: 64)", head_dim);
  VK_UNSUPPORTED_IF(n > 0x7fffffffULL || sequences > 0x7fffffffULL, "attention: too large");
  const size_t len = sequences * n * HD;
  VK_UNSUPPORTED_IF(len >= (size_t{1} << 30), "attention: tensors of 4 GiB or more");
  VK_TRY(check_qkv(q, len, "q"));
  VK_TRY(check_qkv(k, len, "k"));
  VK_TRY(check_qkv(v, len, "v"));
  VK_TRY(check_qkv(out, len, "out"));
  for (const vk_tensor* t : {q, k, v}) {
    const char* a = static_cast<const char*>(t->ptr);
    const char* b = static_cast<const char*>(out->ptr);
    VK_REQUIRE(len == 0 || a + len * 4 <= b || b + len * 4 <= a,
               "attention: out overlaps an input");
  }
  if (len == 0) return VK_OK;
  const int cus = rt->cu_count > 0 ? rt->cu_count : 256;
  const int nkb = static_cast<int>((n + KB - 1) / KB);
  const int provided = vk::attention_splits_to_provide(cus, sequences, n);
  const vk::AttentionPlan plan = vk::attention_plan(cus, sequences, n, provided);
  const int splits = plan.splits, qw = plan.waves;
  const long long tiles = static_cast<long long>(sequences) * ((n + 32 * qw - 1) / (32 * qw));
  const long long blocks = tiles * splits;
  VK_UNSUPPORTED_IF(blocks > 0x7fffffffLL, "attention: %lld workgroups", blocks);
  const auto* Q = static_cast<const float*>(q->ptr);
  const auto* K = static_cast<const float*>(k->ptr);
  const auto* V = static_cast<const float*>(v->ptr);
  auto* O = static_cast<float*>(out->ptr);
  const int S = static_cast<int>(sequences), N = static_cast<int>(n);
  if (provided > 1) {
    const size_t rows = sequences * n;
    const int most = provided > splits ? provided : splits;
    VK_TRY(vk::ensure_work(rt, static_cast<size_t>(most) * rows * (HD + 2), "attention"));
  }
  if (splits > 1) {
    const size_t rows = sequences * n;
    float* part = rt->work;
    if (qw == 8)
      hipLaunchKernelGGL((attention_kernel<true, 8>), dim3(static_cast<unsigned>(blocks)),
                         dim3(512), 0, rt->stream, Q, K, V, O, S, N, splits, part);
    else
      hipLaunchKernelGGL((attention_kernel<true, 4>), dim3(static_cast<unsigned>(blocks)),
                         dim3(256), 0, rt->stream, Q, K, V, O, S, N, splits, part);
    VK_TRY(vk::check_launch("attention_kernel"));
    const long long threads = static_cast<long long>(rows) * 16;
    const dim3 mgrid(static_cast<unsigned>((threads + 255) / 256));
    const long long R = static_cast<long long>(rows);
    switch (splits) {
#define VK_MERGE_CASE(SPN)                                                                     \
  case SPN:                                                                                    \
    hipLaunchKernelGGL(attention_merge_kernel<SPN>, mgrid, dim3(256), 0, rt->stream, part, O, R); \
    break;
      VK_MERGE_CASE(2) VK_MERGE_CASE(3) VK_MERGE_CASE(4) VK_MERGE_CASE(5)
      VK_MERGE_CASE(6) VK_MERGE_CASE(7) VK_MERGE_CASE(8)
#undef VK_MERGE_CASE
      default:
        return vk::set_error(VK_ERR_INVALID, "attention: %d key splits", splits);
    }
    return vk::check_launch("attention_merge_kernel");
  }
  if (nkb == 1)
    hipLaunchKernelGGL(attention_short_kernel, dim3(static_cast<unsigned>(sequences)), dim3(256), 0,
                       rt->stream, Q, K, V, O, S, N);
  else if (qw == 8)
    hipLaunchKernelGGL((attention_kernel<false, 8>), dim3(static_cast<unsigned>(blocks)), dim3(512),
                       0, rt->stream, Q, K, V, O, S, N, 1, nullptr);
  else
    hipLaunchKernelGGL((attention_kernel<false, 4>), dim3(static_cast<unsigned>(blocks)), dim3(256),
                       0, rt->stream, Q, K, V, O, S, N, 1, nullptr);
  return vk::check_launch("attention_kernel");
}

int vk_attention_online_f32(vk_runtime* rt, const vk_tensor* q, const vk_tensor* k,
                            const vk_tensor* v, size_t heads, size_t rows, size_t head_dim,
                            vk_tensor** out) {
  VK_TRY(vk::bind(rt));
  VK_REQUIRE(out, "null argument");
  VK_UNSUPPORTED_IF(head_dim != HD, "attention: head_dim=%zu (qualified: 64)", head_dim);
  vk_tensor* t = nullptr;
  VK_TRY(vk_tensor_alloc(rt, VK_F32, heads * rows * head_dim, &t));
  const int s = vk_attention_into_f32(rt, q, k, v, heads, rows, head_dim, t);
  if (s != VK_OK) {
    vk_tensor_destroy(t);
    return s;
  }
  *out = t;
  return VK_OK;
}

}  // extern "C"
