// The F32 linear on wide tiles for gfx950: the block projections (QKV, proj,
// FC1, FC2) with their per-token epilogues (bias, LayerScale, GELU,
// residual add) fused into the store.
//
// The products run on the f16 matrix cores as three products of two-part
// splits (split_f16.h), F32 in, F32 accumulate.
//
// A workgroup owns a TM x TN output tile (128 x 256 with eight waves, 128 x 128
// with four; 64 x 128 or 64 x 64 for grids of few rows); a wave computes all TM
// rows of 32 columns (64 x 64 tiles: 16) with v_mfma_f32_16x16x32_f16.
//
//  * A (activations, f32) is read by raw buffer loads one stage ahead, split
//    by the thread that loaded it and staged through LDS as [row][part][32 k]
//    f16 rows with a pitch of 144 bytes (16 x odd).  Two buffers: one barrier
//    a stage.
//  * B (weights) was split when the linear was prepared, each column scaled
//    by a power of two, into fragment order (split_weights): a wave's operand
//    of one 16-column tile and part is 1 KiB that its 64 lanes read in order,
//    straight into registers, one stage ahead.  The waves of a workgroup own
//    different columns, so no operand of B is read twice and B takes no LDS
//    space or bandwidth.
//
// A 128 x 128 tile runs 48 MFMAs a wave (768 cycles) per 32 k on 8 x 2
// fragment reads from LDS (4 waves: 512 cycles of its 128 bytes a clock)
// and 16 + 16 KiB from L2; two workgroups a CU cover each other's barriers.  A
// 128 x 256 tile splits and reads A once for twice the columns: 10,392 x 3072
// -> 768 in 129 us against 138 (380 TFLOP/s of the product's FLOP, 1,140 of f16
// MFMA; a large f16 library product reaches 1,243 on the card).  No single unit
// bounds it: at the 2.0 GHz its power allows the matrix pipe is busy 51% of the
// cycles (38% with GELU and 128 MB of output), waves wait 27-31% of theirs, and
// the split's VALU work lies between a stage's MFMAs and its barrier.  Bank
// conflicts of the staging stores do not show (a conflict-free plane layout
// measured the same), lines of A touched more often do (a lane per row instead
// of four: 10-20% slower).
// Grids of few tiles split K over several workgroups per tile (split-K:
// partial sums in the runtime's work buffer, added in split order by
// splitk_reduce_kernel).
//
// Head-major layouts (head_dim 64): the QKV projection can store Q | K | V
// straight into three [heads, rows, 64] tensors (the split the attention
// kernels need), and the output projection can read its input from the
// head-major attention output; tiles start on 64-column head boundaries,
// and 32 k of A never cross a head.  Both are pure address changes: the
// results are the bits of the linear plus the separate permutation.
//
// Q/K-norm + RoPE in the QKV epilogue (QKN != 0): after the last chunk the
// waves holding Q or K heads write their values (acc + b) to LDS, 64 rows at
// a time, and read them back as the Q/K kernel holds a row -- 16 lanes per
// 64-wide row, one float4 each -- and apply the same row transform
// (vkq::qk_row_transform) before storing the row head-major.  The values and
// the code path are those of the separate pass, so the bits are too.
//
// Every output is either the split's sum or, where the split may hold its
// terms less well than F32 does, an F32 one: the wave computes 64 rows of
// its columns again with F32 matrix instructions on the f32 operands and takes
// the outputs in question from there.  Which they are depends on the output's
// own row and column alone (and the split-K run), so no other row or column of
// a tile changes its bits:
//  * the sum is not finite;
//  * the floor of 2^-36 could show.  Rows of A are scaled by a power of two that
//    brings their typical value (of two stages) into [2^6, 2^7), columns of B to
//    [2^10, 2^11).  In groups of 8 k, with G groups in the run, a row counts the
//    groups found to reach 1 (big; three of the eight values are looked at) and
//    those with a value below 2^-13 (tiny), a column its groups of weights all of
//    at least 8 (dense) and its weights below 2^-13 that their parts do not hold
//    exactly (tiny).  Then
//      the floor's share of a sum   <= 2^-24 need,
//        need = min(4 tiny_row, 2^-12 sum |w|) + 16 tiny_col,
//      the sum of its |terms|  s    >= 8 (big + dense - G)  and  >= |sum|,
//    the former because at least big + dense - G groups hold a value of at least 1
//    whose weight is at least 8.  Taken again unless one of the two reaches
//    `need`: the floor then stays below 2^-24 s;
//  * a sum of few terms, which F32 adds with next to no rounding (a one-hot
//    column copies): fewer than a quarter of the run's groups, 8 at most, reach 1
//    in the row, or 8 in the column.
// Ordinary rows (layer-normalised, GELU outputs, attention outputs) and dense
// columns pass as a whole; then an output costs only the test that it is finite.
// The scale and the counts take 0.5 to 1.1 us of a launch of one image (866 x 768
// -> 2304 17.1 -> 18.0 us, projection 12.3 -> 12.8) and 2 to 4% of the large ones
// (10,392 x 768 -> 3072 154 -> 158).  Rows of any scale run at that speed (x 1e-6:
// 20.5 us a call; judged by one fixed scale and taken again tile by tile 69), and
// so do eight decades of sizes in every row at 866 rows (22.8).  A launch that
// takes every output again (NaN throughout) costs about 1.8 times one on F32 matrix
// instructions alone: 10,392 x 3072 -> 768 684 us against 375.
//
// Tiles are numbered XCD-major in groups of at most 1,024 rows (tile_of): the
// workgroups an XCD holds at one time then share both a slice of A and one
// of the weights in its L2.
#include "common.h"
#include "qk_rows.h"
#include "split_f16.h"

namespace {

using vk::LinearArgs;
using namespace vk::linear_epilogue;
using vks::f32x4;
using vks::u32x4;

constexpr int KC = vk::kSplitK;    // k of one stage (and of one MFMA)
// Waves of a tile: one per 32 columns, at least four.
constexpr int waves_for(int tn) { return tn == 256 ? 8 : 4; }
// Values below kTiny have the split's floor; groups of 8 k with a value of A of
// at least kXBig, or weights of at least kWBig, count as big or dense.
constexpr float kTiny = 1.0f / 8192.0f, kXBig = 1.0f, kWBig = 8.0f;
// A row's typical value is brought to [2^kRowBits, 2 x that), its largest one
// (of those looked at) below 2^(kRowMaxBits + 1).
constexpr int kRowBits = 6, kRowMaxBits = 9;
// Sums of fewer groups than this are F32 sums: a quarter of the run's, 2 to 8.
__device__ __forceinline__ int few_groups(int groups) {
  return groups >= 32 ? 8 : (groups >= 8 ? groups / 4 : 2);
}
constexpr int kMaxSplitK = 1 << 18;  // counts of 16 bits; longer sums are F32 sums
constexpr int kZeroColumn = 1 << 20;  // exponent of a column of zeros
constexpr int kZeroRowExp = 126;      // and of a row without a value in the sample
constexpr int kRowBytes = 144;     // LDS pitch of a row of A: 2 parts x 64 bytes + 16
constexpr int kXsPitch = 68;       // f32 pitch of the Q/K epilogue's rows
static_assert(kRowBytes % 16 == 0 && (kRowBytes / 16) % 2 == 1 && kRowBytes >= 4 * KC, "pitch");

enum Layout { kPlain = 0, kQkvHnd = 1, kAHnd = 2 };

// One output value: v = acc + b (then * ls), each step rounded, through the
// epilogue.
template <int EPI>
__device__ __forceinline__ float epi_value(const LinearArgs& g, float acc, float bias, float ls,
                                           float old) {
  float v = acc + bias;
  if (g.ls) v = v * ls;
  if (EPI == kLinGelu) return vkd::gelu1<0>(v);
  if (EPI == kLinGeluErf) return vkd::gelu1<1>(v);
  if (EPI == kLinResidual) return old + v;
  return v;
}

// Address of output element (row, col) in the output layout.
template <int LAY>
__device__ __forceinline__ float* out_addr(const LinearArgs& g, int row, int col) {
  if constexpr (LAY == kQkvHnd) {
    const int embed = g.N / 3;
    const int which = col >= embed ? (col >= 2 * embed ? 2 : 1) : 0;
    const int c = col - which * embed;
    float* base = which == 0 ? g.q_out : (which == 1 ? g.k_out : g.v_out);
    return base + (static_cast<size_t>(c >> 6) * g.M + row) * 64 + (c & 63);
  } else {
    return g.out + static_cast<size_t>(row) * g.N + col;
  }
}

template <int EPI, int LAY>
__device__ __forceinline__ void store_out(const LinearArgs& g, int row, int col, float acc,
                                          float bias, float ls, float old) {
  *out_addr<LAY>(g, row, col) = epi_value<EPI>(g, acc, bias, ls, old);
}

// QKN: 0 none; 1 / 2 Q/K LayerNorm (f32 / f16 parameters) + RoPE; 3 RoPE.
template <int QKN>
struct QknTraits;
template <>
struct QknTraits<1> {
  typedef float PT;
  static constexpr bool kNorm = true;
};
template <>
struct QknTraits<2> {
  typedef uint16_t PT;
  static constexpr bool kNorm = true;
};
template <>
struct QknTraits<3> {
  typedef float PT;
  static constexpr bool kNorm = false;
};

// Q/K-norm + RoPE of one 64-wide head row held as one float4 per lane of a
// 16-lane group (lane l: columns 4l..4l+3), for token `row` (clamped to a
// valid token; rows past M are computed and not stored).
template <int QKN>
__device__ __forceinline__ float4 qk_head_row(const LinearArgs& g, float4 v, int l, bool is_k,
                                              int row) {
  typedef typename QknTraits<QKN>::PT PT;
  const int rowc = row < g.M ? row : g.M - 1;
  float py, px;
  vkq::grid_position(vkd::fmod_(static_cast<uint32_t>(rowc), g.qkn.tpv), g.qkn.n_special,
                     g.qkn.global, g.qkn.gw, &py, &px);
  const PT* gm = static_cast<const PT*>(is_k ? g.qkn.kg : g.qkn.qg);
  const PT* bt = static_cast<const PT*>(is_k ? g.qkn.kb : g.qkn.qb);
  // the pairing is uniform over the launch: a scalar branch
  if (g.qkn.interleaved)
    return vkq::qk_row_transform<PT, QknTraits<QKN>::kNorm, vkq::kPosGrid, vkq::kInterleaved>(
        v, l, gm, bt, py, px, g.qkn.table, g.qkn.table_max, g.qkn.eps);
  return vkq::qk_row_transform<PT, QknTraits<QKN>::kNorm, vkq::kPosGrid, vkq::kRotateHalf>(
      v, l, gm, bt, py, px, g.qkn.table, g.qkn.table_max, g.qkn.eps);
}

// The sum passes are instantiated for split-count buckets SPB of 2, 4 and 8 (a
// plan takes at most kMaxSplits).
static_assert(vk::kMaxSplits <= 8, "split_bucket");
constexpr int split_bucket(int splits) { return splits <= 2 ? 2 : (splits <= 4 ? 4 : 8); }

// The NV float4 at offsets e[i] of every split's slice (splits <= SPB),
// summed in split order.  All SPB x NV loads are issued before the first
// addition (a run-time loop over the splits waited for each iteration's
// load); slots past `splits` re-read the last slice and are not added.
template <int NV, int SPB>
__device__ __forceinline__ void split_sums(const float* __restrict__ partial, size_t mn,
                                           const size_t (&e)[NV], int splits, f32x4 (&acc)[NV]) {
  f32x4 p[NV][SPB];
#pragma unroll
  for (int sp = 0; sp < SPB; ++sp) {
    const size_t slice = static_cast<size_t>(sp < splits ? sp : splits - 1) * mn;
#pragma unroll
    for (int i = 0; i < NV; ++i) p[i][sp] = *reinterpret_cast<const f32x4*>(partial + slice + e[i]);
  }
  // all loads issued before the first addition (the scheduler would
  // otherwise roll them behind the additions, one round trip each)
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    acc[i] = p[i][0];
#pragma unroll
    for (int sp = 1; sp < SPB; ++sp)
      if (sp < splits) acc[i] = acc[i] + p[i][sp];
  }
}

// The tile and split of workgroup `t`: groups of at most 1,024 rows, in a
// group split-major, then column tiles, then the group's row tiles (fastest).
template <int TM>
__device__ __forceinline__ void tile_of(int t, int gmt, int gnt, int splits, int* mt, int* nt,
                                        int* split) {
  constexpr int kGroup = 1024 / TM;
  const int per_group = kGroup * gnt * splits;
  const int grp = t / per_group, r = t - grp * per_group;
  const int left = gmt - grp * kGroup;
  const int rows = left < kGroup ? left : kGroup;
  *mt = grp * kGroup + r % rows;
  const int rest = r / rows;
  *nt = rest % gnt;
  *split = rest / gnt;
}

__device__ __forceinline__ float max_abs4(const float4& x) {
  return fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w)));
}

// Largest value and sum over the four lanes 4 i .. 4 i + 3 (a row's pieces).
__device__ __forceinline__ uint32_t quad_other(uint32_t v, int step) {
  const int x = static_cast<int>(v);  // quad_perm [1, 0, 3, 2] and [2, 3, 0, 1]
  return static_cast<uint32_t>(step == 1 ? __builtin_amdgcn_mov_dpp(x, 0xb1, 0xf, 0xf, true)
                                         : __builtin_amdgcn_mov_dpp(x, 0x4e, 0xf, 0xf, true));
}

__device__ __forceinline__ uint32_t quad_sum(uint32_t v) {
  v += quad_other(v, 1);
  return v + quad_other(v, 2);
}

__device__ __forceinline__ float quad_max(float v) {
  v = fmaxf(v, __uint_as_float(quad_other(__float_as_uint(v), 1)));
  return fmaxf(v, __uint_as_float(quad_other(__float_as_uint(v), 2)));
}

// NP: f16 parts of a weight.  Weights that are f16 values have one (the other
// is all zeros, so the sums are the same): two products, half of B's bytes.
//
// KS: stages of 32 k per barrier (2 for the 64-row tiles, whose 12 or 24
// MFMAs a wave and stage are too few to cover a load's latency).
// What a column's weights are in stages [c_begin, c_end): groups of 8 k all of
// at least kWBig, groups that reach it, weights with a floor (split_weights), from
// the running counts `a` before c_begin and `b` before c_end.
struct ColumnRun {
  int dense, any, tiny;
};

__device__ __forceinline__ ColumnRun column_run(const uint2& a, const uint2& b) {
  return ColumnRun{static_cast<int>((b.x - a.x) & 0xffffu),
                   static_cast<int>((b.x >> 16) - (a.x >> 16)) & 0xffff,
                   static_cast<int>(b.y - a.y)};
}

template <int EPI, int LAY, int QKN, int TM, int TN, int KS, int NP>
__global__ __launch_bounds__(64 * waves_for(TN), 2) void linear_wide_kernel(LinearArgs g) {
  constexpr int kWaves = waves_for(TN), kThreads = 64 * kWaves;
  static_assert(TM == 128 || TM == 64, "tile heights 128 and 64");
  static_assert(TN == 256 || TN == 128 || TN == 64, "tile widths 256, 128 and 64");
  constexpr int WN = TN / kWaves;       // columns of a wave
  constexpr int MT = TM / 16;           // 16-row MFMA tiles of a wave
  constexpr int NU = WN / 16;           // 16-column MFMA tiles of a wave
  constexpr int kSlots = TM * 4 * KS;   // 8-k pieces of A a barrier
  constexpr int kVA = kSlots / kThreads;
  static_assert(kVA * kThreads == kSlots, "slots divide evenly");
  constexpr int kStageBytes = TM * kRowBytes;
  constexpr int kBufBytes = KS * kStageBytes;
  constexpr int kXsBytes = QKN != 0 ? (TN / 64) * 64 * kXsPitch * 4 : 0;
  constexpr int kSmem = 2 * kBufBytes > kXsBytes ? 2 * kBufBytes : kXsBytes;
  __shared__ __align__(16) char smem[kSmem];

  // The arguments lie in host memory: a first read of one of their cache lines
  // takes about 2 us, so all lines are read at once here and not one after the
  // other where the code below first needs them.
  asm volatile("" ::"s"(g.x), "s"(g.M), "s"(g.qkn_mode), "s"(g.qkn.eps), "s"(g.ln_out),
               "s"(gridDim.x));

  const int tid = threadIdx.x;
  __builtin_assume(tid < kThreads);
  const int wave = tid >> 6, lane = tid & 63;
  const int gmt = (g.M + TM - 1) / TM;
  const int gnt = (g.N + TN - 1) / TN;
  int mt, nt, split;
  tile_of<TM>(vkd::xcd_tile(blockIdx.x, gridDim.x), gmt, gnt, g.splits, &mt, &nt, &split);
  const int m0 = mt * TM, n0 = nt * TN;
  const int nch = (g.K + KC - 1) / KC;
  // split <= 8 and nch < 2^26: 32 bits hold the products
  const int c_begin = static_cast<int>(static_cast<uint32_t>(split) * nch / g.splits);
  const int c_end = static_cast<int>(static_cast<uint32_t>(split + 1) * nch / g.splits);

  // A: slot i of a thread is piece s = tid + 256 i: stage s / (4 TM), row
  // (s / 4) % TM, k 8 (s % 4) .. + 8 of that stage.  Rows past M read a
  // clamped, valid row, which only reaches output rows past M.
  const int piece = tid & 3;
  auto slot_row = [&](int i) { return ((tid + kThreads * i) >> 2) % TM; };
  auto slot_stage = [&](int i) { return (kThreads * i) / (4 * TM); };
  uint32_t a_off[kVA];
#pragma unroll
  for (int i = 0; i < kVA; ++i) {
    const int gm = m0 + slot_row(i);
    const uint32_t cm = static_cast<uint32_t>(gm < g.M ? gm : g.M - 1);
    a_off[i] = 4u * (cm * (LAY == kAHnd ? 64u : static_cast<uint32_t>(g.K)) + 8u * piece);
  }
  const uint32_t a_bytes = 4u * static_cast<uint32_t>(g.M) * static_cast<uint32_t>(g.K);
  const __amdgpu_buffer_rsrc_t a_rsrc = vkd::buffer_rsrc(g.x, a_bytes);
  // byte offset of stage ch for every row
  auto a_chunk = [&](int ch) {
    return LAY == kAHnd ? 4u * (static_cast<uint32_t>(ch >> 1) * static_cast<uint32_t>(g.M) * 64u +
                                static_cast<uint32_t>(ch & 1) * 32u)
                        : 4u * static_cast<uint32_t>(ch) * KC;
  };
  float4 ra[kVA][2];
  // k past K, and stages past the split's end, read past the buffer, which
  // gives zeros.
  auto load_a = [&](int ch0, float4 (&ra)[kVA][2]) {
#pragma unroll
    for (int i = 0; i < kVA; ++i) {
      const int at = ch0 + slot_stage(i);
      const int ch = at < c_end ? at : c_end - 1;
      const int left = at < c_end ? g.K - ch * KC : 0;  // uniform
      const uint32_t base = a_chunk(ch);
#pragma unroll
      for (int h = 0; h < 2; ++h)
        ra[i][h] = vkd::buffer_load4(
            a_rsrc, 8 * piece + 4 * h < left ? a_off[i] + 16u * h : 0xfffffff0u, base);
    }
  };
  // Per row of the thread's slots: its scale and the groups counted.
  constexpr int kVR = kVA / KS;
  float rscale[kVR];
  uint32_t rbig[kVR], rtiny[kVR];
  auto store_a = [&](int buf) {
#pragma unroll
    for (int i = 0; i < kVA; ++i) {
      const int rr = i % kVR;
      const float4 x = vks::scale4(ra[i][0], rscale[rr]), y = vks::scale4(ra[i][1], rscale[rr]);
      rbig[rr] += fmaxf(fmaxf(fabsf(x.x), fabsf(x.w)), fabsf(y.z)) >= kXBig;  // three of eight
      rtiny[rr] += vks::min_abs8(x, y) < kTiny;
      u32x4 p0, p1;
      vks::split8(x, y, &p0, &p1);
      char* d = smem + buf * kBufBytes + slot_stage(i) * kStageBytes + slot_row(i) * kRowBytes +
                16 * piece;
      *reinterpret_cast<u32x4*>(d) = p0;
      *reinterpret_cast<u32x4*>(d + 64) = p1;
    }
  };

  // B: 16-column tile j of the weights, stage ch, part p: 64 x 16 bytes at
  // ((j nch + ch) NP + p) KiB.  Tiles past N read the last one; their columns
  // are not stored.
  const int ntiles = (g.N + 15) / 16;
  const u32x4* bptr[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int j = (n0 + wave * WN) / 16 + u;
    const int cj = j < ntiles ? j : ntiles - 1;
    bptr[u] = reinterpret_cast<const u32x4*>(g.wsplit) +
              static_cast<size_t>(cj) * nch * (NP * 64) + lane;
  }
  auto load_b = [&](int ch0, u32x4 (&b)[KS][NU][NP]) {
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      // a stage past the split's end multiplies zeros of A
      const int ch = ch0 + s < c_end ? ch0 + s : c_end - 1;
#pragma unroll
      for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int p = 0; p < NP; ++p)
          b[s][u][p] = bptr[u][static_cast<size_t>(ch) * (NP * 64) + p * 64];
    }
  };
  const char* afrag = smem + (lane & 15) * kRowBytes + 16 * (lane >> 4);
  f32x4 acc[MT][NU], corr[MT][NU];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int u = 0; u < NU; ++u) acc[t][u] = corr[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Fragments of the next 16 rows are read while these rows' MFMAs run.
  auto mma = [&](int buf, const u32x4 (&b)[KS][NU][NP]) {
    u32x4 a[2][2];
    auto read_a = [&](int st, u32x4 (&f)[2]) {
      const char* ar = afrag + buf * kBufBytes + (st / MT) * kStageBytes +
                       (st % MT) * 16 * kRowBytes;
      f[0] = *reinterpret_cast<const u32x4*>(ar);
      f[1] = *reinterpret_cast<const u32x4*>(ar + 64);
    };
    read_a(0, a[0]);
#pragma unroll
    for (int st = 0; st < KS * MT; ++st) {
      const int s = st / MT, t = st % MT;
      if (st + 1 < KS * MT) read_a(st + 1, a[(st + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      const u32x4(&f)[2] = a[st & 1];
#pragma unroll
      for (int u = 0; u < NU; ++u) acc[t][u] = vks::mfma(f[0], b[s][u][0], acc[t][u]);
      if constexpr (NP == 2) {
#pragma unroll
        for (int u = 0; u < NU; ++u) corr[t][u] = vks::mfma(f[0], b[s][u][NP - 1], corr[t][u]);
      }
#pragma unroll
      for (int u = 0; u < NU; ++u) corr[t][u] = vks::mfma(f[1], b[s][u][0], corr[t][u]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // One stage: run its MFMAs, split and store the next one and issue the loads
  // of the one after.  A buffer is written again in the stage after the one
  // that read it, with a barrier in between.
  u32x4 b0[KS][NU][NP], b1[KS][NU][NP];
  const bool split_k = g.K < kMaxSplitK;  // else F32 throughout
  const int k_end = c_end * KC < g.K ? c_end * KC : g.K;
  const int groups = (k_end - c_begin * KC + 7) / 8, few = few_groups(groups);
  auto col_of = [&](int u) { return n0 + wave * WN + u * 16 + (lane & 15); };
  int cexp[NU];
  float cfloor[NU];
  uint2 cr0[NU], cr1[NU];  // read here, and looked at after the loop
  int ch = split_k ? c_begin : c_end;
  if (split_k) {
    load_a(c_begin, ra);
    float4 rm[kVR];  // of the run's middle, for the scale
    const int mid = (c_begin + c_end) >> 1;
#pragma unroll
    for (int i = 0; i < kVR; ++i)
      rm[i] = vkd::buffer_load4(a_rsrc, 8 * piece < g.K - mid * KC ? a_off[i] : 0xfffffff0u,
                                a_chunk(mid));
    load_b(c_begin, b0);
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int col = col_of(u) < g.N ? col_of(u) : g.N - 1;
      const int2 c = g.wcol[col];
      cexp[u] = c.x;
      cfloor[u] = __int_as_float(c.y);
      cr0[u] = g.wstat[static_cast<size_t>(c_begin) * g.N + col];
      cr1[u] = g.wstat[static_cast<size_t>(c_end) * g.N + col];
    }
    // every load issued before the first is waited for
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kVR; ++i) {
      // the pieces of the first stage and half of those of the middle one; the
      // typical size is the lesser of the two, of the row's best piece
      const float first = vks::max_abs8(ra[i][0], ra[i][1]), middle = max_abs4(rm[i]);
      const float m = quad_max(fmaxf(first, middle)), t = quad_max(fminf(first, middle));
      // values in [2^(b - 127), 2^(b - 126)).  No value seen: the largest scale, by
      // which any value met later is beyond f16, or has no floor (a row of zeros
      // is held).
      const int bm = static_cast<int>(__float_as_uint(m) >> 23);
      const int bt = t > 0.0f ? static_cast<int>(__float_as_uint(t) >> 23) : bm;
      int e = kRowBits + 127 - bt;
      e = e < kRowMaxBits + 127 - bm ? e : kRowMaxBits + 127 - bm;
      e = bm == 255 ? 0 : (m == 0.0f || e > 126 ? 126 : e);
      rscale[i] = __uint_as_float(static_cast<uint32_t>(127 + e) << 23);
      rbig[i] = rtiny[i] = 0;
    }
    store_a(0);
    load_a(ch + KS, ra);
  }
  for (; ch + KS < c_end; ch += 2 * KS) {
    __syncthreads();
    load_b(ch + KS, b1);
    mma(0, b0);
    store_a(1);
    load_a(ch + 2 * KS, ra);
    __syncthreads();
    load_b(ch + 2 * KS, b0);
    mma(1, b1);
    if (ch + 2 * KS < c_end) store_a(0);
    load_a(ch + 3 * KS, ra);
  }
  if (ch < c_end) {
    __syncthreads();
    mma(0, b0);
  }

  // lane holds D[4 (lane / 16) + r][lane % 16] of each 16 x 16 tile
  const int g4 = lane >> 4, c16 = lane & 15;
  auto row_of = [&](int t, int r) { return m0 + t * 16 + 4 * g4 + r; };

  // The sums.  Rows' counts and exponents meet in LDS.
  int* row_exp = reinterpret_cast<int*>(smem);
  int* row_cnt = row_exp + TM;
  int* flags = row_cnt + TM;  // one per wave: a row that is not plain
  bool look = !split_k;
  ColumnRun cr[NU];
  if (split_k) {
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      cr[u] = column_run(cr0[u], cr1[u]);
      look |= (cexp[u] != kZeroColumn) &
              ((cr[u].any < few) |
               (8 * (cr[u].dense - groups) - 16 * cr[u].tiny < -6 * groups));
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          acc[t][u][r] = __builtin_fmaf(corr[t][u][r], vks::kDown, acc[t][u][r]);
          look |= !vks::is_finite(acc[t][u][r]);
        }
    __syncthreads();  // every wave is done with the last stage
    bool plain_rows = true;
#pragma unroll
    for (int i = 0; i < kVR; ++i) {
      // pieces past the run's end were zeros and counted
      const int past = 4 * KS * ((c_end - c_begin + KS - 1) / KS) - groups;
      const int tiny = static_cast<int>(quad_sum(rtiny[i])) - past;
      const int big = static_cast<int>(quad_sum(rbig[i]));
      const int e = static_cast<int>(__float_as_uint(rscale[i]) >> 23) - 127;
      plain_rows &= e == kZeroRowExp || (big >= few && 8 * big - 4 * tiny >= 6 * groups);
      if (piece == 0) {
        row_exp[slot_row(i)] = e;
        row_cnt[slot_row(i)] = tiny << 16 | big;
      }
    }
    const bool rows_look = __builtin_amdgcn_ballot_w64(!plain_rows) != 0;
    if (lane == 0) flags[wave] = rows_look;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kWaves; ++w) look |= flags[w] != 0;
  }
  // exponents of rows 16 t + 4 g4 .. + 4
  auto row4 = [&](const int* p, int t) {
    return *reinterpret_cast<const int4*>(p + t * 16 + 4 * g4);
  };
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(look) == 0, 1)) {
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int4 e4 = row4(row_exp, t);
      const int e[4] = {e4.x, e4.y, e4.z, e4.w};
#pragma unroll
      for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          acc[t][u][r] = __builtin_amdgcn_ldexpf(acc[t][u][r], -e[r] - cexp[u]);
    }
  } else {
    // Output by output; 64 rows with any to take again are computed in F32
    // (fragment order: lane group g4 holds k = 16 b + 4 g4 + j of block b in
    // component j), straight from memory and without a barrier.
    const float* wrow[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int col = col_of(u) < g.N ? col_of(u) : g.N - 1;
      wrow[u] = g.wnk + static_cast<size_t>(col) * g.Kp;
    }
#pragma unroll
    for (int t0 = 0; t0 < MT; t0 += 4) {
      uint32_t again[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        again[i] = 0xffffffffu;
        if (!split_k) continue;
        const int t = t0 + i;
        const int4 e4 = row4(row_exp, t), c4 = row4(row_cnt, t);
        const int e[4] = {e4.x, e4.y, e4.z, e4.w}, c[4] = {c4.x, c4.y, c4.z, c4.w};
        again[i] = 0;
#pragma unroll
        for (int u = 0; u < NU; ++u)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float v = acc[t][u][r];
            const int big = c[r] & 0xffff, tiny = (c[r] >> 16) & 0xffff;
            const float need = fminf(static_cast<float>(4 * tiny), cfloor[u]) +
                               static_cast<float>(16 * cr[u].tiny);
            const bool held =
                e[r] == kZeroRowExp || cexp[u] == kZeroColumn ||
                (big >= few && cr[u].any >= few &&
                 fmaxf(static_cast<float>(8 * (big + cr[u].dense - groups)), fabsf(v)) >= need);
            if (!held || !vks::is_finite(v)) again[i] |= 1u << (4 * u + r);
            acc[t][u][r] = __builtin_amdgcn_ldexpf(v, -e[r] - cexp[u]);
          }
      }
      if (__builtin_amdgcn_ballot_w64((again[0] | again[1] | again[2] | again[3]) != 0) == 0)
        continue;
      const float* arow[4];  // the fragments' rows
      f32x4 f[4][NU];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = m0 + (t0 + i) * 16 + c16;
        arow[i] = g.x + static_cast<size_t>(row < g.M ? row : g.M - 1) * (LAY == kAHnd ? 64 : g.K);
#pragma unroll
        for (int u = 0; u < NU; ++u) f[i][u] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      // 16 k ahead in registers; k past K multiplies zeros
      f32x4 a[4], w[NU];
      auto fetch = [&](int b) {
        const int k = 16 * b + 4 * g4;
        const int ck = k < g.K ? k : 0;
        const size_t at = LAY == kAHnd ? static_cast<size_t>(ck >> 6) * g.M * 64 + (ck & 63)
                                       : static_cast<size_t>(ck);
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = *reinterpret_cast<const f32x4*>(arow[i] + at);
#pragma unroll
        for (int u = 0; u < NU; ++u) {
          w[u] = *reinterpret_cast<const f32x4*>(wrow[u] + ck);
#pragma unroll
          for (int j = 0; j < 4; ++j) w[u][j] = k < g.K ? w[u][j] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) a[i][j] = k < g.K ? a[i][j] : 0.0f;
      };
      const int b_end = 2 * c_end < (g.K + 15) / 16 ? 2 * c_end : (g.K + 15) / 16;
      fetch(2 * c_begin);
#pragma unroll 1
      for (int b = 2 * c_begin; b < b_end; ++b) {
        f32x4 ca[4], cw[NU];
#pragma unroll
        for (int i = 0; i < 4; ++i) ca[i] = a[i];
#pragma unroll
        for (int u = 0; u < NU; ++u) cw[u] = w[u];
        fetch(b + 1 < b_end ? b + 1 : b);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int u = 0; u < NU; ++u)
              f[i][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(ca[i][j], cw[u][j], f[i][u], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int u = 0; u < NU; ++u)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if ((again[i] >> (4 * u + r)) & 1) acc[t0 + i][u][r] = f[i][u][r];
    }
  }

  // split-K: raw sums to this split's slice of the partial buffer
  if (g.splits > 1) {
    float* part = g.partial + static_cast<size_t>(split) * g.M * g.N;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int u = 0; u < NU; ++u) {
          const int row = row_of(t, r), col = col_of(u);
          if (row < g.M && col < g.N) part[static_cast<size_t>(row) * g.N + col] = acc[t][u][r];
        }
    return;
  }

  // epilogue.  Parameters and (for the residual) the old values are all
  // loaded, on clamped indices, before the first store.
  if constexpr (QKN != 0) {
    static_assert(LAY == kQkvHnd && EPI == kLinStore, "Q/K epilogue of the QKV projection");
    // A head of Q, K or V is two waves' columns, or all four's of a 64-wide
    // tile; its 64-row halves meet in LDS one after the other.
    constexpr int kHeadWaves = 64 / WN;               // 2 or 4
    constexpr int kRowsPerGroup = 16 / kHeadWaves;    // rows of a 16-lane group a half
    const int head = wave / kHeadWaves, hw = wave % kHeadWaves;
    const int col0 = n0 + head * 64;
    const int embed = g.N / 3;
    const int which = col0 < g.N ? col0 / embed : 2;
    float* xs = reinterpret_cast<float*>(smem) + head * 64 * kXsPitch;
    float* dst = nullptr;
    if (which < 2)
      dst = (which == 0 ? g.q_out : g.k_out) +
            static_cast<size_t>((col0 - which * embed) >> 6) * g.M * 64;
#pragma unroll
    for (int half = 0; half < TM / 64; ++half) {
      __syncthreads();  // every wave is done with what LDS held
      if (which < 2) {
#pragma unroll
        for (int u = 0; u < NU; ++u) {
          const float b = g.bias[col_of(u)];
#pragma unroll
          for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              xs[(t * 16 + 4 * g4 + r) * kXsPitch + hw * WN + u * 16 + c16] =
                  acc[half * 4 + t][u][r] + b;
        }
      }
      __syncthreads();
      if (which < 2) {
#pragma unroll 2
        for (int i = 0; i < kRowsPerGroup; ++i) {
          const int rr = (hw * 4 + g4) * kRowsPerGroup + i;
          const int row = m0 + half * 64 + rr;
          const float4 v = *reinterpret_cast<const float4*>(xs + rr * kXsPitch + 4 * c16);
          const float4 o = qk_head_row<QKN>(g, v, c16, which == 1, row);
          if (row < g.M)
            *reinterpret_cast<float4*>(dst + static_cast<size_t>(row) * 64 + 4 * c16) = o;
        }
      }
    }
    if (which < 2) return;
  }
  // Per 16-column strip u: bias, LayerScale and the address of the column
  // at row 0 (row r adds r x the row stride), computed once; a tile inside
  // the matrix stores without bounds checks.
  const bool interior = m0 + TM <= g.M && n0 + TN <= g.N;
  const size_t rs = LAY == kQkvHnd ? 64 : static_cast<size_t>(g.N);
  float bias[NU], ls[NU];
  float* cptr[NU];
  bool cok[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int col = col_of(u);
    cok[u] = col < g.N;
    const int cc = cok[u] ? col : g.N - 1;
    bias[u] = g.bias[cc];
    ls[u] = g.ls ? g.ls[cc] : 1.0f;
    cptr[u] = out_addr<LAY>(g, 0, cc);
  }
  float old[MT][NU][4];
  if constexpr (EPI == kLinResidual) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = row_of(t, r);
        const size_t cr = static_cast<size_t>(row < g.M ? row : g.M - 1);
#pragma unroll
        for (int u = 0; u < NU; ++u) old[t][u][r] = cptr[u][cr * rs];
      }
  }
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = row_of(t, r);
      const bool rok = row < g.M;
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const float val = epi_value<EPI>(g, acc[t][u][r], bias[u], ls[u],
                                         EPI == kLinResidual ? old[t][u][r] : 0.0f);
        if (interior || (rok && cok[u])) cptr[u][static_cast<size_t>(row) * rs] = val;
      }
    }
}

// Second pass of a split-K linear: one thread per 4 consecutive outputs of a
// row; the splits' partial sums are added in split order, then the epilogue
// of the single-pass kernel is applied.
template <int EPI, int LAY, int QKN, int SPB>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(LinearArgs g) {
  const long long i4 = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  const long long mn = static_cast<long long>(g.M) * g.N;
  if (i4 * 4 >= mn) return;  // whole 16-lane groups (M*N/4 is a multiple of 16 here)
  const size_t e = static_cast<size_t>(i4) * 4;
  const int row = static_cast<int>(e / g.N), col = static_cast<int>(e % g.N);
  const size_t es[1] = {e};
  // the epilogue's loads before the partial sums' and every store: a load
  // after a store to `out` would wait for it (the compiler cannot tell them
  // apart)
  const float4 bias = *reinterpret_cast<const float4*>(g.bias + col);
  const float4 ls = g.ls ? *reinterpret_cast<const float4*>(g.ls + col)
                         : make_float4(1.0f, 1.0f, 1.0f, 1.0f);
  f32x4 old = f32x4{0.f, 0.f, 0.f, 0.f};
  if constexpr (EPI == kLinResidual) old = *reinterpret_cast<const f32x4*>(g.out + e);
  f32x4 accs[1];
  split_sums<1, SPB>(g.partial, static_cast<size_t>(mn), es, g.splits, accs);
  const f32x4 acc = accs[0];
  if constexpr (QKN != 0) {
    // 16 consecutive threads hold one 64-wide head row of one token
    const int embed = g.N / 3;
    const int which = col / embed;
    if (which < 2) {
      const int c = col - which * embed;
      float4 v;
      v.x = acc[0] + bias.x;
      v.y = acc[1] + bias.y;
      v.z = acc[2] + bias.z;
      v.w = acc[3] + bias.w;
      const float4 o = qk_head_row<QKN>(g, v, threadIdx.x & 15, which == 1, row);
      float* dst = (which == 0 ? g.q_out : g.k_out) +
                   (static_cast<size_t>(c >> 6) * g.M + row) * 64 + (c & 63);
      *reinterpret_cast<float4*>(dst) = o;
      return;
    }
  }
  const float bj[4] = {bias.x, bias.y, bias.z, bias.w};
  const float lj[4] = {ls.x, ls.y, ls.z, ls.w};
#pragma unroll
  for (int j = 0; j < 4; ++j) store_out<EPI, LAY>(g, row, col + j, acc[j], bj[j], lj[j], old[j]);
}

// Sum pass of a split-K linear with the residual epilogue, followed by the
// LayerNorm of the finished rows: one wave per row, NV float4 per lane
// (column float4 lane + 64 i).  The partial sums are added in split order
// and the epilogue applied as in splitk_reduce_kernel, the row statistics
// and the normalisation are vkd::row_mean_inv / vkd::ln_apply4 over the same
// lane layout as layernorm_rows: the bits of the two separate passes.
template <int NV, typename PT, int SPB>
__global__ __launch_bounds__(64) void splitk_residual_ln_kernel(LinearArgs g) {
  const int lane = threadIdx.x;
  const size_t row = blockIdx.x;
  const size_t mn = static_cast<size_t>(g.M) * g.N;
  const size_t rb = row * g.N;
  size_t es[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) es[i] = rb + 4 * static_cast<size_t>(lane + 64 * i);
  // Every load of the row -- the residual, bias, LayerScale and LayerNorm
  // parameters, then the partial sums -- is issued before the first store:
  // the compiler cannot tell the stores to `out` from the parameter
  // pointers, so a load placed after a store would wait for it (one memory
  // round trip per float4 column of the lane).
  const PT* gm = static_cast<const PT*>(g.ln_gamma);
  const PT* bt = static_cast<const PT*>(g.ln_beta);
  f32x4 old[NV];
  float4 bias[NV], lsv[NV], lg[NV], lb[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c4 = lane + 64 * i;
    old[i] = *reinterpret_cast<const f32x4*>(g.out + es[i]);
    bias[i] = *reinterpret_cast<const float4*>(g.bias + 4 * c4);
    lsv[i] = g.ls ? *reinterpret_cast<const float4*>(g.ls + 4 * c4)
                  : make_float4(1.0f, 1.0f, 1.0f, 1.0f);
    lg[i] = vkd::Param<PT>::load4(gm, c4);
    lb[i] = vkd::Param<PT>::load4(bt, c4);
  }
  f32x4 accs[NV];
  split_sums<NV, SPB>(g.partial, mn, es, g.splits, accs);
  float4 vv[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const f32x4 acc = accs[i];
    float4 v;
    v.x = epi_value<kLinResidual>(g, acc[0], bias[i].x, lsv[i].x, old[i][0]);
    v.y = epi_value<kLinResidual>(g, acc[1], bias[i].y, lsv[i].y, old[i][1]);
    v.z = epi_value<kLinResidual>(g, acc[2], bias[i].z, lsv[i].z, old[i][2]);
    v.w = epi_value<kLinResidual>(g, acc[3], bias[i].w, lsv[i].w, old[i][3]);
    *reinterpret_cast<float4*>(g.out + es[i]) = v;
    vv[i] = v;
  }
  float mean, inv;
  vkd::row_mean_inv<NV, true>(vv, lane, g.N, g.ln_eps, &mean, &inv);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c4 = lane + 64 * i;
    *reinterpret_cast<float4*>(g.ln_out + rb + 4 * static_cast<size_t>(c4)) =
        vkd::ln_apply4(vv[i], mean, inv, lg[i], lb[i]);
  }
}

}  // namespace

namespace vk {

namespace {

template <int EPI, int LAY, int QKN, int NP>
void launch_tiles(vk_runtime* rt, const LinearArgs& g, const LinearPlan& plan, dim3 grid) {
  if (plan.tn == 256)
    hipLaunchKernelGGL((linear_wide_kernel<EPI, LAY, QKN, 128, 256, 1, NP>), grid, dim3(512), 0,
                       rt->stream, g);
  else if (plan.tm == 128)
    hipLaunchKernelGGL((linear_wide_kernel<EPI, LAY, QKN, 128, 128, 1, NP>), grid, dim3(256), 0,
                       rt->stream, g);
  else if (plan.tn == 128)
    hipLaunchKernelGGL((linear_wide_kernel<EPI, LAY, QKN, 64, 128, 2, NP>), grid, dim3(256), 0,
                       rt->stream, g);
  else
    hipLaunchKernelGGL((linear_wide_kernel<EPI, LAY, QKN, 64, 64, 2, NP>), grid, dim3(256), 0,
                       rt->stream, g);
}

template <int EPI, int LAY, int QKN = 0>
void launch_pair(vk_runtime* rt, const LinearArgs& g, const LinearPlan& plan, dim3 grid,
                 bool sum_pass = true) {
  if (g.wparts == 1)
    launch_tiles<EPI, LAY, QKN, 1>(rt, g, plan, grid);
  else
    launch_tiles<EPI, LAY, QKN, 2>(rt, g, plan, grid);
  if (g.splits > 1 && sum_pass) {
    const long long n4 = static_cast<long long>(g.M) * g.N / 4;
    const dim3 sgrid(static_cast<unsigned>((n4 + 255) / 256));
    switch (split_bucket(g.splits)) {
      case 2:
        hipLaunchKernelGGL((splitk_reduce_kernel<EPI, LAY, QKN, 2>), sgrid, dim3(256), 0,
                           rt->stream, g);
        break;
      case 4:
        hipLaunchKernelGGL((splitk_reduce_kernel<EPI, LAY, QKN, 4>), sgrid, dim3(256), 0,
                           rt->stream, g);
        break;
      default:
        hipLaunchKernelGGL((splitk_reduce_kernel<EPI, LAY, QKN, 8>), sgrid, dim3(256), 0,
                           rt->stream, g);
        break;
    }
  }
}

}  // namespace

// Per weight column: the split's exponent e, which brings the column's largest
// |w| to 2^e |w| in [2^10, 2^11), so that every value down to 2^-24 of it has both
// parts (kZeroColumn for a column of zeros); and the floor's share of a sum whose
// other factors are all tiny, 2^24 x 2^-36 x the sum of the scaled |w|.
__global__ __launch_bounds__(256) void weight_column_kernel(const float* __restrict__ wnk,
                                                            int2* __restrict__ wcol, int N,
                                                            int Kp) {
  if (blockIdx.x == 0 && threadIdx.x == 0) wcol[N].x = 0;  // split_weights_kernel's flag
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= N) return;
  uint32_t m = 0;
  for (int k = lane; k < Kp; k += 64) {
    const uint32_t b = __float_as_uint(wnk[static_cast<size_t>(row) * Kp + k]) & 0x7fffffffu;
    if (b < 0x7f800000u) m = b > m ? b : m;
  }
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) {
    const uint32_t o = __shfl_xor(m, s, 64);
    m = o > m ? o : m;
  }
  int e = 0;
  if (m) (void)frexpf(__uint_as_float(m), &e);  // m in [2^(e-1), 2^e)
  e = m ? 11 - e : kZeroColumn;
  float sum = 0.0f;
  for (int k = lane; k < Kp; k += 64) {
    const float w = fabsf(ldexpf(wnk[static_cast<size_t>(row) * Kp + k], e));
    if (vks::is_finite(w)) sum += w;
  }
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) sum += __shfl_xor(sum, s, 64);
  // a little more than the sum, for its rounding
  if (lane == 0) wcol[row] = make_int2(e, __float_as_int(sum * (1.01f / 4096.0f)));
}

// The f16 parts of the scaled rows 2^wcol[n].x wnk[n] of [N, Kp] in the order
// the wide kernel's lanes read them: 16-row tile j, 32-k stage ch, part p of
// `parts`, lane l (row 16 j + l % 16, k 32 ch + 8 (l / 16) .. + 8), 16 bytes
// each.  Rows past N and k past Kp are zeros.  One part: *rest becomes 1 if
// any second part is not zero.  stat[1 + ch][n] counts the stage's groups of 8 k
// of row n: x the dense ones and, in the high half, those that reach kWBig; y
// the weights below kTiny that the parts do not hold (column_run).
__global__ __launch_bounds__(256) void split_weights_kernel(const float* __restrict__ wnk,
                                                            const int2* __restrict__ wcol,
                                                            u32x4* __restrict__ dst, int N, int Kp,
                                                            int nch, long long pieces, int parts,
                                                            int* __restrict__ rest,
                                                            uint2* __restrict__ stat) {
  const long long i = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= pieces) return;
  const int lane = static_cast<int>(i & 63);
  const long long jc = i >> 6;
  const int ch = static_cast<int>(jc % nch);
  const long long row = (jc / nch) * 16 + (lane & 15);
  const int k0 = ch * KC + 8 * (lane >> 4);
  const int e = row < N ? wcol[row].x : 0;
  auto at = [&](int h) {
    return row < N && k0 + h < Kp ? ldexpf(wnk[static_cast<size_t>(row) * Kp + k0 + h], e) : 0.0f;
  };
  const float4 x = make_float4(at(0), at(1), at(2), at(3));
  const float4 y = make_float4(at(4), at(5), at(6), at(7));
  u32x4 p0, p1;
  vks::split8(x, y, &p0, &p1);
  const float w8[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
  uint32_t tiny = 0;
#pragma unroll
  for (int h = 0; h < 8; ++h) {
    const auto part = [&](const u32x4& p) {
      return static_cast<float>(__builtin_bit_cast(vks::f16x8, p)[h]);
    };
    tiny += fabsf(w8[h]) < kTiny && __builtin_fmaf(part(p1), vks::kDown, part(p0)) != w8[h];
  }
  uint32_t groups = (vks::min_abs8(x, y) >= kWBig ? 1u : 0u) +
                    (vks::max_abs8(x, y) >= kWBig ? 0x10000u : 0u);
#pragma unroll
  for (int s = 16; s < 64; s <<= 1) {  // the stage's four groups of a row
    groups += static_cast<uint32_t>(__shfl_xor(static_cast<int>(groups), s, 64));
    tiny += static_cast<uint32_t>(__shfl_xor(static_cast<int>(tiny), s, 64));
  }
  if (lane < 16 && row < N) stat[static_cast<size_t>(ch + 1) * N + row] = make_uint2(groups, tiny);
  dst[jc * parts * 64 + lane] = p0;
  if (parts == 2)
    dst[jc * 128 + 64 + lane] = p1;
  else if (((p1[0] | p1[1] | p1[2] | p1[3]) & 0x7fff7fffu) != 0)
    *rest = 1;
}

// Running totals of the stages' counts: stat[ch] becomes those of the stages
// before ch.
__global__ __launch_bounds__(256) void stage_totals_kernel(uint2* __restrict__ stat, int N,
                                                           int nch) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n >= N) return;
  uint2 sum = make_uint2(0, 0);
  stat[n] = sum;
  constexpr int kAhead = 16;  // loads in flight (the stores would order them one by one)
  for (int c0 = 1; c0 <= nch; c0 += kAhead) {
    uint2 v[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
      v[i] = stat[static_cast<size_t>(c0 + i <= nch ? c0 + i : nch) * N + n];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      // the halves of x wrap on their own (read back as differences)
      sum = make_uint2(((sum.x + v[i].x) & 0xffffu) | ((sum.x & 0xffff0000u) + (v[i].x & 0xffff0000u)),
                       sum.y + v[i].y);
      if (c0 + i <= nch) stat[static_cast<size_t>(c0 + i) * N + n] = sum;
    }
  }
}

int split_weights(vk_linear* lin, bool f16_values) {
  if (lin->in_features % 4 != 0) return VK_OK;  // never on the wide kernel
  const long long ntiles = (static_cast<long long>(lin->out_features) + 15) / 16;
  const long long nch = (static_cast<long long>(lin->in_features) + KC - 1) / KC;
  const long long pieces = ntiles * nch * 64;
  const long long blocks = (pieces + 255) / 256;
  VK_UNSUPPORTED_IF(blocks > 0x7fffffffLL, "linear too large");
  const int n = static_cast<int>(lin->out_features), kp = static_cast<int>(lin->k_pitch);
  // f16 values have one part unless a column's range is wider than f16's
  // (its smallest values then leave remainders): tried first, and split in two
  // where the kernel finds a remainder.
  for (int parts = f16_values ? 1 : 2; parts <= 2; ++parts) {
    // one allocation: the parts, the stages' counts, the columns, the remainder flag
    const size_t bytes = static_cast<size_t>(pieces) * 16 * parts;
    const size_t stat_bytes = (static_cast<size_t>(nch) + 1) * n * sizeof(uint2);
    VK_HIP(hipMalloc(&lin->weight_split,
                     bytes + stat_bytes + (static_cast<size_t>(n) + 1) * sizeof(int2)));
    char* base = static_cast<char*>(lin->weight_split);
    lin->weight_stat = reinterpret_cast<uint2*>(base + bytes);
    lin->weight_col = reinterpret_cast<int2*>(base + bytes + stat_bytes);
    lin->weight_parts = parts;
    hipLaunchKernelGGL(weight_column_kernel, dim3((n + 3) / 4), dim3(256), 0, nullptr,
                       lin->weight_nk, lin->weight_col, n, kp);
    VK_TRY(check_launch("weight_column_kernel"));
    hipLaunchKernelGGL(split_weights_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0,
                       nullptr, lin->weight_nk, lin->weight_col,
                       static_cast<u32x4*>(lin->weight_split), n, kp, static_cast<int>(nch),
                       pieces, parts, &lin->weight_col[n].x, lin->weight_stat);
    VK_TRY(check_launch("split_weights_kernel"));
    hipLaunchKernelGGL(stage_totals_kernel, dim3((n + 255) / 256), dim3(256), 0, nullptr,
                       lin->weight_stat, n, static_cast<int>(nch));
    VK_TRY(check_launch("stage_totals_kernel"));
    if (parts == 2) break;
    int rest = 0;
    VK_HIP(hipMemcpy(&rest, &lin->weight_col[n].x, sizeof(int), hipMemcpyDeviceToHost));
    if (!rest) return VK_OK;
    VK_HIP(hipFree(lin->weight_split));
    lin->weight_split = nullptr;
  }
  VK_HIP(hipStreamSynchronize(nullptr));
  return VK_OK;
}

int launch_linear_wide(vk_runtime* rt, const LinearArgs& g0, int epi, float* partial,
                       size_t partial_floats) {
  LinearArgs g = g0;
  // An output element's bits depend on its row of x, its column of W and the
  // plan, and the plan on (M, N, K) alone, so every layout and epilogue of one
  // shape gives the same bits.
  const long long cus = rt->cu_count > 0 ? rt->cu_count : 256;
  const int provided = linear_slices_to_provide(cus, g.M, g.N, g.K);
  const LinearPlan plan = linear_plan(cus, g.M, g.N, g.K, provided);
  g.splits = plan.splits;
  g.partial = nullptr;
  VK_UNSUPPORTED_IF(plan.tiles * g.splits > 0x7fffffffLL, "linear: %lld tiles", plan.tiles);
  // the staging loads address A and B rows with 32-bit byte offsets
  VK_UNSUPPORTED_IF(4LL * g.M * g.K >= (1LL << 32) || 4LL * g.N * g.Kp >= (1LL << 32),
                    "linear: operands of 4 GiB or more (M=%d, N=%d, K=%d)", g.M, g.N, g.K);
  if (provided > 1) {
    VK_REQUIRE(g.N % 4 == 0, "linear: split-K needs out_features % 4 == 0");
    const size_t mn = static_cast<size_t>(g.M) * g.N;
    const int most = provided > g.splits ? provided : g.splits;
    if (partial) {
      VK_UNSUPPORTED_IF(most * mn > partial_floats,
                        "linear (M=%d, N=%d, K=%d): %d split-K slices need %zu floats of "
                        "scratch, more than the %zu available",
                        g.M, g.N, g.K, most, most * mn, partial_floats);
      g.partial = partial;
    } else {
      VK_TRY(vk::ensure_work(rt, most * mn, "linear (split-K)"));
      g.partial = rt->work;
    }
  }
  VK_REQUIRE(g.splits == 1 || g.partial, "linear: a split plan without partial sums");
  const dim3 grid(static_cast<unsigned>(plan.tiles * g.splits));
  // LayerNorm after the residual epilogue: in the sum pass when there is
  // one and a row is 768 or 1024 floats, else as a separate pass
  const bool post_ln = g.ln_out != nullptr;
  VK_REQUIRE(!post_ln || (epi == kLinResidual && !g.q_out),
             "linear: the LayerNorm follows the residual epilogue only");
  const bool fused_ln = post_ln && g.splits > 1 && (g.N == 768 || g.N == 1024);
  if (g.q_out) {
    VK_REQUIRE(epi == kLinStore, "linear: the Q|K|V split takes the store epilogue");
    switch (g.qkn_mode) {
      case 0: launch_pair<kLinStore, kQkvHnd>(rt, g, plan, grid); break;
      case 1: launch_pair<kLinStore, kQkvHnd, 1>(rt, g, plan, grid); break;
      case 2: launch_pair<kLinStore, kQkvHnd, 2>(rt, g, plan, grid); break;
      case 3: launch_pair<kLinStore, kQkvHnd, 3>(rt, g, plan, grid); break;
      default: return set_error(VK_ERR_INVALID, "linear: unknown Q/K epilogue %d", g.qkn_mode);
    }
  } else if (g.a_hnd) {
    if (epi == kLinResidual)
      launch_pair<kLinResidual, kAHnd>(rt, g, plan, grid, !fused_ln);
    else if (epi == kLinStore)
      launch_pair<kLinStore, kAHnd>(rt, g, plan, grid);
    else
      return set_error(VK_ERR_INVALID, "linear: head-major input takes store or residual");
  } else {
    switch (epi) {
      case kLinStore: launch_pair<kLinStore, kPlain>(rt, g, plan, grid); break;
      case kLinGelu: launch_pair<kLinGelu, kPlain>(rt, g, plan, grid); break;
      case kLinGeluErf: launch_pair<kLinGeluErf, kPlain>(rt, g, plan, grid); break;
      default: launch_pair<kLinResidual, kPlain>(rt, g, plan, grid, !fused_ln); break;
    }
  }
  VK_TRY(check_launch("linear_wide_kernel"));
  if (fused_ln) {
    const dim3 rows(static_cast<unsigned>(g.M));
    const bool f16 = g.ln_f16 != 0;
    const int nv = g.N == 768 ? 3 : 4;
    const int spb = split_bucket(g.splits);
#define VK_SKLN(NVV, PTT, SPBB)                                                                \
  if (nv == NVV && f16 == (sizeof(PTT) == 2) && spb == SPBB)                                    \
    hipLaunchKernelGGL((splitk_residual_ln_kernel<NVV, PTT, SPBB>), rows, dim3(64), 0,          \
                       rt->stream, g);
    VK_SKLN(3, float, 2) VK_SKLN(3, float, 4) VK_SKLN(3, float, 8)
    VK_SKLN(3, uint16_t, 2) VK_SKLN(3, uint16_t, 4) VK_SKLN(3, uint16_t, 8)
    VK_SKLN(4, float, 2) VK_SKLN(4, float, 4) VK_SKLN(4, float, 8)
    VK_SKLN(4, uint16_t, 2) VK_SKLN(4, uint16_t, 4) VK_SKLN(4, uint16_t, 8)
#undef VK_SKLN
    return check_launch("splitk_residual_ln_kernel");
  }
  if (post_ln)
    return layernorm_raw(rt, g.out, g.ln_out, g.ln_gamma, g.ln_beta, g.ln_f16 != 0, g.M, g.N,
                         g.ln_eps);
  return VK_OK;
}

}  // namespace vk
