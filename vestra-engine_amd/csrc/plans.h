// How the wide linear and the attention share their work out: tile shapes, split
// counts and the partial results' buffer, from the sizes alone.  Plain C++, so
// that a host without a GPU evaluates the same rules.
#pragma once

#include <cstddef>
#include <initializer_list>

namespace vk {

// ---------------------------------------------------------------------------
// Linear (linear.hip)
// ---------------------------------------------------------------------------
constexpr int kSplitK = 32;    // k of one stage of the wide kernel
constexpr int kMaxSplits = 8;  // most split-K slices a sum pass reads
// Most floats of split-K partial sums that a plan takes beyond what
// linear_slices_to_provide says: the allocation-free entry point's scratch.
constexpr long long kMaxPartialFloats = 8LL << 20;

struct LinearPlan {
  int tm, tn;
  int splits;
  long long tiles;
};

inline long long tile_count(int tm, int tn, int M, int N) {
  return static_cast<long long>((M + tm - 1) / tm) * static_cast<long long>((N + tn - 1) / tn);
}

// Partial slices a caller must be ready to provide for: 1 where the shape
// never splits (it can be captured before any eager call of its kind), else
// the count that the allocation-free entry point's scratch is held against.
// This is the interface's rule, held apart from what a plan takes so that what is
// refused, and what needs an eager call before capture, does not move with the
// plans' constants; a plan never takes more floats than this count, or
// kMaxPartialFloats.  It costs what no plan uses: 866 x 768 -> 768 runs unsplit
// and asks for three slices, 3,458 x 4096 -> 1024 takes two that fit the
// allocation-free scratch and is refused for eight, and a shape for which this is
// 1 never splits.  The rule: the
// cheapest of 128 x 128, 64 x 128 and 64 x 64 tiles in runs of 64-wide K
// chunks, at 5.5 us per chunk of the busiest CU's 128 x 128 tiles (0.6 and
// 0.28 of that for the others) plus the partial sums' traffic at 5.5 TB/s
// and 2 us for the sum pass; on ties the larger tile, then the smaller count.
inline int linear_slices_to_provide(long long cus, int M, int N, int K) {
  constexpr double kChunkUs = 5.5, kBytesPerUs = 5.5e6, kSumLaunchUs = 2.0;
  struct Shape {
    int tm, tn;
    double cost;
  };
  constexpr Shape kShapes[] = {{128, 128, 1.0}, {64, 128, 0.6}, {64, 64, 0.28}};
  const int nch = (K + 63) / 64;
  const long long mn = static_cast<long long>(M) * N;
  int best = 0;
  double best_us = 0.0;
  for (const Shape& sh : kShapes) {
    const long long tiles = tile_count(sh.tm, sh.tn, M, N);
    for (int sp = 1; sp == 1 || (sp <= kMaxSplits && 2 * sp <= nch && sp * mn <= (1LL << 26));
         ++sp) {
      const long long load = (tiles * sp + cus - 1) / cus * ((nch + sp - 1) / sp);
      double us = kChunkUs * sh.cost * static_cast<double>(load);
      if (sp > 1) us += 8.0 * static_cast<double>(sp * mn) / kBytesPerUs + kSumLaunchUs;
      if (best == 0 || us < best_us) {
        best = sp;
        best_us = us;
      }
    }
  }
  return best;
}

// Tile shape and split count, from a cost model fitted to plan sweeps of
// the ViT-B and ViT-L projections at 100 to 10,392 rows.  Workgroups are
// dealt round-robin to the CUs, so the busiest CU runs ceil(tiles * s / CUs)
// workgroups of up to ceil(stages / s) 32-wide K stages each: 1.3 us per stage
// of a 128 x 256 tile (and 3 us per tile that nothing else on the CU covers),
// 0.85 of a 128 x 128, 0.43 of a 64 x 128 and 0.26 of a 64 x 64 one; of the
// latter three, a CU with one workgroup has nothing to cover its waits and
// counts 1.3.  A split adds its partial sums (s x M x N floats written, then
// read by the sum pass, at about 5.5 TB/s) and the sum pass's launch (about 2
// us).  The cheapest plan wins; on ties the first shape, then the smaller
// count.  At least four stages per
// split; where the shape may split, at most kMaxStages of them: a run's
// rounding grows as the root of its length (2.0e-7 of the 64-bit result at 768 k,
// 3.0e-7 at 2,048, 3.6e-7 at 3,072, 4.1e-7 at 4,096, 5.9e-7 at 8,192), and 96
// stages keep ViT-B's longest sum in one run and let ViT-L's (K = 4096) take two,
// which is also the faster there (3,458 rows: 90 us against 97).  Measured (model's choice; neighbours): 866 x 768 ->
// 2304, 64 x 64 17.2 us (64 x 128 18.2, 128 x 128 29); 866 x 3072 -> 768, 64 x
// 64 x 3 24.4 (unsplit 35, 64 x 128 x 6 24.3); 1500 x 768 -> 2304, 64 x 128 24.3
// (64 x 64 27, 128 x 128 30); 3458 x 4096 -> 1024, 128 x 256 x 2 90 (64 x 128
// 97, 128 x 128 x 2 99); 10,392 x 3072 -> 768, 128 x 256 127 (128 x 128 136, 64
// x 128 154).
constexpr int kMaxStages = 96;

inline LinearPlan linear_plan(long long cus, int M, int N, int K, int provided) {
  constexpr double kBytesPerUs = 5.5e6, kSumLaunchUs = 2.0, kAlone = 1.3;
  // tile shape, us of one of its K stages, of one of its tiles, and the load
  // that a lone workgroup counts
  struct Shape {
    int tm, tn;
    double us, tile_us, alone;
  };
  constexpr Shape kShapes[] = {{128, 256, 1.3, 3.0, 1.0},
                               {128, 128, 0.85, 0.0, kAlone},
                               {64, 128, 0.43, 0.0, kAlone},
                               {64, 64, 0.26, 0.0, kAlone}};
  const int nch = (K + kSplitK - 1) / kSplitK;
  const long long mn = static_cast<long long>(M) * N;
  const auto may = [&](int sp) {
    return sp == 1 || (provided > 1 && sp <= kMaxSplits && 4 * sp <= nch &&
                       (sp <= provided || sp * mn <= kMaxPartialFloats));
  };
  LinearPlan best{0, 0, 1, 0};
  double best_us = 0.0;
  for (const Shape& sh : kShapes) {
    const long long tiles = tile_count(sh.tm, sh.tn, M, N);
    for (int sp = 1; may(sp); ++sp) {
      const int stages = (nch + sp - 1) / sp;
      if (stages > kMaxStages && may(sp + 1)) continue;
      const double load = static_cast<double>((tiles * sp + cus - 1) / cus);
      double us = (sh.us * stages + sh.tile_us) * (load > 1.0 ? load : sh.alone);
      if (sp > 1) us += 8.0 * static_cast<double>(sp * mn) / kBytesPerUs + kSumLaunchUs;
      if (best.tm == 0 || us < best_us) {
        best = LinearPlan{sh.tm, sh.tn, sp, tiles};
        best_us = us;
      }
    }
  }
  return best;
}

// ---------------------------------------------------------------------------
// Attention (attention.hip)
// ---------------------------------------------------------------------------
constexpr int kKeyBlock = 64;  // keys of one block
constexpr int kHeadDim = 64;

// Key splits a caller must be ready to provide for: 1 where the shape never
// splits (it can be captured before any eager call of its kind).  This is the
// interface's rule, held apart from the splits that are taken as the linear's is
// (12 x 10,392 runs unsplit and asks for three): 64-query tiles
// of fewer than two workgroups per CU split to about two (at least two key
// blocks each, at most 8); fuller grids where a model of 2.2 us per key block of the busiest CU,
// the partial results' traffic at 5.5 TB/s and 3 us for the merge pass puts a
// split at least 1% below the unsplit launch.
inline int attention_splits_to_provide(int cus, size_t sequences, size_t n) {
  const long long tiles64 = static_cast<long long>(sequences) * ((n + 63) / 64);
  const int nkb = static_cast<int>((n + kKeyBlock - 1) / kKeyBlock);
  int splits = 1;
  if (tiles64 < 2LL * cus) {
    splits = static_cast<int>((2.0 * cus) / static_cast<double>(tiles64) + 0.5);
    if (splits > nkb / 2) splits = nkb / 2;
    if (splits > 8) splits = 8;
    if (splits < 1) splits = 1;
  } else {
    constexpr double kBlockUs = 2.2, kBytesPerUs = 5.5e6, kMergeUs = 3.0;
    const double row_bytes = 4.0 * (kHeadDim + 2) * static_cast<double>(sequences * n);
    const double unsplit = kBlockUs * static_cast<double>((tiles64 + cus - 1) / cus * nkb);
    double best = unsplit;
    for (int sp = 2; sp <= 8 && 2 * sp <= nkb; ++sp) {
      const long long load = (tiles64 * sp + cus - 1) / cus * ((nkb + sp - 1) / sp);
      const double us = kBlockUs * static_cast<double>(load) +
                        2.0 * sp * row_bytes / kBytesPerUs + kMergeUs;
      if (us < best && us < 0.99 * unsplit) {
        best = us;
        splits = sp;
      }
    }
  }
  return splits;
}

// Waves per workgroup (eight: 256 queries, one workgroup a CU, half the K and V
// staging per query; four: 128 queries, two a CU) and key splits, from a cost
// model fitted to sweeps of 12 to 192 sequences of 256 to 10,392 rows: the
// busiest CU runs ceil(tiles * s / CUs) workgroups of ceil(key blocks / s)
// blocks each, 2.7 us per block of an eight-wave workgroup, 1.65 of a
// four-wave one (2.0 where the CU has no second); a split adds its partial
// results' traffic (s slices of rows x 66 floats written and read back at 5.5
// TB/s) and the merge pass (about 3 us).  Measured (choice; neighbours): 12 x
// 10,392 eight waves unsplit 920 us (2 splits 946, four waves 1064); 16 x 3,458
// eight waves unsplit 150 (2 splits 165, four waves 178); 144 x 866 four waves
// 104 (eight 124); 12 x 866 four waves in 3 splits 22.1 (unsplit 34.5, eight
// waves in 4 splits 25.0); 12 x 1,732 eight waves in 3 splits 43 (four waves
// 47, 2 splits 47).
struct AttentionPlan {
  int waves, splits;
};

inline AttentionPlan attention_plan(int cus, size_t sequences, size_t n, int provided) {
  constexpr double kBytesPerUs = 5.5e6, kMergeUs = 3.0;
  constexpr double kEightUs = 2.7, kFourUs = 1.65, kFourAloneUs = 2.0;
  const long long nkb = static_cast<long long>((n + kKeyBlock - 1) / kKeyBlock);
  const double row_bytes = 4.0 * (kHeadDim + 2) * static_cast<double>(sequences * n);
  AttentionPlan best{4, 1};
  double best_us = 0.0;
  for (const int w : {4, 8}) {
    const long long tiles = static_cast<long long>(sequences * ((n + 32 * w - 1) / (32 * w)));
    for (int sp = 1; sp == 1 || (provided > 1 && sp <= 8 && sp <= nkb); ++sp) {
      const long long load = (tiles * sp + cus - 1) / cus, blocks = (nkb + sp - 1) / sp;
      double us = static_cast<double>(load * blocks) *
                  (w == 8 ? kEightUs : (load > 1 ? kFourUs : kFourAloneUs));
      if (sp > 1) us += 2.0 * sp * row_bytes / kBytesPerUs + kMergeUs;
      if (best_us == 0.0 || us < best_us) {
        best = AttentionPlan{w, sp};
        best_us = us;
      }
    }
  }
  return best;
}

}  // namespace vk
