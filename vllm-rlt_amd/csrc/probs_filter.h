// Row-split form of the filtered sampling distributions (top-k and / or top-p; gfx950).
//
// rlt_probs_kernel (probabilities.hip) keeps a row on one CU, which bounds a launch by what
// one CU pulls and leaves the others idle when there are fewer rows than CUs; rows past
// 65536 columns do not fit there and are re-read on every pass.  This form spreads each row
// over S workgroups of 256 threads, each owning one slice of 8192 columns in registers, in
// three launches:
//
//   1. slice: the slice's maximum (and argmax key), its masses relative to its own anchor,
//      their float64 total, and a mass (and count) histogram of its larger masses;
//   2. row: one 1024-thread workgroup per row finds the cut bins from the slices'
//      histograms, lists the row's tokens of those bins and ranks them, which gives the last
//      kept token and the kept total;
//   3. write: every slice's workgroup writes its slice (a token stays iff it does not come
//      after the last kept one), and forms what the acceptance sampler or the draft step
//      wants of it.
//
// What bounds it: the slice launch's instructions per column and its reductions (19 us of 80
// rows of 151936 fp32 logits at top-p 0.9, at four workgroups a CU; write 15; row 13, its chain of
// dependent reads).  80 bf16 rows, top-k and top-p mixed, in an acceptance call: slices and the
// drafts' sums 26, row 36 (the chain three times over, one search per cut), write 18; the call
// 210 -> 102 us against one workgroup per row.  Top-p 0.9 of 160 fp32 rows 150 -> 76 us, of 8 rows
// 88 -> 27.  The earlier forms of this split that were measured: the cut and the ranking repeated
// by every slice's workgroup (the launches were latency chains of 10 us at four workgroups a
// CU: 1.5x slower), the row launch reading whole rows instead of the slices that hold tokens
// of the cut bins (608 KB by one CU: 5 to 10 us slower).
//
// Masses.  With c = log2(e) / T and A_s the slice's anchor (its maximum's l c, rounded to an
// integer), a token's mass is e = 2^(l c - A_s) (one fma, then the hardware exponential); the
// largest lies in [0.69, 1.45).  Anchors are integers, so a row's masses are its slices' times
// powers of two.
//
// Bins.  A token's bin comes from floor(64 l c), the product rounded once to fp32: it never
// falls as l grows, and equal logits share it in every slice, so bins agree with the order in
// which tokens are kept and written.  (Bins taken from the masses did not: the fma rounds
// l c - A_s by the slice's anchor, equal logits of two slices could fall on two sides of a
// bin's edge, and a row then kept one token more or less than it counted.)  Octave o of a
// slice holds the tokens with l c - A_s in [-o, 1 - o), a histogram has 64 bins in each of
// octaves 0 .. 24 and 4 in each of 25 .. 125, and a slice whose anchor is d below the row's
// moves d octaves on.  l c is rounded by at most 2^-5 (|l c| <= 2^20), so a bin's masses are
// within 7% of each other: 25-bit integers times one power of two, at most 2^18 of them, whose
// float64 sums are exact in any order (so are an octave's).
//
// Depth.  A slice's histogram ends at octave 16 unless a cut may lie deeper: at 24 when the
// mass below octave 16 exceeds a tenth of the 1 - p that a top-p cut may drop, at 125 when the
// slice has fewer than k tokens in octaves 0 .. 16 (with k of them, the row's k-th token lies
// there too).  Slices decide that alone, so a row's top-p cut can still lie below the histogram
// of one of them (its peak's slice holds little mass below octave 16, the others much): the row
// launch then reads the row and bins what lies past the octaves that all slices hold
// (deep_cut).  Rows that this form does not decide -- more tokens in the cut bins than the list
// holds (flat rows, large tie groups), logits out of range -- run the exact path
// (probs_exact.h) in the second launch.
//
// The order of tokens is the single-workgroup form's: logit descending, column ascending.
// Included inside probabilities.hip's anonymous namespace.

#pragma once

namespace filt {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / RLT_WAVE;
constexpr int E = 32;                // columns per thread
constexpr int kSlice = kThreads * E; // 8192: also one group of the cascade row sums
constexpr int kMaxSlices = 32;
constexpr int kOctaves = 126;        // [0, 126): their masses are normal floats
constexpr int kFine = 25;            // octaves of 64 bins; the others have 4
constexpr int kShallow = 16;         // last octave of the usual histogram
constexpr int kFineBins = 64, kCoarseBins = 4;
constexpr int kBins = kFine * kFineBins + (kOctaves - kFine) * kCoarseBins;
constexpr int kListCap = 2048;       // listed tokens per row
constexpr int kDeepBins = 2048;      // steps that deep_cut bins: 32 octaves
constexpr int kRowThreads = 1024;    // the row launch
constexpr int kRowWaves = kRowThreads / RLT_WAVE;
constexpr float kMaxScaled = 1048576.f;  // |l c| of a slice's maximum: 2^20
constexpr int kNoAnchor = -(1 << 28);    // a slice without any mass

struct SliceStat {
  unsigned long long best;  // argmax key: (order key, NaN highest) << 32 | ~column
  double z;                 // float64 mass relative to 2^anchor
  int32_t anchor;           // kNoAnchor: no logit of the slice has a mass
  int32_t depth;            // last octave in the histogram; -1: out of range (exact path)
};

struct Hist {
  double octave_mass[kOctaves + 1];
  uint32_t octave_cnt[kOctaves + 1];
  double mass[kBins];
  uint32_t cnt[kBins];
};

// kDeep: only inside the row launch
enum State { kNanRow = 0, kUnfiltered = 1, kCut = 2, kExact = 3, kDeep = 4 };

// What the row launch found.
struct RowCut {
  int32_t state;
  int32_t anchor;
  // bins [b_lo, b_hi] hold the last cut (their tokens are listed): earlier bins are kept,
  // later ones dropped; kBins + f: step f alone (deep_cut).  k_bin: the bin of the top-k cut
  // (listed too), or -1
  int32_t b_lo, b_hi, k_bin;
  int32_t reach;           // (kDeep) last octave that every slice's histogram holds
  uint32_t k_cnt_before;   // tokens before k_bin
  double mass_before;      // mass before b_lo
  double k_mass_before;    // mass before k_bin
  double z;                // the row's total
  // prefilter of the listed tokens' logits (a little wider than their bins)
  float l_lo, l_hi;
  float mx;                  // the row's maximum
  double kept;               // kept mass relative to 2^anchor
  unsigned long long last;   // the last kept token
};

struct View {
  SliceStat* stats;     // [(n_dist + n_arg) S]
  Hist* hist;           // [row_n S]
  RowCut* cuts;         // [n_dist]
  int S;
  int64_t n_dist, n_arg;
  // the launches' distribution rows: [row0, row0 + row_n) of the n_dist
  int64_t row0, row_n;
  int64_t* targets;     // argmax outputs, or nullptr
  int fused;            // distribution row r's argmax goes to targets[r]
  int skip_drawn;       // argmax-only rows listed in rows[] are left to the draws
  float* pm_out;        // torch-order row-sum partials of the written rows, or nullptr
  double* tile_sum;     // totals and flags of the written rows' 4096-column tiles, or nullptr
  uint32_t* tile_flags;
  int tiles;
  // the S histograms of distribution row r
  __device__ __forceinline__ Hist* row_hist(int64_t r) const { return hist + (r - row0) * S; }
};

struct Filter {
  const float* temperature;
  const int64_t* top_k;
  const float* top_p;
  int max_top_k, apply_top_p;
};

// One row's cut rule.
struct Rule {
  float c, p;
  unsigned long long kk;
  bool do_k, do_p, ok;
  __device__ __forceinline__ Rule(const Filter& f, int64_t r, int V) {
    const float temp = f.temperature[r];
    c = 1.44269504088896341f / temp;
    ok = temp > 0.f && isfinite(c);
    const int64_t k_req = f.top_k[r];
    const int64_t k_eff = (k_req > 0 && k_req < V) ? k_req : (int64_t)V;
    do_k = f.max_top_k > 0 && k_eff < V;
    kk = (unsigned long long)(k_eff < (int64_t)f.max_top_k ? k_eff : (int64_t)f.max_top_k);
    p = f.top_p[r];
    do_p = f.apply_top_p && p < 1.f;
  }
  // top-p keeps every token whose preceding mass is at most this (p <= 0 keeps one)
  __device__ __forceinline__ double limit(double z) const { return p > 0.f ? (double)p * z : 0.0; }
};

// Mass of logit l relative to 2^anchor (0 for -inf, which pads the row).
__device__ __forceinline__ float mass_of(float l, float c, float anchor) {
  return __builtin_amdgcn_exp2f(__builtin_fmaf(l, c, -anchor));
}

// First bin of octave o.
__device__ __forceinline__ int octave_bin(int o) {
  return o < kFine ? o * kFineBins : kFine * kFineBins + (o - kFine) * kCoarseBins;
}
// Step of logit l below `anchor`: 64 to the octave, 0 the first of octave 0 (a slice's own
// logits start at 31).  -inf, which pads the row, and logits far below lie past every octave.
__device__ __forceinline__ int step_of(float l, float c, int anchor) {
  return 64 * (anchor + 1) - 1 - (int)floorf(64.f * fmaxf(l * c, -4.f * kMaxScaled));
}
// Bin of a step, and the first step of a bin.
__device__ __forceinline__ int bin_of_step(int f) {
  return f < kFine * kFineBins ? f : kFine * kFineBins + ((f - kFine * kFineBins) >> 4);
}
__device__ __forceinline__ int first_step(int b) {
  return b < kFine * kFineBins ? b : kFine * kFineBins + ((b - kFine * kFineBins) << 4);
}

// Element j of thread t in a slice at column c0: c0 + 4 (256 (j / 4) + t) + j % 4.
__device__ __forceinline__ uint32_t elem_col(uint32_t base, int j) {
  return base + (uint32_t)(4 * kThreads * (j >> 2) + (j & 3));
}

// Four columns from col on (col % 4 == 0); padding past V reads -inf.  kVec: V % 4 == 0 and
// the row base aligned to four elements.  Other rows use the same wide loads on addresses
// aligned to an element only (global loads need no more), and single ones at the row's end.
template <int DT, bool kVec>
__device__ __forceinline__ void load_quad(const void* __restrict__ src, uint32_t col, int V, float* x) {
  if (kVec ? col < (uint32_t)V : col + 3 < (uint32_t)V) {
    if (DT == RLT_F32) {
      float f[4];
      const float* at = (const float*)src + col;
      if (kVec) at = (const float*)__builtin_assume_aligned(at, 16);
      __builtin_memcpy(f, at, 16);
#pragma unroll
      for (int k = 0; k < 4; ++k) x[k] = f[k];
    } else {
      uint32_t u[2];
      const uint16_t* at = (const uint16_t*)src + col;
      if (kVec) at = (const uint16_t*)__builtin_assume_aligned(at, 8);
      __builtin_memcpy(u, at, 8);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint16_t h = (uint16_t)(u[k >> 1] >> (16 * (k & 1)));
        x[k] = DT == RLT_BF16 ? bf16_bits_to_f32(h) : f16_bits_to_f32(h);
      }
    }
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      x[k] = !kVec && col + k < (uint32_t)V ? load_as_f32<DT>(src, col + k) : -INFINITY;
  }
}

template <int DT, bool kVec>
__device__ __forceinline__ void load_slice(const void* __restrict__ src, int64_t c0, int V,
                                           float (&x)[E]) {
  const uint32_t base = (uint32_t)c0 + 4 * threadIdx.x;
#pragma unroll
  for (int q = 0; q < E / 4; ++q) load_quad<DT, kVec>(src, elem_col(base, 4 * q), V, x + 4 * q);
}

template <typename T>
__device__ __forceinline__ T lane_sum(T v) {
  v += xor_val<32>(v);
  v += xor_val<16>(v);
  v += xor_val<8>(v);
  v += xor_val<4>(v);
  v += xor_val<2>(v);
  v += xor_val<1>(v);
  return v;
}

// ---------------------------------------------------------------- launch 1

struct SliceShared {
  double mass[kBins];
  uint32_t cnt[kBins];
  float mx[kWaves];
  uint32_t nan[kWaves];
  uint32_t col[kWaves];
  double z[kWaves];
  double top_mass[kWaves];
  uint32_t top_cnt[kWaves];
};

// Workgroups [0, row_n S): slices of distribution rows r = row0 + (logits row rows[r], or r);
// then n_arg S: argmax-only slices of logits rows 0 .. n_arg - 1; then the draft rows' float32 row-sum partials of the acceptance sampler (eight 8192-float groups
// per workgroup) when qm_src is set.
template <int DT, bool kVec>
__global__ __launch_bounds__(kThreads, 4) void rlt_filter_slice_kernel(
    const void* __restrict__ logits, const int64_t* __restrict__ rows, int64_t n_src,
    int64_t row_stride, int V, Filter flt, View v, const float* __restrict__ qm_src,
    int64_t qm_rows, float* __restrict__ qm_out) {
  __shared__ union {
    SliceShared s;
    cascade::ChunkSums cs[kThreads / cascade::kGroupThreads];
  } lds;
  const int t = threadIdx.x, w = t >> 6, lane = t & 63;
  const int64_t n_slices = (v.row_n + v.n_arg) * v.S;
  if ((int64_t)blockIdx.x >= n_slices) {
    const cascade::RowGeom geo = cascade::row_geom(V);
    const int sub = t / cascade::kGroupThreads, st = t % cascade::kGroupThreads;
    const int64_t task = ((int64_t)blockIdx.x - n_slices) * (kThreads / cascade::kGroupThreads) + sub;
    const int64_t qrow = geo.groups > 0 ? task / geo.groups : qm_rows;
    const int64_t g = geo.groups > 0 ? task % geo.groups : 0;
    const bool live = qrow < qm_rows;
    const float* x = qm_src + qrow * V;
    if (live) {
      if (V % 4 == 0 && (uintptr_t)qm_src % 16 == 0)
        cascade::group_chunk_sums<true>(x, g, geo.full_chunks, st, lds.cs[sub]);
      else
        cascade::group_chunk_sums<false>(x, g, geo.full_chunks, st, lds.cs[sub]);
    }
    __syncthreads();
    if (live)
      cascade::group_stream_sums(g, geo.full_chunks, st, lds.cs[sub],
                                 qm_out + (qrow * geo.groups + g) * cascade::kStreams);
    return;
  }
  SliceShared& sh = lds.s;
  const int64_t at = (int64_t)blockIdx.x / v.S;
  const int s = (int)((int64_t)blockIdx.x % v.S);
  const bool dist = at < v.row_n;
  const int64_t r = dist ? v.row0 + at : v.n_dist + at - v.row_n;
  SliceStat* stat = v.stats + r * v.S + s;
  if (!dist && v.skip_drawn && rows) {
    // an argmax-only row that is also drawn: an empty key, no logits read
    int hit = 0;
    for (int64_t i = t; i < v.n_dist; i += kThreads) hit |= rows[i] == r - v.n_dist;
    if (__syncthreads_or(hit)) {
      if (t == 0) stat->best = 0;
      return;
    }
  }
  int64_t src_r = dist ? (rows ? rows[r] : r) : r - v.n_dist;
  if (src_r < 0 || src_r >= n_src) src_r = 0;  // the row is written as NaN (launch 3)
  const int64_t c0 = (int64_t)s * kSlice;
  const void* src = (const char*)logits + src_r * row_stride * (DT == RLT_F32 ? 4 : 2);
  float x[E];
  load_slice<DT, kVec>(src, c0, V, x);
  if (dist) {
    for (int i = t; i < kBins; i += kThreads) {
      sh.mass[i] = 0.0;
      sh.cnt[i] = 0;
    }
  }
  // the first maximal column; a NaN is the maximum (the padding after the row's columns is
  // -inf and never the first)
  const uint32_t base = (uint32_t)c0 + 4 * t;
  float mx = -INFINITY;
  bool nan = false;
#pragma unroll
  for (int j = 0; j < E; ++j) {
    nan |= x[j] != x[j];
    mx = fmaxf(mx, x[j]);
  }
  const float own = mx;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, xor_at<true>(mx, off));
  const bool wave_nan = __ballot(nan) != 0;
  if (lane == 0) {
    sh.mx[w] = mx;
    sh.nan[w] = wave_nan;
  }
  __syncthreads();
  bool any_nan = false;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) {
    mx = fmaxf(mx, sh.mx[i]);
    any_nan |= sh.nan[i] != 0;
  }
  uint32_t col = 0xffffffffu;
  if (any_nan) {
#pragma unroll
    for (int j = E - 1; j >= 0; --j) col = x[j] != x[j] ? elem_col(base, j) : col;
  } else if (own == mx) {
#pragma unroll
    for (int j = E - 1; j >= 0; --j) col = x[j] == mx ? elem_col(base, j) : col;
  }
  col = min(col, xor_val<32>(col));
  col = min(col, xor_val<16>(col));
  col = min(col, xor_val<8>(col));
  col = min(col, xor_val<4>(col));
  col = min(col, xor_val<2>(col));
  col = min(col, xor_val<1>(col));
  if (lane == 0) sh.col[w] = col;
  // (each of the following meets a barrier before the waves' columns are read)
  auto best_key = [&]() {
    uint32_t first = sh.col[0];
#pragma unroll
    for (int i = 1; i < kWaves; ++i) first = min(first, sh.col[i]);
    return ((unsigned long long)(any_nan ? 0xffffffffu : order_key(mx)) << 32) | (0xffffffffu - first);
  };
  if (!dist) {
    __syncthreads();
    if (t == 0) stat->best = best_key();
    return;
  }
  const Rule rule(flt, r, V);
  const float y = mx * rule.c;
  // a slice whose logits are all -inf or far below any row maximum in range has no mass
  const bool none = !any_nan && (mx == -INFINITY || y < -kMaxScaled);
  const bool range = rule.ok && !any_nan && fabsf(y) <= kMaxScaled;
  const int anchor = range ? (int)rintf(y) : kNoAnchor;
  if (!range) {  // uniform over the workgroup
    __syncthreads();
    if (t == 0) {
      stat->best = best_key();
      stat->z = 0.0;
      stat->anchor = kNoAnchor;
      stat->depth = none ? kOctaves : -1;
    }
    return;
  }
  // the masses' total and the histogram of octaves 0 .. kShallow
  const float fa = (float)anchor;
  const bool cuts = rule.do_k || rule.do_p;
  double z = 0.0;
  // tokens with steps in [lo, hi) go to the histogram (one pass with counts, one without: a
  // branch on it per token cost as much as the rest)
  auto add = [&](int lo, int hi, auto counts, auto total) {
#pragma unroll
    for (int j = 0; j < E; ++j) {
      const float e = mass_of(x[j], rule.c, fa);
      if constexpr (decltype(total)::value) z += (double)e;
      const int f = step_of(x[j], rule.c, anchor);
      if ((uint32_t)(f - lo) < (uint32_t)(hi - lo)) {
        const int b = bin_of_step(f);
        atomicAdd(&sh.mass[b], (double)e);
        if constexpr (decltype(counts)::value) atomicAdd(&sh.cnt[b], 1u);
      }
    }
  };
  constexpr int kShallowSteps = (kShallow + 1) * kFineBins;
  if (rule.do_k) {
    add(0, kShallowSteps, std::true_type{}, std::true_type{});
  } else if (rule.do_p) {
    add(0, kShallowSteps, std::false_type{}, std::true_type{});
  } else {
#pragma unroll
    for (int j = 0; j < E; ++j) z += (double)mass_of(x[j], rule.c, fa);
  }
  z = lane_sum(z);
  if (lane == 0) sh.z[w] = z;
  __syncthreads();
  z = 0.0;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) z += sh.z[i];  // fixed order
  int depth = kShallow;
  if (cuts) {
    Hist* hist = v.row_hist(r) + s;
    double top = 0.0;
    uint32_t n_top = 0;
    auto put = [&](int o) {  // a fine octave, by one wave
      const int i = o * kFineBins + lane;
      const double m = sh.mass[i];
      hist->mass[i] = m;
      const double om = lane_sum(m);
      uint32_t on = 0;
      if (rule.do_k) {
        const uint32_t n = sh.cnt[i];
        hist->cnt[i] = n;
        on = lane_sum(n);
      }
      if (lane == 0) {
        hist->octave_mass[o] = om;
        hist->octave_cnt[o] = on;
      }
      top += om;
      n_top += on;
    };
#pragma unroll 1
    for (int o = w; o <= kShallow; o += kWaves) put(o);
    if (lane == 0) {
      sh.top_mass[w] = top;
      sh.top_cnt[w] = n_top;
    }
    __syncthreads();
    top = 0.0;
    n_top = 0;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) {
      top += sh.top_mass[i];
      n_top += sh.top_cnt[i];
    }
    if (rule.do_p && z - top > 0.1 * (1.0 - (double)rule.p) * z) depth = kFine - 1;
    if (rule.do_k && n_top < rule.kk) depth = kOctaves - 1;
    if (depth > kShallow) {  // uniform over the workgroup
      add(kShallowSteps, (depth + 1) * kFineBins, std::true_type{}, std::false_type{});
      __syncthreads();
#pragma unroll 1
      for (int o = kShallow + 1 + w; o < kFine; o += kWaves) put(o);
      for (int o = kFine + t; o <= depth; o += kThreads) {
        const int i = octave_bin(o);
        double om = 0.0;
        uint32_t on = 0;
#pragma unroll
        for (int k = 0; k < kCoarseBins; ++k) {
          hist->mass[i + k] = sh.mass[i + k];
          hist->cnt[i + k] = sh.cnt[i + k];
          om += sh.mass[i + k];
          on += sh.cnt[i + k];
        }
        hist->octave_mass[o] = om;
        hist->octave_cnt[o] = on;
      }
    }
  }
  if (t == 0) {
    stat->best = best_key();
    stat->z = z;
    stat->anchor = anchor;
    stat->depth = depth;
  }
}

// ---------------------------------------------------------------- launch 2

struct Entry {
  unsigned long long at;  // composite: position in the token order
  double mass;            // 0 once dropped by the top-k cut
};

struct RowShared {
  union {
    struct {
      union {
        Entry list[kListCap];
        double deep[kDeepBins];
      };
      double m[kRowWaves][RLT_WAVE];
      uint32_t n[kRowWaves][RLT_WAVE];
      int anchor[kMaxSlices];
    };
    exact::SharedT<kMaxStreamChunks> ex;
    cascade::ChunkSums cs[kRowThreads / cascade::kGroupThreads];
  };
  uint32_t list_n;
  unsigned long long last[kRowWaves];
  double sum[kRowWaves];
  uint32_t flag[kRowWaves];
};

// The row's histogram, gathered from the slices' by the whole workgroup: wave w reads
// slices w and w + 16, the waves' sums meet in LDS (sums over a bin or an octave are exact, so
// their order is free) and every wave holds the results.
struct RowHist {
  const Hist* hist;  // the row's slices
  int S;
  int shift, depth;  // lane s: slice s's shift to the row's anchor, its last octave; lanes
                     // from S on hold shifts past every octave
  bool counts;
  RowShared* sh;

  __device__ __forceinline__ void meet(double& m, uint32_t& n) const {
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    sh->m[w][lane] = m;
    sh->n[w][lane] = n;
    __syncthreads();
    m = 0.0;
    n = 0;
#pragma unroll
    for (int i = 0; i < kRowWaves; ++i) {
      m += sh->m[i][lane];
      n += sh->n[i][lane];
    }
    __syncthreads();
  }
  template <class F>
  __device__ __forceinline__ void slices(F f) const {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int u = 0; u < kMaxSlices / kRowWaves; ++u) {
      const int s = w + u * kRowWaves;
      f(hist[s < S ? s : 0], __builtin_amdgcn_readlane(shift, s), __builtin_amdgcn_readlane(depth, s));
    }
  }
  // Mass and count of the row's octave oct (a lane each).
  __device__ __forceinline__ void octave(int oct, double& m, uint32_t& n) const {
    m = 0.0;
    n = 0;
    slices([&](const Hist& x, int sh, int d) {
      const int o = oct - sh;
      if (o >= 0 && o <= min(d, kOctaves - 1)) {
        m += ldexp(x.octave_mass[o], -sh);
        if (counts) n += x.octave_cnt[o];
      }
    });
    meet(m, n);
  }
  // Bin `lane` of the row's octave `oct`: 64 bins, or 4 past kFine, where a slice's own
  // octave may still be a fine one (its bins are added by sixteens).
  __device__ __forceinline__ void bins(int oct, double& m, uint32_t& n) const {
    const int lane = threadIdx.x & 63;
    m = 0.0;
    n = 0;
    slices([&](const Hist& x, int sh, int d) {
      const int o = oct - sh;
      if (o < 0 || o > min(d, kOctaves - 1)) return;
      if (oct < kFine) {
        m += ldexp(x.mass[o * kFineBins + lane], -sh);
        if (counts) n += x.cnt[o * kFineBins + lane];
      } else if (lane < kCoarseBins) {
        const int per = o < kFine ? kFineBins / kCoarseBins : 1;
        const int i = octave_bin(o) + per * lane;
        double a = 0.0;
#pragma unroll 1
        for (int k = 0; k < per; ++k) {
          a += x.mass[i + k];
          if (counts) n += x.cnt[i + k];
        }
        m += ldexp(a, -sh);
      }
    });
    meet(m, n);
  }
  // Whether every slice's histogram reaches octave o of the row.
  __device__ __forceinline__ bool reaches(int o) const {
    const int lane = threadIdx.x & 63;
    return __ballot(lane < S && o - shift > depth) == 0;
  }
};

struct Crossing {
  int bin;  // -1: none, or below a slice's histogram
  double mass_before, mass;
  uint32_t cnt_before;
};

// Inclusive prefix sum over the lanes by fixed shift steps.
__device__ __forceinline__ double lane_scan(double x) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double y = __shfl_up(x, off, RLT_WAVE);
    if (lane >= off) x += y;
  }
  return x;
}

// The first bin whose cumulative mass exceeds `limit` (kMass) or whose cumulative count
// reaches `count` (the whole workgroup calls it, with the same values in every wave; every
// lane returns the same).
template <bool kMass>
__device__ __forceinline__ Crossing find(const RowHist& h, double limit, uint32_t count) {
  const int lane = threadIdx.x & 63;
  Crossing out{-1, 0.0, 0.0, 0};
  double mb = 0.0, mi = 0.0;
  uint32_t nb = 0, ni = 0;
  uint64_t hit = 0;
  int oct = 0;
  double m;
  uint32_t n;
  for (; oct < kOctaves; oct += RLT_WAVE) {
    h.octave(oct + lane, m, n);
    mi = mb + lane_scan(m);
    ni = kMass ? 0u : nb + wave_incl_scan<true>(n);
    hit = __ballot(kMass ? mi > limit : ni >= count);
    if (hit) break;
    mb = __shfl(mi, 63, RLT_WAVE);
    nb = __shfl(ni, 63, RLT_WAVE);
  }
  if (hit == 0) return out;
  int b = __ffsll((unsigned long long)hit) - 1;
  // the sums before the octave (the inclusive ones of the lane before)
  const double m_prev = __shfl(mi, b > 0 ? b - 1 : 0, RLT_WAVE);
  const uint32_t n_prev = __shfl(ni, b > 0 ? b - 1 : 0, RLT_WAVE);
  mb = b > 0 ? m_prev : mb;
  nb = b > 0 ? n_prev : nb;
  oct += b;
  if (!h.reaches(oct)) return out;
  h.bins(oct, m, n);
  mi = mb + lane_scan(m);
  ni = kMass ? 0u : nb + wave_incl_scan<true>(n);
  const int nbins = oct < kFine ? kFineBins : kCoarseBins;
  hit = __ballot(lane < nbins && (kMass ? mi > limit : ni >= count));
  // (a rounding of the two levels' sums apart: the octave's last bin)
  b = hit ? __ffsll((unsigned long long)hit) - 1 : nbins - 1;
  out.bin = octave_bin(oct) + b;
  const double mbb = __shfl(mi, b > 0 ? b - 1 : 0, RLT_WAVE);
  const uint32_t nbb = __shfl(ni, b > 0 ? b - 1 : 0, RLT_WAVE);
  out.mass_before = b > 0 ? mbb : mb;
  out.cnt_before = b > 0 ? nbb : nb;
  out.mass = __shfl(m, b, RLT_WAVE);
  return out;
}

// The logits of steps [f_lo, f_hi) of the row's anchor, widened by more than what the product
// and this quotient round.
__device__ __forceinline__ void step_range(RowCut& cut, const Rule& rule, int f_lo, int f_hi) {
  const float slack = 1e-3f + 1e-6f * fabsf((float)cut.anchor);
  auto edge = [&](int f) {  // upper edge of a step's l c
    return (float)(cut.anchor + 1) - (float)f * (1.f / kFineBins);
  };
  cut.l_hi = (edge(f_lo) + slack) / rule.c;
  cut.l_lo = (edge(f_hi) - slack) / rule.c;
}

// The row's cut bins from its slices (the whole workgroup; every lane returns the same, and
// every branch is on the row's values, so all waves meet at every barrier).
__device__ __forceinline__ RowCut row_cut(const View& v, const Rule& rule, int64_t r, bool src_ok,
                                          RowShared& sh) {
  const int lane = threadIdx.x & 63;
  RowCut cut;
  cut.state = kNanRow;
  cut.anchor = kNoAnchor;
  cut.b_lo = cut.b_hi = cut.k_bin = -1;
  cut.reach = -1;
  cut.k_cnt_before = 0;
  cut.mass_before = cut.k_mass_before = cut.z = 0.0;
  cut.l_lo = cut.l_hi = 0.f;
  cut.mx = 0.f;
  cut.kept = 0.0;
  cut.last = ~0ull;
  SliceStat st;
  st.best = 0;
  st.z = 0.0;
  st.anchor = kNoAnchor;
  st.depth = kOctaves;
  if (lane < v.S) st = v.stats[r * v.S + lane];
  unsigned long long best = st.best;
  int anchor = st.anchor;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const unsigned long long o = xor_at<true>(best, off);
    best = o > best ? o : best;
    anchor = max(anchor, xor_at<true>(anchor, off));
  }
  const uint32_t key = (uint32_t)(best >> 32);
  const float mx = key_value(key);
  if (!src_ok || !rule.ok || key == 0xffffffffu || !isfinite(mx)) return cut;
  cut.anchor = anchor;
  cut.mx = mx;
  cut.state = kExact;
  // (half the slices' range: a slice below it then has no mass next to this maximum)
  if (__ballot(st.depth < 0) || !(fabsf(mx * rule.c) <= 0.5f * kMaxScaled)) return cut;
  // the total by a fixed lane tree, relative to the row's anchor
  const int shift = anchor - st.anchor;
  const double z = lane_sum(ldexp(st.z, shift > 4096 ? -4096 : -shift));
  cut.z = cut.kept = z;
  if (threadIdx.x < (unsigned)v.S) sh.anchor[threadIdx.x] = st.anchor;
  if (!rule.do_k && !rule.do_p) {
    cut.state = kUnfiltered;
    return cut;
  }
  const RowHist h{v.row_hist(r), v.S, shift, st.depth, rule.do_k, &sh};
  double z_lo = z, z_hi = z;
  if (rule.do_k) {
    const Crossing k = find<false>(h, 0.0, (uint32_t)rule.kk);
    if (k.bin < 0) return cut;
    cut.b_lo = cut.b_hi = cut.k_bin = k.bin;
    cut.k_cnt_before = k.cnt_before;
    cut.mass_before = cut.k_mass_before = k.mass_before;
    // the survivors' mass, known up to the k bin's dropped tokens
    z_lo = k.mass_before;
    z_hi = k.mass_before + k.mass;
  }
  if (rule.do_p) {
    const Crossing lo = find<true>(h, rule.limit(z_lo), 0);
    if (lo.bin < 0) {
      // (with top-k every slice reaches its cut, and this one lies before it)
      if (rule.do_k) return cut;
      int reach = lane < v.S ? min(shift, kOctaves) + st.depth : kOctaves;
      for (int off = 32; off >= 1; off >>= 1) reach = min(reach, __shfl_xor(reach, off, RLT_WAVE));
      if (reach >= kOctaves - 1) return cut;
      for (int o = 0; o <= reach; o += RLT_WAVE) {
        double m;
        uint32_t n;
        h.octave(o + lane, m, n);
        cut.mass_before += lane_sum(o + lane <= reach ? m : 0.0);
      }
      cut.reach = reach;
      cut.state = kDeep;
      return cut;
    }
    const Crossing hi = rule.do_k ? find<true>(h, rule.limit(z_hi), 0) : lo;
    if (hi.bin < 0) return cut;
    cut.b_lo = lo.bin;
    cut.b_hi = hi.bin;
    cut.mass_before = lo.mass_before;
  }
  cut.state = kCut;
  step_range(cut, rule, first_step(cut.b_lo), first_step(max(cut.b_hi, cut.k_bin) + 1));
  return cut;
}

__device__ __forceinline__ double block_sum(RowShared& sh, double x) {
  x = lane_sum(x);
  if ((threadIdx.x & 63) == 0) sh.sum[threadIdx.x >> 6] = x;
  __syncthreads();
  x = 0.0;
  for (int i = 0; i < kRowWaves; ++i) x += sh.sum[i];
  __syncthreads();
  return x;
}

// The step of a top-p cut past octave cut.reach, which the slices' histograms do not all hold:
// one pass over the row's logits bins the 32 octaves from there on by steps (as much of a row
// as a float32 top-p below 1 can cut: 2^18 tokens past them have less than 2^-30 of its mass).
// Returns the cut at that step, or kExact.
//
// What bounds it: one CU's reads of the row and the LDS additions of the binned tokens, 15 to 30
// us of the rows that need it, where the exact path took 300 to 700: 160 rows of 151936, T = 1,
// logits of deviation 3, top-p 0.95: 704 -> 116 us (one workgroup per row: 212); 64 of 100003, T
// = 0.6, top-p 0.99: 360 -> 45 (58).  Slices that go to octave 24 already for a tenth of the
// droppable mass below octave 16 keep most rows out of it (for half of it the last case took 64,
// and no other case less than 3% less).
template <int DT, bool kVec>
__device__ __forceinline__ void deep_cut(const char* __restrict__ src, int V, const Rule& rule,
                                         RowShared& sh, RowCut& cut) {
  const int t = threadIdx.x, w = t >> 6, lane = t & 63;
  const int base = (cut.reach + 1) * kFineBins;
  __syncthreads();
  for (int i = t; i < kDeepBins; i += kRowThreads) sh.deep[i] = 0.0;
  if (t == 0) sh.list_n = kDeepBins;
  __syncthreads();
  constexpr int Q = 8;  // loads in flight (four columns each); two per slice
  static_assert(kSlice == 2 * 4 * kRowThreads && Q % 2 == 0, "two loads of the workgroup cover a slice");
  for (int s0 = 0; s0 * kSlice < V; s0 += Q / 2) {
    float x[Q][4];
#pragma unroll
    for (int q = 0; q < Q; ++q)
      load_quad<DT, kVec>(src, (uint32_t)s0 * kSlice + 4 * (kRowThreads * q + t), V, x[q]);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int s = s0 + q / 2;
      const int a = __builtin_amdgcn_readfirstlane(s * kSlice < V ? sh.anchor[s] : kNoAnchor);
      if (a != kNoAnchor) {  // uniform: the slice has mass
        const double unit = ldexp(1.0, a - cut.anchor);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int f = step_of(x[q][k], rule.c, cut.anchor) - base;
          if ((uint32_t)f < (uint32_t)kDeepBins)
            atomicAdd(&sh.deep[f], unit * (double)mass_of(x[q][k], rule.c, (float)a));
        }
      }
    }
  }
  __syncthreads();
  // the first step whose cumulative mass exceeds the limit: two steps a thread
  const double limit = rule.limit(cut.z);
  const double d0 = sh.deep[2 * t], d1 = sh.deep[2 * t + 1];
  const double own = lane_scan(d0 + d1);
  if (lane == 63) sh.sum[w] = own;
  __syncthreads();
  double before = cut.mass_before;
  for (int i = 0; i < w; ++i) before += sh.sum[i];
  before += own - (d0 + d1);
  const int first = before + d0 > limit ? 2 * t : before + d0 + d1 > limit ? 2 * t + 1 : kDeepBins;
  if (first < kDeepBins) atomicMin(&sh.list_n, (uint32_t)first);
  __syncthreads();
  const int at = (int)sh.list_n;
  if (first == at && at < kDeepBins) sh.m[0][0] = at & 1 ? before + d0 : before;
  __syncthreads();
  cut.state = kExact;
  if (at < kDeepBins) {
    const int f = base + at;
    cut.state = kCut;
    cut.mass_before = sh.m[0][0];
    cut.b_lo = cut.b_hi = kBins + f;
    step_range(cut, rule, f, f + 1);
  }
  __syncthreads();
}

// Bin of a listed token, from its logit.
__device__ __forceinline__ int listed_bin(unsigned long long at, const Rule& rule, const RowCut& cut) {
  return bin_of_step(step_of(key_value(~(uint32_t)(at >> 32)), rule.c, cut.anchor));
}

// Decides the n listed tokens (in no particular order: ranks and masses before a token are
// found by comparing it with every other, and sums over one bin are exact).  Returns the
// row's kept mass, and the position of the last kept token in `last`.
__device__ __forceinline__ double pick_listed(RowShared& sh, const RowCut& cut, const Rule& rule,
                                              int n, unsigned long long& last) {
  const int t = threadIdx.x;
  constexpr int kPer = kListCap / kRowThreads;
  Entry own[kPer];
  bool keep[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int idx = t + i * kRowThreads;
    keep[i] = idx < n;
    own[i] = keep[i] ? sh.list[idx] : Entry{0, 0.0};
  }
  double kept = 0.0;
  if (rule.do_k) {
    // the k bin's tokens follow all other listed ones; those past the k-th are dropped
    bool in_k[kPer];
    uint32_t rank[kPer];
    double others = 0.0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      in_k[i] = keep[i] && listed_bin(own[i].at, rule, cut) == cut.k_bin;
      others += keep[i] && !in_k[i] ? 1.0 : 0.0;
      rank[i] = 0;
    }
    if ((t & ~63) < n) {  // a wave that owns tokens
#pragma unroll 4
      for (int j = 0; j < n; ++j) {
        const unsigned long long o = sh.list[j].at;
#pragma unroll
        for (int i = 0; i < kPer; ++i) rank[i] += o < own[i].at;
      }
    }
    const uint32_t before = (uint32_t)block_sum(sh, others);
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      if (in_k[i] && cut.k_cnt_before + (rank[i] - before) >= rule.kk) {
        keep[i] = false;
        own[i].mass = 0.0;
      }
      if (in_k[i]) kept += own[i].mass;
    }
    kept = cut.k_mass_before + block_sum(sh, kept);
  }
  if (rule.do_p) {
    const double limit = rule.limit(rule.do_k ? kept : cut.z);
    if (rule.do_k) {
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int idx = t + i * kRowThreads;
        if (idx < n) sh.list[idx].mass = own[i].mass;
      }
      __syncthreads();
    }
    double before[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) before[i] = 0.0;
    if ((t & ~63) < n) {
#pragma unroll 4
      for (int j = 0; j < n; ++j) {
        const Entry o = sh.list[j];
#pragma unroll
        for (int i = 0; i < kPer; ++i) before[i] += o.at < own[i].at ? o.mass : 0.0;
      }
    }
    kept = 0.0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      keep[i] = keep[i] && cut.mass_before + before[i] <= limit;
      kept += keep[i] ? own[i].mass : 0.0;
    }
    kept = cut.mass_before + block_sum(sh, kept);
  }
  last = 0;
#pragma unroll
  for (int i = 0; i < kPer; ++i)
    if (keep[i] && own[i].at > last) last = own[i].at;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const unsigned long long o = xor_at<true>(last, off);
    last = o > last ? o : last;
  }
  if ((t & 63) == 0) sh.last[t >> 6] = last;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kRowWaves; ++i) last = sh.last[i] > last ? sh.last[i] : last;
  return kept;
}

// pick_listed for n <= 64 on one wave, token `own` of lane i: the results in sh.sum[0]
// and sh.last[0].
__device__ __forceinline__ void pick_few(RowShared& sh, const RowCut& cut, const Rule& rule, int n,
                                         Entry own) {
  const int lane = threadIdx.x & 63;
  bool keep = lane < n;
  double kept = 0.0;
  auto other = [&](unsigned long long x, int j) {
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)x, j);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(x >> 32), j);
    return ((unsigned long long)hi << 32) | lo;
  };
  if (rule.do_k) {
    const bool in_k = keep && listed_bin(own.at, rule, cut) == cut.k_bin;
    uint32_t rank = 0;
    for (int j = 0; j < n; ++j) rank += other(own.at, j) < own.at;
    const uint32_t before = (uint32_t)__popcll(__ballot(keep && !in_k));
    if (in_k && cut.k_cnt_before + (rank - before) >= rule.kk) {
      keep = false;
      own.mass = 0.0;
    }
    kept = cut.k_mass_before + lane_sum(in_k ? own.mass : 0.0);
  }
  if (rule.do_p) {
    const double limit = rule.limit(rule.do_k ? kept : cut.z);
    const unsigned long long bits = (unsigned long long)__double_as_longlong(own.mass);
    double before = 0.0;
    for (int j = 0; j < n; ++j)
      before += other(own.at, j) < own.at ? __longlong_as_double((long long)other(bits, j)) : 0.0;
    keep = keep && cut.mass_before + before <= limit;
    kept = cut.mass_before + lane_sum(keep ? own.mass : 0.0);
  }
  unsigned long long last = keep ? own.at : 0ull;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const unsigned long long o = xor_at<true>(last, off);
    last = o > last ? o : last;
  }
  if (lane == 0) {
    sh.sum[0] = kept;
    sh.last[0] = last;
  }
}

// One value of a draw tile: its total and flag bits (1 NaN, 2 +inf, 4 negative, 8 positive;
// see slice_tiles of probs_split.h).
__device__ __forceinline__ void tile_value(float z, double& d, uint32_t& f) {
  if (isnan(z)) f |= 1u;
  else if (isinf(z) && z > 0.f) f |= 2u;
  if (z < 0.f) f |= 4u;
  if (z > 0.f) f |= 8u;
  d += (double)z;
}
__device__ __forceinline__ uint32_t wave_flags(uint32_t f) {
  return (__ballot(f & 1u) ? 1u : 0u) | (__ballot(f & 2u) ? 2u : 0u) |
         (__ballot(f & 4u) ? 4u : 0u) | (__ballot(f & 8u) ? 8u : 0u);
}

// The slices whose histograms hold tokens in the cut bins (bit s; every lane the same): lane
// s looks at slice s's bins, those of a range past one octave counting as held.
__device__ __forceinline__ uint64_t slices_with(const View& v, int64_t r, const RowCut& cut,
                                                const RowShared& sh) {
  const int s = threadIdx.x & 63;
  bool held = s < v.S && sh.anchor[s] != kNoAnchor;
  if (held && cut.b_hi < kFine * kFineBins && cut.b_hi - cut.b_lo < 8 &&
      cut.k_bin < kFine * kFineBins) {
    const double* mass = v.row_hist(r)[s].mass;
    const int shift = (cut.anchor - sh.anchor[s]) * kFineBins;
    // (bins before the slice's first octave are empty)
    held = cut.k_bin >= shift && mass[cut.k_bin - shift] != 0.0;
    for (int b = max(cut.b_lo, shift); b <= cut.b_hi; ++b) held |= mass[b - shift] != 0.0;
  }
  return __ballot(held);
}

// One workgroup per distribution row.
template <int DT, bool kVec>
__global__ __launch_bounds__(kRowThreads) void rlt_filter_row_kernel(
    const void* __restrict__ logits, const int64_t* __restrict__ rows, int64_t n_src,
    int64_t row_stride, int V, Filter flt, View v, float* __restrict__ out, int64_t out_stride) {
  __shared__ RowShared sh;
  const int t = threadIdx.x, w = t >> 6, lane = t & 63;
  const int64_t r = v.row0 + blockIdx.x;
  int64_t src_r = rows ? rows[r] : r;
  const bool src_ok = src_r >= 0 && src_r < n_src;
  if (!src_ok) src_r = 0;
  const char* src = (const char*)logits + src_r * row_stride * (DT == RLT_F32 ? 4 : 2);
  const Rule rule(flt, r, V);
  RowCut cut = row_cut(v, rule, r, src_ok, sh);
  if (cut.state == kDeep) deep_cut<DT, kVec>(src, V, rule, sh, cut);  // uniform
  if (t == 0) sh.list_n = 0;
  __syncthreads();
  if (cut.state == kCut) {
    const bool deep = cut.b_lo >= kBins;
    // the tokens of the cut bins (a look at the logit first), each with the mass that its own
    // slice's histogram counted
    auto look = [&](float l, uint32_t col) {
      if (!(l >= cut.l_lo && l <= cut.l_hi)) return;
      const int f = step_of(l, rule.c, cut.anchor);
      const int b = deep ? kBins + f : bin_of_step(f);
      if (!((b >= cut.b_lo && b <= cut.b_hi) || b == cut.k_bin)) return;
      const uint32_t at = atomicAdd(&sh.list_n, 1u);
      const int a = sh.anchor[col / kSlice];
      if (at < (uint32_t)kListCap)
        sh.list[at] = Entry{composite(order_key(l), col),
                            ldexp((double)mass_of(l, rule.c, (float)a), a - cut.anchor)};
    };
    // only the slices that hold such tokens: a top-k cut's bin holds a few, in as many slices
    uint64_t left = slices_with(v, r, cut, sh);
    constexpr int U = 4;  // slices in flight
    while (left) {
      float x[2 * U][4];
      uint32_t col[2 * U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int s = left ? __ffsll((unsigned long long)left) - 1 : kMaxSlices;  // (past V: -inf)
        left &= left - 1;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          col[2 * u + q] = (uint32_t)s * kSlice + 4 * (kRowThreads * q + t);
          load_quad<DT, kVec>(src, col[2 * u + q], V, x[2 * u + q]);
        }
      }
#pragma unroll
      for (int u = 0; u < 2 * U; ++u) {
        bool any = false;
#pragma unroll
        for (int k = 0; k < 4; ++k) any |= x[u][k] >= cut.l_lo && x[u][k] <= cut.l_hi;
        if (any) {
#pragma unroll
          for (int k = 0; k < 4; ++k) look(x[u][k], col[u] + k);
        }
      }
    }
    __syncthreads();
    const int n = (int)min(sh.list_n, 0x7fffffffu);
    if (n > kListCap) {
      cut.state = kExact;  // crowded
    } else if (n <= RLT_WAVE) {
      // the common case, on one wave: lane i decides token i
      if (t < RLT_WAVE) pick_few(sh, cut, rule, n, t < n ? sh.list[t] : Entry{0, 0.0});
      __syncthreads();
      cut.kept = sh.sum[0];
      cut.last = sh.last[0];
    } else {
      cut.kept = pick_listed(sh, cut, rule, n, cut.last);
    }
  }
  if (t == 0) v.cuts[r] = cut;
  if (cut.state != kExact) return;  // uniform over the workgroup
  __syncthreads();
  exact::exact_row<DT>(sh.ex, r, logits, src_r, row_stride, V, flt.temperature, flt.top_k,
                       flt.top_p, flt.max_top_k, flt.apply_top_p, out, out_stride);
  // the written row is read back for what the callers want of it (the barrier makes every
  // wave's stores visible to the workgroup)
  const float* x = out + r * out_stride;
  __syncthreads();
  if (v.pm_out) {
    const cascade::RowGeom geo = cascade::row_geom(V);
    const int sub = t / cascade::kGroupThreads, st = t % cascade::kGroupThreads;
    constexpr int kPer = kRowThreads / cascade::kGroupThreads;
    for (int64_t g0 = 0; g0 < geo.groups; g0 += kPer) {
      const int64_t g = g0 + sub;
      if (g < geo.groups) cascade::group_chunk_sums<false>(x, g, geo.full_chunks, st, sh.cs[sub]);
      __syncthreads();
      if (g < geo.groups)
        cascade::group_stream_sums(g, geo.full_chunks, st, sh.cs[sub],
                                   v.pm_out + (r * geo.groups + g) * cascade::kStreams);
      __syncthreads();
    }
  }
  for (int k = 0; v.tile_sum && k < v.tiles; ++k) {
    double d = 0.0;
    uint32_t f = 0;
    for (int i = 0; i < 4; ++i) {
      const int64_t col = (int64_t)k * split::kBlockCols + i * kRowThreads + t;
      if (col < V) tile_value(x[col], d, f);
    }
    d = lane_sum(d);
    f = wave_flags(f);
    if (lane == 0) {
      sh.sum[w] = d;
      sh.flag[w] = f;
    }
    __syncthreads();
    if (t == 0) {
      d = 0.0;
      f = 0;
      for (int i = 0; i < kRowWaves; ++i) {
        d += sh.sum[i];
        f |= sh.flag[i];
      }
      v.tile_sum[r * v.tiles + k] = d;
      v.tile_flags[r * v.tiles + k] = f;
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------- launch 3

struct WriteShared {
  float stage[kSlice];
  cascade::ChunkSums cs;
  double tile[2][kWaves];
  uint32_t tile_flag[2][kWaves];
};

// What the callers want of a written slice's values y: torch-order float32 row-sum partials
// (cascade.h; the slice is one group), and the draw's totals and flags of its two 4096-column
// tiles.
__device__ __forceinline__ void finish_slice(WriteShared& sh, const float (&y)[E], int64_t s, int V,
                                             const View& v, int64_t r) {
  const int t = threadIdx.x, w = t >> 6, lane = t & 63;
  if (v.pm_out) {
    const cascade::RowGeom geo = cascade::row_geom(V);
#pragma unroll
    for (int q = 0; q < E / 4; ++q)
      *(float4*)(sh.stage + 4 * (kThreads * q + t)) =
          make_float4(y[4 * q], y[4 * q + 1], y[4 * q + 2], y[4 * q + 3]);
    __syncthreads();
    const int64_t fc = geo.full_chunks - s * cascade::kGroupChunks;
    const bool live = t < cascade::kGroupThreads && fc > 0;
    if (live) cascade::group_chunk_sums<true>(sh.stage, 0, fc, t, sh.cs);
    __syncthreads();
    if (live)
      cascade::group_stream_sums(0, fc, t, sh.cs,
                                 v.pm_out + (r * geo.groups + s) * cascade::kStreams);
  }
  if (v.tile_sum) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      double d = 0.0;
      uint32_t f = 0;
#pragma unroll
      for (int j = 16 * k; j < 16 * k + 16; ++j) {
        const float z = y[j];
        if (elem_col((uint32_t)(s * kSlice) + 4 * t, j) >= (uint32_t)V) continue;
        tile_value(z, d, f);
      }
      d = lane_sum(d);
      const uint32_t wf = wave_flags(f);
      if (lane == 0) {
        sh.tile[k][w] = d;
        sh.tile_flag[k][w] = wf;
      }
    }
    __syncthreads();
    const int64_t tile = 2 * s + t;
    if (t < 2 && tile < v.tiles) {
      double d = 0.0;
      uint32_t f = 0;
#pragma unroll
      for (int i = 0; i < kWaves; ++i) {
        d += sh.tile[t][i];
        f |= sh.tile_flag[t][i];
      }
      v.tile_sum[r * v.tiles + tile] = d;
      v.tile_flags[r * v.tiles + tile] = f;
    }
  }
}

template <int DT, bool kVec>
__global__ __launch_bounds__(kThreads) void rlt_filter_write_kernel(
    const void* __restrict__ logits, const int64_t* __restrict__ rows, int64_t n_src,
    int64_t row_stride, int V, Filter flt, View v, float* __restrict__ out, int64_t out_stride,
    int out_vec) {
  __shared__ WriteShared sh;
  const int t = threadIdx.x;
  const int64_t n_slices = v.row_n * v.S;
  if ((int64_t)blockIdx.x >= n_slices) {
    // argmax-only rows, one thread each; a row left to its draw has empty keys
    const int64_t i = ((int64_t)blockIdx.x - n_slices) * kThreads + t;
    if (i >= v.n_arg || !v.targets) return;
    const SliceStat* st = v.stats + (v.n_dist + i) * v.S;
    unsigned long long best = 0;
    for (int s = 0; s < v.S; ++s) best = st[s].best > best ? st[s].best : best;
    if (v.skip_drawn && best == 0) return;
    v.targets[i] = split::argmax_column(best);
    return;
  }
  const int64_t r = v.row0 + (int64_t)blockIdx.x / v.S;
  const int s = (int)((int64_t)blockIdx.x % v.S);
  int64_t src_r = rows ? rows[r] : r;
  const bool src_ok = src_r >= 0 && src_r < n_src;
  if (!src_ok) src_r = 0;
  const int64_t c0 = (int64_t)s * kSlice;
  const void* src = (const char*)logits + src_r * row_stride * (DT == RLT_F32 ? 4 : 2);
  float y[E];
  load_slice<DT, kVec>(src, c0, V, y);
  const Rule rule(flt, r, V);
  const RowCut cut = v.cuts[r];
  if (v.fused && v.targets && s == 0 && t < RLT_WAVE) {
    unsigned long long best = t < v.S ? v.stats[r * v.S + t].best : 0ull;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      const unsigned long long o = xor_at<true>(best, off);
      best = o > best ? o : best;
    }
    if (t == 0) v.targets[r] = split::argmax_column(best);
  }
  float* dst = out + r * out_stride;
  if (cut.state == kExact) return;  // written by the row launch
  const uint32_t base = (uint32_t)c0 + 4 * t;
  if (cut.state == kNanRow) {
#pragma unroll
    for (int j = 0; j < E; ++j) y[j] = NAN;
  } else {
    // outputs from the logits' distance to the row's maximum, so that the largest carry the
    // exponential's smallest error; the maximum's share of that error leaves the total too
    const double top = exp2(__builtin_fma((double)cut.mx, (double)rule.c, -(double)cut.anchor));
    const double summed = (double)mass_of(cut.mx, rule.c, (float)cut.anchor);
    // (in two floats: rounded to one, every value of a row was off by up to 6e-8 the same way;
    // 64 rows of 151936, bf16, T = 0.7, top-p 0.9: 4.2e-8 -> 3.9e-8 from float64, one workgroup 4.3e-8)
    const double share = top / (cut.kept - summed + top);
    const float inv = (float)share;
    const float inv_lo = (float)(share - (double)inv);
    auto value = [&](float l) {
      const float e = __builtin_amdgcn_exp2f((l - cut.mx) * rule.c);
      return __builtin_fmaf(e, inv, e * inv_lo);
    };
    if (cut.state == kCut) {
      const float l_last = key_value(~(uint32_t)(cut.last >> 32));
      const uint32_t c_last = (uint32_t)cut.last;
#pragma unroll
      for (int j = 0; j < E; ++j) {
        const bool keep = y[j] > l_last || (y[j] == l_last && elem_col(base, j) <= c_last);
        y[j] = keep ? value(y[j]) : 0.f;
      }
    } else {
#pragma unroll
      for (int j = 0; j < E; ++j) y[j] = value(y[j]);
    }
  }
  // streamed stores: no pass of the launch reads the row back, and lines left dirty in the
  // L2 would be written back at the kernel boundary, ahead of the next launch's work.  Rows
  // not aligned to 16 bytes take the same wide stores on 4-byte aligned addresses (a wave's
  // store still covers whole lines but two)
  typedef float f32v4u __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
  for (int q = 0; q < E / 4; ++q) {
    const uint32_t col = elem_col(base, 4 * q);
    const split::f32v4 x = {y[4 * q], y[4 * q + 1], y[4 * q + 2], y[4 * q + 3]};
    if (out_vec) {
      if (col + 3 < (uint32_t)V) __builtin_nontemporal_store(x, (split::f32v4*)(dst + col));
    } else {
      if (col + 3 < (uint32_t)V) __builtin_nontemporal_store((f32v4u)x, (f32v4u*)(dst + col));
    }
    if (col < (uint32_t)V && col + 3 >= (uint32_t)V) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (col + k < (uint32_t)V) dst[col + k] = y[4 * q + k];
    }
  }
  finish_slice(sh, y, s, V, v, r);
}

}  // namespace filt
