// Device token sampling: temperature / top-k / top-p over the vocabulary, one
// workgroup per row, the row held in registers.
//
// Reference semantics restated:
//   * temperature + softmax: top_k_top_p_filter (attention/top_k_top_p_filter.cuh:55-88):
//       x_i = logit_i / T;  p_i = exp(x_i - max x) / (sum_j exp(x_j - max x) + 1e-6)
//   * filter: apply_topk_topp_filter (attention_cpu/softmax_lut.cpp:233-256): in
//     descending-probability order, token i is dropped when its rank >= top_k
//     (top_k > 0) or when the mass ranked above it has reached top_p
//     (top_p < 1); the two tests are independent.
//   * draw: the reference's device draw is `top_indices[rand() % top_k]`
//     (top_k_top_p_filter.cuh:107), which has no defined device RNG; this build
//     draws u ~ U[0,1) from a counter-based hash of (seed, row, counter) and takes
//     the inverse CDF of the kept mass in token-index order — deterministic and
//     replayable inside a hipGraph (the counter is device memory).
//   * greedy (T <= 0 or top_k == 1): argmax, first maximum wins
//     (sample_from_logits, decoder/cuda_decoder.cu:7-14).
//
// The rank and mass thresholds are patterns of (non-negative) fp32 probabilities.
// A small top_k leaves few tokens that can matter, and these are ranked one against
// the other (pick_few).  Else they are found ten bits at a time from histograms in
// LDS: three passes over the registers for each.  64 rows of 50,257, top_k 40 and top_p
// 0.9: 35 us by histograms, now 19.7 (top_k 50 alone 31 and 19, top_p 0.95 alone 34, neither
// 15).  Bound by the vector instructions over a row's registers, one row being one
// workgroup: of 37,000 clocks the exponentials take 11,600, the temperature 3,600, the loads
// 5,200, the choice of the few 9,500, cells and draw 6,400.  A row over several workgroups would need
// its maximum and its sum from all of them, in the present order: two launches more, 13 us by
// the same count, and memory that the entry point does not have.  Masses are added as whole
// multiples of 2^-50, so their sums are exact to 2^-34 and do not depend on the order
// of the atomics.
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "exp_below.hpp"
#include "row_ops.hpp"

namespace llm {

constexpr int kSampleThreads = 1024;
constexpr int kSampleWaves = kSampleThreads / 64;
constexpr int kSampleSeg = 4 * kSampleThreads;  // tokens of a segment: 256 per wave, 4 per lane
constexpr int kSampleSegments = 16;             // of the longest row
constexpr int kBins = 1024;

// uniform in [0, 1) with 24 random bits (exactly representable in fp32)
__host__ __device__ __forceinline__ float sample_uniform(uint64_t seed, int row, int counter) {
  uint64_t z = seed ^ ((uint64_t)(uint32_t)row << 32) ^ (uint64_t)(uint32_t)counter;
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return (float)(z >> 40) * (1.0f / 16777216.0f);
}

struct SampleArgs {
  const float* logits;
  int V;
  float temperature;
  int top_k;
  float top_p;
  uint64_t seed;
  const int32_t* counter;  // per-row draw counter (device), or NULL -> counter0
  int counter0;
  int row0;                // row id of this launch's first row (for the draw)
  int32_t* out;
  int32_t* out2;  // optional second destination (stride out2_stride)
  int out2_stride;
};

template <typename T, typename Op>
__device__ __forceinline__ T block_reduce(T v, T* sh, Op op) {
  v = wave_reduce(v, op);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  T t = sh[0];
  for (int i = 1; i < kSampleThreads / 64; ++i) t = op(t, sh[i]);  // fixed order
  return t;
}

__device__ __forceinline__ void put_token(const SampleArgs& a, int r, int tok) {
  a.out[r] = tok;
  if (a.out2) a.out2[(size_t)r * a.out2_stride] = tok;
}

// p as a multiple of 2^-50 (p in [0, 1])
__device__ __forceinline__ unsigned long long mass_of(uint32_t bits) {
  const int e = (int)(bits >> 23) - 100;
  const unsigned long long m = (bits & 0x7FFFFFu) | (bits >> 23 ? 0x800000u : 0u);
  return e >= 0 ? m << e : e > -24 ? m >> -e : 0;
}

// Of histogram bins hist[0 .. kBins): the largest bin whose sum with all bins above
// it reaches `want`, and what is still wanted of that bin.  bin -1: all together do
// not.  One bin per thread; every thread gets the answer.
template <typename W>
struct Found {
  int bin;
  W left;
};
template <typename W>
__device__ __forceinline__ Found<W> find_bin(const W* hist, W want, W* part, Found<W>* found) {
  static_assert(kBins == kSampleThreads);
  const int lane = lane_id(), w = threadIdx.x >> 6;
  const W own = hist[threadIdx.x];
  W sum = own;  // of this wave's bins from here on
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const W o = __shfl_down(sum, off, 64);
    if (lane + off < 64) sum += o;
  }
  if (lane == 0) part[w] = sum;
  if (threadIdx.x == 0) *found = {-1, want};
  __syncthreads();
  for (int i = w + 1; i < kSampleWaves; ++i) sum += part[i];
  if (sum >= want && sum - own < want) *found = {(int)threadIdx.x, want - (sum - own)};
  __syncthreads();
  return *found;
}

// The largest pattern of the values (from `floor` on) that the weights of the values
// from it on reach `want`; 0: all together do not.
template <int NS, typename W, typename F>
__device__ __forceinline__ uint32_t find_pattern(const float (&v)[NS][4], uint32_t floor, W want, W* hist,
                                                 W* part, Found<W>* found, F weight) {
  uint32_t at = 0;
#pragma unroll 1
  for (int shift = 20; shift >= 0; shift -= 10) {
    hist[threadIdx.x] = 0;
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t bits = __float_as_uint(v[s][j]);
        asm volatile("" : "+v"(bits));  // (weights kept over the passes would not fit the registers)
        if (bits != 0 && bits >= floor && bits >> shift >> 10 == at)
          atomicAdd(&hist[bits >> shift & (kBins - 1)], weight(bits));
      }
    __syncthreads();
    const Found<W> f = find_bin(hist, want, part, found);
    if (f.bin < 0) return 0;
    at = at << 10 | (uint32_t)f.bin;
    want = f.left;
    __syncthreads();
  }
  return at;
}

// The thresholds of a top_k of at most kFewK, where no more than kFew tokens can be among
// the top_k: the row's threads form 128 groups of eight, and top_k groups' largest values
// are at least the top_k-th largest of the groups' largest, so nothing below that is kept.
// What is left is counted against one another: a value's rank and the mass above it.
// False: too many left, or groups without a value; nothing is found then.  Both thresholds
// are what find_pattern gives.
constexpr int kFewK = 64, kFew = 256, kGroups = kSampleThreads / 8;
struct Few {
  float most[kGroups];
  uint32_t bits[kFew];
  unsigned long long mass[kFew];
  float floor;
  int count;
  uint32_t rank_least, mass_least;
};
// What a value counts: those above it and beside it, and their masses.
struct Above {
  int above = 0, same = 0;
  unsigned long long mass_above = 0, mass_same = 0;

  template <int CTRL>
  __device__ __forceinline__ void add_lane() {
    above += mov_lanes<CTRL>(above);
    same += mov_lanes<CTRL>(same);
    mass_above += lane<CTRL>(mass_above);
    mass_same += lane<CTRL>(mass_same);
  }
  template <int CTRL>
  static __device__ __forceinline__ unsigned long long lane(unsigned long long x) {
    return (unsigned long long)(uint32_t)mov_lanes<CTRL>((int)(x >> 32)) << 32 | (uint32_t)mov_lanes<CTRL>((int)x);
  }
};
// v times `inv` are the probabilities; seg receives a thread's largest v of each segment.
template <int NS>
__device__ __forceinline__ bool pick_few(const float (&v)[NS][4], float inv, int top_k, unsigned long long want,
                                         Few& few, float (&seg)[NS], uint32_t* least) {
  const int t = threadIdx.x;
  float top = 0.f;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    seg[s] = fmaxf(fmaxf(v[s][0], v[s][1]), fmaxf(v[s][2], v[s][3]));
    top = fmaxf(top, seg[s]);
  }
  top *= inv;
  top = fmaxf(top, mov_dpp<0xB1>(top));
  top = fmaxf(top, mov_dpp<0x4E>(top));
  top = fmaxf(top, mov_dpp<0x141>(top));
  if (t % 8 == 0) few.most[t / 8] = top;
  if (t == 0) {
    few.floor = 0.f;
    few.count = 0;
    few.rank_least = few.mass_least = 0;
  }
  __syncthreads();
  {  // eight threads a group, each against sixteen others
    const int h0 = t % 8 * (kGroups / 8);
    int above = 0, from = 0;
#pragma unroll
    for (int k = 0; k < kGroups / 8; k += 4) {
      const f32x4 o = *reinterpret_cast<const f32x4*>(&few.most[h0 + k]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        above += o[e] > top;
        from += o[e] >= top;
      }
    }
    above += mov_lanes<0xB1>(above);
    from += mov_lanes<0xB1>(from);
    above += mov_lanes<0x4E>(above);
    from += mov_lanes<0x4E>(from);
    above += mov_lanes<0x141>(above);
    from += mov_lanes<0x141>(from);
    if (t % 8 == 0 && above < top_k && from >= top_k) few.floor = top;  // (equal ones write the same)
  }
  __syncthreads();
  const float floor = few.floor;
  if (!(floor > 0.f)) return false;
  // (v times inv reaches the floor only from `low` on, whose product is 2^-22 below it; products
  // with few bits round further)
  const float low = floor < 0x1p-100f ? 0.f : floor / inv * (1.f - 0x1p-22f);
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    if (!__ballot(seg[s] >= low)) continue;  // most waves have none in most segments
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float p = v[s][j] * inv;
      if (p >= floor) {
        const int at = atomicAdd(&few.count, 1);
        if (at < kFew) few.bits[at] = __float_as_uint(p);
      }
    }
  }
  __syncthreads();
  const int n = few.count;
  if (n > kFew) return false;
  if (t < n) few.mass[t] = mass_of(few.bits[t]);
  __syncthreads();
  // as many threads a value as n leaves, four at least
  const int per = n <= 64 ? 16 : n <= 128 ? 8 : 4, at = t / per;
  const uint32_t own = at < n ? few.bits[at] : 0u;
  Above a;
  if (own)
#pragma unroll 4
    for (int i = t % per; i < n; i += per) {
      const uint32_t o = few.bits[i];
      const unsigned long long m = few.mass[i];
      a.above += o > own;
      a.same += o == own;
      a.mass_above += o > own ? m : 0;
      a.mass_same += o == own ? m : 0;
    }
  a.add_lane<0xB1>();
  a.add_lane<0x4E>();
  if (per >= 8) a.add_lane<0x141>();  // row_half_mirror, row_mirror
  if (per >= 16) a.add_lane<0x140>();
  if (own && a.above < top_k && a.above + a.same >= top_k) few.rank_least = own;
  // (a value below the top_k-th counts for nothing: what is above it holds the mass already,
  // or nothing more is dropped)
  if (own && a.mass_above < want && a.mass_above + a.mass_same >= want) few.mass_least = own;
  __syncthreads();
  *least = max(few.rank_least, few.mass_least);
  return true;
}

// temperature <= 0 or top_k 1: the first maximum
__global__ __launch_bounds__(kSampleThreads) void sample_greedy_kernel(SampleArgs a) {
  __shared__ float shf[kSampleWaves];
  __shared__ int shi[kSampleWaves];
  const float* lg = a.logits + (size_t)blockIdx.x * a.V;
  float best = -INFINITY;
  int bi = 0x7fffffff;
#pragma unroll 8
  for (int i = threadIdx.x; i < a.V; i += kSampleThreads) {
    const float v = lg[i];
    if (v > best) {
      best = v;
      bi = i;
    }
  }
  const float m = block_reduce(best, shf, [](float x, float y) { return fmaxf(x, y); });
  int cand = (best == m) ? bi : 0x7fffffff;
  cand = block_reduce(cand, shi, [](int x, int y) { return min(x, y); });
  if (threadIdx.x == 0) put_token(a, blockIdx.x, cand == 0x7fffffff ? 0 : cand);
}

// A thread's tokens: 4 of each of NS segments, 64 apart, so that loads are whole
// lines and a wave's 256 tokens of a segment (a cell) follow one another.
template <int NS>
__global__ __launch_bounds__(kSampleThreads) void sample_rows_kernel(SampleArgs a) {
  __shared__ float shf[kSampleWaves];
  __shared__ uint32_t ranks[kBins], rank_part[kSampleWaves];
  __shared__ unsigned long long masses[kBins], mass_part[kSampleWaves];
  __shared__ Found<uint32_t> rank_found;
  __shared__ Found<unsigned long long> mass_found;
  __shared__ float cells[NS * kSampleWaves];
  __shared__ int cell;
  __shared__ float cell_left;
  __shared__ __attribute__((aligned(16))) Few few;
  const int r = blockIdx.x, lane = lane_id(), w = wave_id_uniform();
  const float* lg = a.logits + (size_t)r * a.V;
  const auto token = [&](int s, int j) { return s * kSampleSeg + w * 256 + j * 64 + lane; };
  const auto done = [&](int tok) { put_token(a, r, tok); };
  const float u = sample_uniform(a.seed, a.row0 + r, a.counter ? a.counter[r] : a.counter0);
  float v[NS][4];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    if ((s + 1) * kSampleSeg <= a.V) {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[s][j] = lg[token(s, j)];
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[s][j] = token(s, j) < a.V ? lg[token(s, j)] : -INFINITY;
    }
  }

  // temperature + softmax (reference: logits /= T; exp(x - max); / (sum + 1e-6))
  // The product with 1 / T in 64 bits is off by 2^-52 of the quotient, which lies no nearer
  // than 2^-49 to the middle of two floats: rounded, it is the quotient (a division takes
  // four times the cycles).
  const double by = 1.0 / (double)a.temperature;
  float mloc = -INFINITY;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[s][j] = (float)((double)v[s][j] * by);
      mloc = fmaxf(mloc, v[s][j]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  const float m = block_reduce(mloc, shf, [](float x, float y) { return fmaxf(x, y); });
  float sloc = 0.f;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[s][j] = exp_below(v[s][j] - m);
      sloc += v[s][j];
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  const float sum = block_reduce(sloc, shf, [](float x, float y) { return x + y; });
  if (!(sum < INFINITY)) {  // a logit that is no number, or none that is finite
    if (threadIdx.x == 0) done(0);
    return;
  }
  const float inv = 1.0f / (sum + 1e-6f);

  // top-k: the largest pattern that top_k probabilities reach (fewer that are not
  // zero: all stay).  top-p: the largest pattern whose probabilities and those above
  // hold a mass of top_p; whatever lies below has at least that much ranked above it.
  // What top-k drops cannot change that: where the mass that it leaves is less than
  // top_p, top-p drops nothing more.  A top_p below the masses' unit wants one of it: the
  // most probable alone have nothing ranked above them.
  uint32_t least = 0;
  const unsigned long long want = a.top_p < 1.0f ? max(mass_of(__float_as_uint(a.top_p)), 1ull) : ~0ull;
  // (a short row has fewer groups, the last ones of few tokens: a top_k near their number finds
  // too low a value or none.  40 rows of 1,057 tokens, top_k 50: 9.9 us, 11.3 with the attempt;
  // 64 of 1,600: 10.7 and 13.8)
  const int groups = min(kGroups, a.V / 256 * 8);
  float seg[NS];
  const bool few_found = a.top_k > 0 && a.top_k < a.V && a.top_k <= min(kFewK, groups / 4 * 3) &&
                         pick_few(v, inv, a.top_k, want, few, seg, &least);
  if (!few_found) {
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int j = 0; j < 4; ++j) v[s][j] = v[s][j] * inv;
    if (a.top_k > 0 && a.top_k < a.V)
      least = find_pattern<NS>(v, 0u, (uint32_t)a.top_k, ranks, rank_part, &rank_found,
                               [](uint32_t) { return 1u; });
    if (a.top_p < 1.0f)
      least = max(least, find_pattern<NS>(v, least, want, masses, mass_part, &mass_found,
                                          [](uint32_t bits) { return mass_of(bits); }));
  }

  // kept mass in token order: per cell, then over the cells.  Of the few only the segments that
  // hold some are walked.
  const auto keep = [&](auto by_seg) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      float part = 0.f;
      if (!decltype(by_seg)::value || __ballot(__float_as_uint(seg[s] * inv) >= least)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float p = decltype(by_seg)::value ? v[s][j] * inv : v[s][j];
          v[s][j] = __float_as_uint(p) >= least ? p : 0.f;
          part += v[s][j];
        }
        if (__ballot(part > 0.f)) part = group_sum<64>(part);
      }
      if (lane == 0) cells[s * kSampleWaves + w] = part;
    }
  };
  if (few_found) keep(std::true_type());
  else keep(std::false_type());
  __syncthreads();
  constexpr int CELLS = NS * kSampleWaves, PER = (CELLS + 63) / 64;
  if (w == 0) {
    float c[PER], own = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      c[i] = lane * PER + i < CELLS ? cells[lane * PER + i] : 0.f;
      own += c[i];
    }
    float incl = own;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float o = __shfl_up(incl, off, 64);
      if (lane >= off) incl += o;
    }
    const float Z = __shfl(incl, 63, 64);
    const float target = u * Z;
    // the first cell whose end lies past the target, else (rounding at the top of the
    // range) the last one that holds any mass
    float lo = __shfl_up(incl, 1, 64);
    if (lane == 0) lo = 0.f;
    int hit = 0x7fffffff, last = -1;
    float left = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (c[i] > 0.f) {
        last = lane * PER + i;
        if (hit == 0x7fffffff && target < lo + c[i]) {
          hit = last;
          left = target - lo;
        }
      }
      lo += c[i];
    }
    const int first = wave_reduce(hit, [](int x, int y) { return min(x, y); });
    last = wave_reduce(last, [](int x, int y) { return max(x, y); });
    if (first != 0x7fffffff) {
      if (hit == first) {
        cell = first;
        cell_left = left;
      }
    } else if (lane == 0) {
      cell = last;
      cell_left = INFINITY;
    }
  }
  __syncthreads();
  const int at = cell;
  if (at < 0) {
    if (threadIdx.x == 0) done(0);
    return;
  }
  if (w != at % kSampleWaves) return;
  // the wave's four of that segment, by one copy of what follows: with one for every segment the
  // kernel of 13 was 58 KB, now 42
  const int which = at / kSampleWaves;
  float x[4] = {};
#pragma unroll
  for (int s = 0; s < NS; ++s)
    if (s == which) {
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = v[s][j];
    }
  const float target = cell_left;
  float lo = 0.f, incl[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    incl[j] = x[j];
    if (!__ballot(x[j] > 0.f)) continue;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float o = __shfl_up(incl[j], off, 64);
      if (lane >= off) incl[j] += o;
    }
  }
  int pick = 0x7fffffff, last = -1;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (x[j] > 0.f) {
      last = token(which, j);
      if (target < lo + incl[j]) pick = min(pick, token(which, j));
    }
    lo += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, incl[j]), 63));
  }
  pick = wave_reduce(pick, [](int p, int q) { return min(p, q); });
  last = wave_reduce(last, [](int p, int q) { return max(p, q); });
  if (lane == 0) done(pick == 0x7fffffff ? last : pick);
}

template <int NS>
hipError_t launch_sample_segments(const SampleArgs& a, int rows, hipStream_t st) {
  hipLaunchKernelGGL(sample_rows_kernel<NS>, dim3(rows), dim3(kSampleThreads), 0, st, a);
  return hipGetLastError();
}
// A kernel for every number of segments: its passes walk all of its registers, so a row
// takes the time of its own length (top_k 40 and top_p 0.9, us: 20,000 tokens 20 with 5
// segments and 24 with 8; 40,000 30 with 10 and 34 with 13; 50,257 35 with 13).
template <size_t... I>
hipError_t launch_sample_n(std::index_sequence<I...>, int segments, const SampleArgs& a, int rows,
                           hipStream_t st) {
  using Launch = hipError_t (*)(const SampleArgs&, int, hipStream_t);
  static constexpr Launch launch[] = {launch_sample_segments<(int)I + 1>...};
  return launch[segments - 1](a, rows, st);
}

hipError_t launch_sample_rows(const SampleArgs& a, int rows, hipStream_t st) {
  if (a.V > kSampleSegments * kSampleSeg) return hipErrorInvalidValue;
  if (a.temperature <= 0.f || a.top_k == 1) {
    hipLaunchKernelGGL(sample_greedy_kernel, dim3(rows), dim3(kSampleThreads), 0, st, a);
    return hipGetLastError();
  }
  return launch_sample_n(std::make_index_sequence<kSampleSegments>(), (a.V + kSampleSeg - 1) / kSampleSeg, a,
                         rows, st);
}

}  // namespace llm

using namespace llm;

extern "C" int sample_rows(const float* logits, int rows, int V, float temperature, int top_k,
                           float top_p, uint64_t seed, int counter, int32_t* out, void* stream) {
  LLM_REQUIRE(rows >= 0 && V > 0, "sample_rows: bad shape");
  if (rows == 0) return LLM_OK;
  LLM_REQUIRE(logits && out, "sample_rows: NULL pointer");
  LLM_REQUIRE(V <= kSampleSegments * kSampleSeg, "sample_rows: V > 65536");
  LLM_REQUIRE(top_k >= 0 && top_p > 0.f && top_p <= 1.0f, "sample_rows: top_k >= 0, 0 < top_p <= 1");
  SampleArgs a{logits, V, temperature, top_k, top_p, seed, nullptr, counter, 0, out, nullptr, 0};
  LLM_HIP_RET(launch_sample_rows(a, rows, as_stream(stream)));
  return LLM_OK;
}

hipError_t llm::launch_sample(const float* logits, int rows, int row0, int V, float temperature,
                              int top_k, float top_p, uint64_t seed, const int32_t* counter,
                              int32_t* out, hipStream_t st) {
  SampleArgs a{logits, V, temperature, top_k, top_p, seed, counter, 0, row0, out, nullptr, 0};
  return launch_sample_rows(a, rows, st);
}

extern "C" float sample_uniform_host(uint64_t seed, int row, int counter) {
  return sample_uniform(seed, row, counter);
}
