// Paged attention with the reference's optional stages: top-k / top-p / EOS
// filtering of the attention weights and the attention-weight / score outputs.
//
// This is the full contract of cpu_paged_attention_forward
// (attention_cpu/cpu_attention_kernel.cpp:37-129) and its input/output structs
// CPUAttentionInput / CPUAttentionOutput (attention_cpu/attention_cpu.hpp:8-43:
// temperature, top_k, top_p, eos_token, eos_threshold; attention_weights,
// logits), which the GPU kernel of the reference tries to offer through its
// top_k / top_p / rerank_scores arguments
// (attention/paged_flash_attention_kernel_fused.cu:5-90, broken: Appendix A #2,
// #5).  The hot decode path never enables these stages (pa_decode.hip); this
// kernel runs when a caller asks for them.
//
// One workgroup per (row b, head h).  The whole row of scores lives in LDS
// (T <= 8192), or, for longer rows, in the caller's workspace (the row's
// scores and the list of what stays, pa_decode_ex_workspace_bytes; only its own workgroup
// touches them, so the barriers that order the LDS form order these too):
// scores -> softmax -> (the cut of the ranking by (prob, index) descending ->
// top-k / top-p mask) -> EOS threshold -> AV.  Probabilities are >= 0, so the
// unsigned order of (prob bits, index) is exactly std::greater on
// pair<float, int> — the order apply_topk_topp_filter sorts by
// (attention_cpu/softmax_lut.cpp:233-256), ties broken toward the larger index.
#include "common.hpp"
#include "pa_decode.hpp"

#include <algorithm>
#include <string>
#include <type_traits>

namespace llm {

constexpr int kFilterThreads = 1024;
constexpr int kFilterMaxT = 8192;

struct PaFilterArgs {
  const uint8_t* k_pool;
  const uint8_t* v_pool;
  const int32_t* page_table;
  const float* q;
  float* out;         // [B][H][D]
  float* probs_out;   // [B][H][T] or null
  float* scores_out;  // [B][H][T] or null
  const int32_t* beam_ids;
  const int32_t* context_lens;
  int B, H, D, T, TS;
  int num_pages, num_beams, max_tiles;
  size_t page_stride;  // elements from page p to page p + 1
  float temperature;
  uint64_t* ws_key;   // [B*H][Tp] what stays (the workspace form)
  float* ws_sc;       // [B*H][Tp] scores / probabilities (the workspace form)
  int Tp;             // row stride of ws_key / ws_sc
  int top_k;
  float top_p;
  int eos;
  float eos_thr;
  int lpt;    // lanes of a token's 16-byte pieces (a power of two); 0: rows that are no such pieces
  int shift;  // log2 of TS; -1: no power of two (a division costs some 30 instructions)
};

template <int KVT>
__device__ __forceinline__ float kv_elem(const uint8_t* pool, size_t i) {
  if constexpr (KVT == LLM_F16) {
    return (float)reinterpret_cast<const _Float16*>(pool)[i];
  } else if constexpr (KVT == LLM_BF16) {
    return __uint_as_float((uint32_t)reinterpret_cast<const uint16_t*>(pool)[i] << 16);
  } else if constexpr (KVT == LLM_F32) {
    return reinterpret_cast<const float*>(pool)[i];
  } else {
    return (float)reinterpret_cast<const int8_t*>(pool)[i];
  }
}

// Element e of a 16-byte piece.
template <int KVT>
__device__ __forceinline__ float kv_elem(const u32x4& r, int e) {
  if constexpr (KVT == LLM_F16) {
    return (float)__builtin_bit_cast(f16x8, r)[e];
  } else if constexpr (KVT == LLM_BF16) {
    return __uint_as_float(e & 1 ? r[e >> 1] & 0xFFFF0000u : r[e >> 1] << 16);
  } else if constexpr (KVT == LLM_F32) {
    return __uint_as_float(r[e]);
  } else {
    return (float)((int32_t)(r[e >> 2] << (24 - 8 * (e & 3))) >> 24);
  }
}

// Block-wide reduction of one value per thread (all threads get the result).
template <bool MAX>
__device__ __forceinline__ float block_reduce(float x, float* sh) {
  x = MAX ? wave_max(x) : wave_sum(x);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[w] = x;
  __syncthreads();
  float r = sh[0];
  for (int i = 1; i < kFilterThreads / 64; ++i) r = MAX ? fmaxf(r, sh[i]) : r + sh[i];
  return r;
}

// The cut of the ranking by (probability, index) descending: entries at or above (bits,
// index) stay.  Found digit by digit, 11 bits a pass, from a histogram of counts and masses
// of the entries that agree so far.  Masses are whole numbers of 2^-44, so that their sums
// do not depend on the order.
constexpr int kDigitBits = 11, kDigits = 1 << kDigitBits;
constexpr float kMassUnit = 17592186044416.f;  // 2^44
static_assert(kDigits == 2 * kFilterThreads, "the scan gives every thread two digits");

struct FilterHist {
  uint64_t mass[kDigits];
  uint32_t count[kDigits];
};
struct FilterCut {
  uint64_t mass;         // of the entries above the digit's
  uint32_t count, held;  // entries above the digit's, the digit's own
  int digit;             // -1: the whole row stays
};

__device__ __forceinline__ uint64_t filter_mass(float p) { return p > 0.f ? (uint64_t)(p * kMassUnit) : 0; }

// x of the lane that a row shift or a broadcast of a row's last lane names; 0 where there is none
// or in rows outside ROWS
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ uint32_t lane_from(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROWS, 0xF, true);
}
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ uint64_t lane_from(uint64_t x) {
  return (uint64_t)lane_from<CTRL, ROWS>((uint32_t)(x >> 32)) << 32 | lane_from<CTRL, ROWS>((uint32_t)x);
}
// sums over the lanes up to one's own, in rows of 16 lanes, then over the wave
template <typename T>
__device__ __forceinline__ T row_scan(T x) {
  x += lane_from<0x111>(x);
  x += lane_from<0x112>(x);
  x += lane_from<0x114>(x);
  x += lane_from<0x118>(x);
  return x;
}
template <typename T>
__device__ __forceinline__ T wave_scan(T x) {
  x = row_scan(x);
  x += lane_from<0x142, 0xA>(x);  // row_bcast 15
  x += lane_from<0x143, 0xC>(x);  // row_bcast 31
  return x;
}
__device__ __forceinline__ uint32_t lane_value(uint32_t x, int l) {
  return (uint32_t)__builtin_amdgcn_readlane((int)x, l);
}
__device__ __forceinline__ uint64_t lane_value(uint64_t x, int l) {
  return (uint64_t)lane_value((uint32_t)(x >> 32), l) << 32 | lane_value((uint32_t)x, l);
}

// The digit, from the top, at which `need` entries (0: any number) or a mass of `limit`
// (0: any) are reached; `from` holds what lies above the histogram.  Sums over lanes by register
// moves, those over the waves before one's own too (6,400 clocks a digit by
// shuffles and a walk over the waves, now 4,200).
__device__ __forceinline__ void filter_digit(const FilterHist& hist, uint32_t need, uint64_t limit,
                                             const FilterCut& from, FilterCut* out, uint64_t* sh_mass,
                                             uint32_t* sh_count) {
  static_assert(kFilterThreads / 64 <= 16, "a row of lanes sums the waves");
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int top = kDigits - 1 - 2 * tid;
  const uint32_t c0 = hist.count[top], c1 = hist.count[top - 1];
  const uint64_t m0 = hist.mass[top], m1 = hist.mass[top - 1];
  uint32_t c = wave_scan(c0 + c1);
  uint64_t m = wave_scan(m0 + m1);
  if (lane == 63) {
    sh_count[w] = c;
    sh_mass[w] = m;
  }
  if (tid == 0) out->digit = -1;
  __syncthreads();
  const bool before = lane < w;  // (w < 16)
  c += lane_value(row_scan(before ? sh_count[lane] : 0u), 15) + from.count - c0 - c1;
  m += lane_value(row_scan(before ? sh_mass[lane] : (uint64_t)0), 15) + from.mass - m0 - m1;
  const auto reached = [&](uint32_t n, uint64_t x) { return (need && n >= need) || (limit && x >= limit); };
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const uint32_t n = k ? c1 : c0;
    const uint64_t x = k ? m1 : m0;
    if (!reached(c, m) && reached(c + n, m + x)) {
      out->digit = top - k;
      out->count = c;
      out->mass = m;
      out->held = n;
    }
    c += n;
    m += x;
  }
  __syncthreads();
}

// Rows of up to kRankRow tokens: every entry's own count and mass of the entries above it,
// each against all (kRankParts threads an entry), in place of the histograms, whose six
// passes over the digits take 8 us however short the row is.  The same whole numbers.
constexpr int kRankRow = 256, kRankParts = kFilterThreads / kRankRow;
struct FilterRank {
  uint64_t key[kRankRow], own[kRankRow];      // (probability bits, index); mass
  uint64_t mass[kRankParts][kRankRow];        // of the part's entries above
  uint32_t count[kRankParts][kRankRow];
};

// A small top_k: the row's threads form 128 groups of eight; the top_k-th largest of the groups'
// largest entries has top_k entries from it on, so that whatever stays is among those.  Where
// they are few they are ranked one against the other, in place of the histograms (16 rows x 12
// heads of 2048, top 64 and 0.9: 8.8 us of 30, now 3.8).  The same whole numbers.  Its memory is the
// histograms' too: where it finds nothing they go over it behind a barrier of its own, as a wave
// that still read `count` would find it cleared and stay for barriers that no other meets.
constexpr int kFewK = 64, kFew = 256, kFewGroups = kFilterThreads / 8;
struct FilterFew {
  uint64_t key[kFew], mass[kFew];  // (probability bits, index); mass
  alignas(16) float most[kFewGroups];
  uint32_t index[kFew];            // of what stays; ~0: it does not
  uint64_t cut;
  float floor;
  uint32_t count;
};
template <int CTRL>
__device__ __forceinline__ uint32_t lane_sum(uint32_t x) {
  return x + (uint32_t)__builtin_amdgcn_mov_dpp((int)x, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
__device__ __forceinline__ uint64_t lane_sum(uint64_t x) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)x, CTRL, 0xF, 0xF, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(x >> 32), CTRL, 0xF, 0xF, true);
  return x + ((uint64_t)hi << 32 | lo);
}
// over 4, 8 or 16 neighbouring lanes: exchanges inside quads, half rows, rows
template <typename T>
__device__ __forceinline__ T lanes_sum(T x, int per) {
  x = lane_sum<0xB1>(x);
  x = lane_sum<0x4E>(x);
  if (per >= 8) x = lane_sum<0x141>(x);
  if (per >= 16) x = lane_sum<0x140>(x);
  return x;
}
// sc[0 .. Tb): probabilities, `most` the largest of this thread's (t = tid, tid + kFilterThreads,
// ..).  Lists what stays in the order of its index and gives the least of it; 0: too many, or
// groups without an entry; nothing is found then.
__device__ __forceinline__ int filter_few(const float* sc, int Tb, float most, uint32_t k, uint64_t limit, FilterFew& few,
                          uint64_t* list, uint32_t* cut_bits, int* cut_index) {
  const int tid = threadIdx.x;
  most = fmaxf(most, mov_dpp<0xB1>(most));
  most = fmaxf(most, mov_dpp<0x4E>(most));
  most = fmaxf(most, mov_dpp<0x141>(most));
  if (tid % 8 == 0) few.most[tid / 8] = most;
  if (tid == 0) {
    few.floor = 0.f;
    few.count = 0;
  }
  __syncthreads();
  {  // eight threads a group, each against sixteen others
    const int h0 = tid % 8 * (kFewGroups / 8);
    uint32_t above = 0, from = 0;
#pragma unroll
    for (int i = 0; i < kFewGroups / 8; i += 4) {
      const f32x4 o = *reinterpret_cast<const f32x4*>(&few.most[h0 + i]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        above += o[e] > most;
        from += o[e] >= most;
      }
    }
    above = lanes_sum(above, 8);
    from = lanes_sum(from, 8);
    if (tid % 8 == 0 && above < k && from >= k) few.floor = most;  // (equal ones write the same)
  }
  __syncthreads();
  const float floor = few.floor;
  if (!(floor > 0.f)) {
    __syncthreads();
    return 0;
  }
  if (most >= floor)
    for (int t = tid; t < Tb; t += kFilterThreads) {
      const float p = sc[t];
      if (!(p >= floor)) continue;
      const uint32_t at = atomicAdd(&few.count, 1u);
      if (at < kFew) {
        few.key[at] = (uint64_t)__float_as_uint(p) << 32 | (uint32_t)t;
        few.mass[at] = filter_mass(p);
      }
    }
  __syncthreads();
  const uint32_t n = few.count;
  if (n > kFew) {
    __syncthreads();
    return 0;
  }
  // as many threads an entry as n leaves, four at least
  const int per = n <= 64 ? 16 : n <= 128 ? 8 : 4;
  const uint32_t i = (uint32_t)(tid / per);
  const uint64_t key = i < n ? few.key[i] : 0;
  uint32_t above = 0;
  uint64_t mass = 0;
  if (i < n)
#pragma unroll 4
    for (uint32_t j = tid % per; j < n; j += per) {
      const bool over = few.key[j] > key;
      const uint64_t m = few.mass[j];
      above += over;
      mass += over ? m : 0;
    }
  above = lanes_sum(above, per);
  mass = lanes_sum(mass, per);
  const bool stays = i < n && above < k && (!limit || mass < limit);
  if (i < n && tid % per == 0) few.index[i] = stays ? (uint32_t)key : ~0u;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll 4
  for (uint32_t j = tid % per; j < n; j += per) {
    const uint32_t index = few.index[j];
    all += index != ~0u;
    before += index < (uint32_t)key;
  }
  all = lanes_sum(all, per);
  before = lanes_sum(before, per);
  if (stays && tid % per == 0) {
    list[before] = key;
    if (above == all - 1) few.cut = key;
  }
  if (tid == 0) few.count = all;
  __syncthreads();
  *cut_bits = (uint32_t)(few.cut >> 32);
  *cut_index = (int)(uint32_t)few.cut;
  return (int)few.count;
}

// One workgroup per (row, head).  The scores take one pass over K: 16-byte pieces, a
// token's pieces in adjacent lanes, 8 or 16 tokens of a group in flight.  The entries
// that stay are listed in the order of their index, and only their V rows are read, by all
// lanes.  16 rows x 12 heads of 64, 2048 tokens, top 64: 70 us with a token a thread, a
// sort of the row and a walk over all of it for the values, now 21.4: 11 of them the scores.  Bound by the
// latency of its steps; the 192 workgroups are one a CU.
constexpr int kValueTokens = 4;

// Sums of x[0 .. N) over lanes c, each lane giving half of what it holds to lane c ^ OFF, then OFF / 2:
// in the order in which a whole exchange at every step would add them.
template <int OFF, int N>
__device__ __forceinline__ void halve_sums(float* x, int c) {
  static_assert(OFF <= 8);
  if constexpr (N == 1) {
    x[0] += lane_xor<OFF>(x[0]);
  } else {
    const bool up = (c & OFF) != 0;
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      const float keep = up ? x[i + N / 2] : x[i], give = up ? x[i] : x[i + N / 2];
      x[i] = keep + lane_xor<OFF>(give);
    }
  }
  if constexpr (OFF > 1) halve_sums<OFF / 2, (N > 1 ? N / 2 : 1)>(x, c);
}

// FORM: kShort: rows of up to kRankRow tokens, a kernel of its own that is a third of the code (which
// a launch waits for) and of the LDS, so that a CU holds two; kLds; kWs.
// (top 50 of 100 tokens, 12 heads: one row 11.9 us in the LDS form, 10.8 in this; 32 rows 22.3, 20.0)
enum FilterForm { kShort, kLds, kWs };
template <int KVT, FilterForm FORM>
__global__ __launch_bounds__(kFilterThreads) void pa_filter_kernel(PaFilterArgs a) {
  constexpr bool WS = FORM == kWs, SHORT = FORM == kShort;
  constexpr int ES = KVT == LLM_F32 ? 4 : KVT == LLM_I8 ? 1 : 2;
  constexpr int EPL = 16 / ES;
  constexpr int kWaves = kFilterThreads / 64;
  // scores, then probabilities; the sums of the values at the end
  __shared__ float lsc[FORM != kLds ? kWaves * 256 : kFilterMaxT];
  // the histograms, then the list of what stays
  __shared__ alignas(16) uint64_t llist[SHORT ? sizeof(FilterRank) / 8 : WS ? sizeof(FilterHist) / 8 : kFilterMaxT];
  __shared__ float qs[256];
  __shared__ float sh[kWaves];
  __shared__ uint64_t sh_mass[kWaves];
  __shared__ uint32_t sh_count[kWaves];
  __shared__ FilterCut found;
  static_assert(kFewK * 8 % alignof(FilterFew) == 0 && alignof(FilterFew) <= 16);
  static_assert(sizeof(FilterRank) <= sizeof(llist) && kFewK * 8 + sizeof(FilterFew) <= sizeof(llist) &&
                    (SHORT || sizeof(FilterHist) <= sizeof(llist)),
                "the histograms and ranks lie in the list's memory, the few behind their list");
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bh = blockIdx.x;
  float* sc = WS ? a.ws_sc + (size_t)bh * a.Tp : lsc;
  uint64_t* list = WS ? a.ws_key + (size_t)bh * a.Tp : llist;
  const int b = bh / a.H, h = bh % a.H;
  const int D = a.D;
  const int r = a.beam_ids ? a.beam_ids[b] : b;
  int Tb = a.context_lens ? a.context_lens[b] : a.T;
  Tb = min(max(Tb, 0), a.T);
  const bool row_ok = r >= 0 && r < a.num_beams;
  const int32_t* table = a.page_table + ((size_t)(row_ok ? r : 0) * a.H + h) * a.max_tiles;
  auto page_of = [&](int t) -> int {  // KVTileCache::get (kv_tile_cache.hpp:21-26)
    const int tile = a.shift >= 0 ? t >> a.shift : t / a.TS;
    if (!row_ok || tile >= a.max_tiles) return -1;
    const int p = table[tile];
    return (p < 0 || p >= a.num_pages) ? -1 : p;
  };
  // element of (page, token in it)
  auto at = [&](int page, int t) {
    const int in = a.shift >= 0 ? t & ((1 << a.shift) - 1) : t % a.TS;
    return (size_t)page * a.page_stride + (size_t)in * D;
  };
  // lanes per token, tokens of a wave at a time
  const int lpt = a.lpt, tpw = lpt ? 64 / lpt : 0, c = lpt ? lane % lpt : 0, g = lpt ? lane / lpt : 0;

  // scores[t] = dot(q, k_t) / temperature; -1e9 where the tile is missing
  // (cpu_attention_kernel.cpp:61,68-86)
  if (lpt) {
    float qv[EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) qv[e] = a.q[(size_t)bh * D + c * EPL + e];
    // the waves take turns of tpw tokens each, so that short rows are spread over them
    const int step = kWaves * tpw;
    // N tokens of a group in flight; LPT lanes a token where that is known (0: lpt)
    const auto scores = [&](auto n_tokens, auto lanes) {
      constexpr int N = decltype(n_tokens)::value, LPT = decltype(lanes)::value;
      int page[N];
      auto pages = [&](int t0) {
#pragma unroll
        for (int u = 0; u < N; ++u) {
          const int t = t0 + u * step + g;
          page[u] = t < Tb ? page_of(t) : -1;
        }
      };
      if (w * tpw < Tb) pages(w * tpw);
      for (int t0 = w * tpw; t0 < Tb; t0 += N * step) {
        u32x4 k[N];
        uint32_t there = 0;
#pragma unroll
        for (int u = 0; u < N; ++u) {
          const int t = t0 + u * step + g;
          k[u] = u32x4{0u, 0u, 0u, 0u};
          if (page[u] >= 0) {
            there |= 1u << u;
            k[u] = *reinterpret_cast<const u32x4*>(a.k_pool + at(page[u], t) * ES + c * 16);
          }
        }
        if (t0 + N * step < Tb) pages(t0 + N * step);
        float dot[N];
#pragma unroll
        for (int u = 0; u < N; ++u) {
          dot[u] = 0.f;
          if (t0 + u * step < Tb) {  // (the same for the wave)
#pragma unroll
            for (int e = 0; e < EPL; ++e) dot[u] = fmaf(qv[e], kv_elem<KVT>(k[u], e), dot[u]);
          }
        }
        if constexpr (LPT > 0) {
          // every exchange halves the tokens a lane holds: lane c ends with those from c N / LPT on
          halve_sums<LPT / 2, N>(dot, c);
#pragma unroll
          for (int i = 0; i < max(N / LPT, 1); ++i) {
            const int u = c * N / LPT + i, t = t0 + u * step + g;
            if (t < Tb) sc[t] = there >> u & 1 ? dot[i] / a.temperature : -1e9f;
          }
        } else {
          for (int off = lpt >> 1; off; off >>= 1)
#pragma unroll
            for (int u = 0; u < N; ++u)
              if (t0 + u * step < Tb) dot[u] += __shfl_xor(dot[u], off, 64);
#pragma unroll
          for (int u = 0; u < N; ++u) {
            const int t = t0 + u * step + g;
            if (t0 + u * step < Tb && c == 0 && t < Tb) sc[t] = there >> u & 1 ? dot[u] / a.temperature : -1e9f;
          }
        }
      }
    };
    const std::integral_constant<int, 8> eight;
    const std::integral_constant<int, 16> sixteen;
    const bool turns = Tb > 8 * step;  // (12 heads of 64, 16 rows of 2048: 28,400 clocks by 8 tokens, 23,400)
    if (!SHORT && lpt == 8 && turns) scores(sixteen, eight);
    else if (!SHORT && lpt == 16 && turns) scores(sixteen, sixteen);
    else scores(eight, std::integral_constant<int, 0>());
  } else {
    for (int d = tid; d < D; d += kFilterThreads) qs[d] = a.q[(size_t)bh * D + d];
    __syncthreads();
    for (int t = tid; t < Tb; t += kFilterThreads) {
      const int p = page_of(t);
      float s = -1e9f;
      if (p >= 0) {
        const size_t base = at(p, t);
        float dot = 0.f;
        for (int d = 0; d < D; ++d) dot += qs[d] * kv_elem<KVT>(a.k_pool, base + d);
        s = dot / a.temperature;
      }
      sc[t] = s;
    }
  }
  __syncthreads();
  if (a.scores_out)
    for (int t = tid; t < a.T; t += kFilterThreads)
      a.scores_out[(size_t)bh * a.T + t] = t < Tb ? sc[t] : -1e9f;

  // softmax_lut_vec (softmax_lut.cpp:203-231): exp((s - max) / temperature) / (sum + 1e-6)
  float mx = -1e9f;
  for (int t = tid; t < Tb; t += kFilterThreads) mx = fmaxf(mx, sc[t]);
  mx = block_reduce<true>(mx, sh);
  float sum = 0.f;
  for (int t = tid; t < Tb; t += kFilterThreads) {
    const float e = expf((sc[t] - mx) / a.temperature);
    sc[t] = e;
    sum += e;
  }
  sum = block_reduce<false>(sum, sh);
  const float inv = 1.0f / (sum + 1e-6f);
  float most = 0.f;
  for (int t = tid; t < Tb; t += kFilterThreads) {
    const float p = sc[t] * inv;
    sc[t] = p;
    most = fmaxf(most, p);
  }

  // apply_topk_topp_filter (softmax_lut.cpp:233-256): rank by (prob, index)
  // descending; zero rank >= top_k and every entry whose preceding mass
  // (cum of the higher-ranked probabilities) is >= top_p; no renormalisation.
  uint32_t cut_bits = 0;
  int cut_index = 0;
  const bool cuts = (a.top_k > 0 || a.top_p < 1.0f) && Tb > 0;
  const uint32_t k = a.top_k > 0 ? (uint32_t)a.top_k : 0u;
  const uint64_t limit = a.top_p < 1.0f ? max((uint64_t)ceilf(a.top_p * kMassUnit), (uint64_t)1) : 0;
  // (rows of fewer groups than that find too low a bound or none)
  const bool try_few = !SHORT && k && k <= kFewK && Tb > kRankRow && (int)k <= min(Tb, kFilterThreads) / 8 / 4 * 3;
  int n_few = 0;
  if (try_few)
    n_few = filter_few(sc, Tb, most, k, limit, *reinterpret_cast<FilterFew*>(llist + kFewK), list, &cut_bits,
                       &cut_index);
  if (n_few) {
  } else if (cuts && (SHORT || Tb <= kRankRow)) {
    FilterRank& rank = *reinterpret_cast<FilterRank*>(llist);
    if (tid < Tb) {  // (the thread that wrote sc[tid])
      rank.key[tid] = (uint64_t)__float_as_uint(sc[tid]) << 32 | (uint32_t)tid;
      rank.own[tid] = filter_mass(sc[tid]);
    }
    __syncthreads();
    const int i = tid % kRankRow, part = tid / kRankRow, each = (Tb + kRankParts - 1) / kRankParts;
    if (i < Tb) {
      const uint64_t key = rank.key[i];
      const int end = min((part + 1) * each, Tb);
      uint32_t n = 0;
      uint64_t m = 0;
      for (int j = part * each; j < end; ++j) {
        const bool above = rank.key[j] > key;
        n += above ? 1u : 0u;
        m += above ? rank.own[j] : 0;
      }
      rank.count[part][i] = n;
      rank.mass[part][i] = m;
    }
    __syncthreads();
    if (tid < Tb) {
      uint32_t n = 0;
      uint64_t m = 0;
#pragma unroll
      for (int j = 0; j < kRankParts; ++j) {
        n += rank.count[j][tid];
        m += rank.mass[j][tid];
      }
      if ((k && n >= k) || (limit && m >= limit)) sc[tid] = 0.f;
    }
  } else if (!SHORT && cuts) {
    FilterHist& hist = *reinterpret_cast<FilterHist*>(llist);
    // digit `level` (0: the highest) of the bits, then of the index
    const auto histogram = [&](auto digit_of) {
      for (int i = tid; i < kDigits; i += kFilterThreads) {
        hist.mass[i] = 0;
        hist.count[i] = 0;
      }
      __syncthreads();
      for (int t = tid; t < Tb; t += kFilterThreads) {
        const float p = sc[t];
        const int d = digit_of(__float_as_uint(p), (uint32_t)t);
        if (d < 0) continue;
        atomicAdd(&hist.count[d], 1u);
        atomicAdd(reinterpret_cast<unsigned long long*>(&hist.mass[d]),
                  (unsigned long long)filter_mass(p));
      }
      __syncthreads();
    };
    FilterCut cut{0, 0, 0, 0};
    bool all = false;
    // three digits of the bits: 11, 11 and 10 of them
    for (int level = 0; level < 3 && !all; ++level) {
      const int shift = level == 0 ? 21 : level == 1 ? 10 : 0;
      const uint32_t mask = level == 2 ? 1023u : 2047u;
      const uint32_t above = level == 0 ? 0u : ~0u << (shift + (level == 2 ? 10 : 11));
      histogram([&](uint32_t bits, uint32_t) {
        return (bits & above) == cut_bits ? (int)(bits >> shift & mask) : -1;
      });
      filter_digit(hist, k, limit, cut, &found, sh_mass, sh_count);
      all = found.digit < 0;
      if (!all) {
        cut = found;
        cut_bits |= (uint32_t)cut.digit << shift;
      }
      __syncthreads();
    }
    if (all) {
      cut_bits = 0;
    } else {
      // of the equal ones at the cut the first `keep` stay, those of the largest index
      const uint64_t each = filter_mass(__uint_as_float(cut_bits));
      uint64_t keep = cut.held;
      if (k) keep = min(keep, (uint64_t)(k - cut.count));
      if (limit && each) keep = min(keep, (limit - cut.mass + each - 1) / each);
      if (keep < cut.held) {
        FilterCut from{0, 0, 0, 0};
        uint32_t index = 0;
        for (int level = 0; level < 3; ++level) {
          const int shift = 22 - 11 * level;
          const uint32_t above = level == 0 ? 0u : ~0u << (shift + 11);
          histogram([&](uint32_t bits, uint32_t t) {
            return bits == cut_bits && (t & above) == index ? (int)(t >> shift & 2047u) : -1;
          });
          filter_digit(hist, (uint32_t)keep, 0, from, &found, sh_mass, sh_count);
          from = found;
          index |= (uint32_t)from.digit << shift;
          __syncthreads();
        }
        cut_index = (int)index;
      }
    }
  }
  if (!n_few) __syncthreads();  // (the few end with theirs, and nothing they hold is written again)
  const auto stays = [&](int t) -> float {
    const float p = sc[t];
    const uint32_t bits = __float_as_uint(p);
    return bits > cut_bits || (bits == cut_bits && t >= cut_index) ? p : 0.f;
  };
  // EOS hard threshold: keep only the EOS position when its weight exceeds it
  const bool only = a.eos >= 0 && a.eos < Tb && stays(a.eos) > a.eos_thr;
  const bool whole = !cuts && !only;  // the row as it is: no list
  int n = whole ? Tb : 0;             // entries listed
  if (n_few && !only) {               // the list is there
    n = n_few;
    if (a.probs_out)
      for (int t = tid; t < a.T; t += kFilterThreads)
        a.probs_out[(size_t)bh * a.T + t] = t < Tb ? stays(t) : 0.f;
  } else for (int t0 = 0; t0 < a.T; t0 += kFilterThreads) {
    const int t = t0 + tid;
    const float p = t < Tb && !(only && t != a.eos) ? stays(t) : 0.f;
    if (a.probs_out && t < a.T) a.probs_out[(size_t)bh * a.T + t] = p;
    if (whole || t0 >= Tb) continue;
    const uint64_t kept = __ballot(p != 0.f);
    if (lane == 0) sh_count[w] = (uint32_t)__popcll(kept);
    __syncthreads();
    int before = n;
    for (int i = 0; i < kWaves; ++i) {
      before += i < w ? (int)sh_count[i] : 0;
      n += (int)sh_count[i];
    }
    if (p != 0.f)
      list[before + __popcll(kept & ((1ull << lane) - 1))] =
          (uint64_t)__float_as_uint(p) << 32 | (uint32_t)t;
    __syncthreads();
  }

  // entry j < n: (probability bits, index); a value of weight 0 is not read
  const auto entry = [&](int j) -> uint64_t {
    return whole ? (uint64_t)__float_as_uint(sc[j]) << 32 | (uint32_t)j : list[j];
  };
  // The values' sums go over the probabilities, where the loop above has its barriers behind its reads
  // of them, or there is one below; behind the few, whose probabilities others may still be reading.
  constexpr int kBehind = kFewK + sizeof(FilterFew) / 8;
  static_assert(FORM != kLds || kBehind * 8 + kWaves * 256 * sizeof(float) <= sizeof(llist));
  float* sums = FORM == kLds && n_few && !only ? reinterpret_cast<float*>(llist + kBehind) : lsc;
  const auto page_of_entry = [&](uint64_t e) { return e >> 32 ? page_of((int)(uint32_t)e) : -1; };

  // out = sum_t p_t v_t over present tiles (cpu_attention_kernel.cpp:103-117)
  if (lpt) {
    float acc[EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) acc[e] = 0.f;
    for (int j0 = w * tpw + g; j0 < n; j0 += kValueTokens * kWaves * tpw) {
      u32x4 v[kValueTokens];
      float p[kValueTokens];
#pragma unroll
      for (int u = 0; u < kValueTokens; ++u) {
        const int j = j0 + u * kWaves * tpw;
        const uint64_t item = j < n ? entry(j) : 0;
        const int t = (int)(uint32_t)item, pg = page_of_entry(item);
        p[u] = pg < 0 ? 0.f : __uint_as_float((uint32_t)(item >> 32));
        v[u] = u32x4{0u, 0u, 0u, 0u};
        if (pg >= 0) v[u] = *reinterpret_cast<const u32x4*>(a.v_pool + at(pg, t) * ES + c * 16);
      }
#pragma unroll
      for (int u = 0; u < kValueTokens; ++u)
#pragma unroll
        for (int e = 0; e < EPL; ++e) acc[e] = fmaf(p[u], kv_elem<KVT>(v[u], e), acc[e]);
    }
    if (whole) __syncthreads();
    if (w * tpw < n) {  // (the other waves' sums are not read)
      for (int off = lpt; off < 64; off <<= 1)
#pragma unroll
        for (int e = 0; e < EPL; ++e) acc[e] += __shfl_xor(acc[e], off, 64);
      if (g == 0)
#pragma unroll
        for (int e = 0; e < EPL; ++e) sums[w * D + c * EPL + e] = acc[e];
    }
  } else {
    // thread -> (dim d, group g of the list), groups summed in order at the end
    const int G = kFilterThreads / D, d = tid % D, gr = tid / D;
    float acc = 0.f;
    if (gr < G)
      for (int j = gr; j < n; j += G) {
        const uint64_t item = entry(j);
        const int t = (int)(uint32_t)item, pg = page_of_entry(item);
        if (pg < 0) continue;
        acc += __uint_as_float((uint32_t)(item >> 32)) * kv_elem<KVT>(a.v_pool, at(pg, t) + d);
      }
    if (whole) __syncthreads();
    if (gr < G) sums[gr * D + d] = acc;
  }
  __syncthreads();
  const int groups = lpt ? min(kWaves, (n + tpw - 1) / tpw) : kFilterThreads / D;
  if (tid < D) {
    float o = 0.f;
    for (int i = 0; i < groups; ++i) o += sums[i * D + tid];
    a.out[(size_t)bh * D + tid] = o;
  }
}

}  // namespace llm

using namespace llm;

namespace {
// The longest row the filtered form takes: the workspace's row stride, a power of two, must
// stay an int, and 2^30 tokens is far past any context.  (A row needs T entries; callers
// have sized the workspace by the power of two from the first version on.)
constexpr int kFilterRowMaxT = 1 << 30;
int filter_row_stride(int T) {
  int Tp = 1;
  while (Tp < T) Tp <<= 1;
  return Tp;
}
}  // namespace

extern "C" size_t pa_decode_ex_workspace_bytes(int B, int H, int T) {
  if (B <= 0 || H <= 0 || T <= kFilterMaxT || T > kFilterRowMaxT) return 0;
  return (size_t)B * H * filter_row_stride(T) * (sizeof(uint64_t) + sizeof(float));
}

extern "C" int pa_decode_ex(const pa_kv_view* kv, const float* q, float* out,
                            const int32_t* beam_ids, const int32_t* context_lens, int B, int H,
                            int D, int T, const pa_decode_options* opt, void* workspace,
                            size_t workspace_bytes, void* stream) {
  LLM_REQUIRE(kv != nullptr && opt != nullptr, "pa_decode_ex: kv / opt is NULL");
  LLM_REQUIRE(B >= 0 && H > 0 && D > 0 && T >= 0, "pa_decode_ex: bad B/H/D/T");
  LLM_REQUIRE(opt->temperature > 0.f, "pa_decode_ex: temperature must be > 0");
  const bool filtered = opt->top_k > 0 || opt->top_p < 1.0f || opt->eos_token >= 0 ||
                        opt->probs_out || opt->scores_out;
  if (!filtered) {
    // the hot path: identical maths with sm_scale = 1 / temperature^2 (Appendix A #13)
    return pa_decode(kv, q, out, beam_ids, context_lens, B, H, D, T,
                     1.0f / (opt->temperature * opt->temperature), 0, workspace,
                     workspace_bytes, stream);
  }
  if (B == 0) return LLM_OK;
  LLM_REQUIRE(q && out && kv->k_pool && kv->v_pool && kv->page_table, "pa_decode_ex: NULL pointer");
  LLM_REQUIRE(kv->num_heads == H && kv->head_dim == D, "pa_decode_ex: H/D differ from the kv view");
  LLM_REQUIRE(kv->page_size > 0 && kv->num_pages > 0 && kv->num_beams > 0 && kv->max_tiles > 0,
              "pa_decode_ex: empty kv view");
  LLM_REQUIRE(opt->top_p > 0.f, "pa_decode_ex: top_p must be > 0");
  LLM_REQUIRE(kv->page_stride == 0 ||
                  (kv->page_stride >= (int64_t)kv->page_size * kv->head_dim *
                                          kv_elem_size(kv->kv_dtype) &&
                   kv->page_stride % 16 == 0),
              "pa_decode_ex: page_stride must be 0 or >= one page and a multiple of 16");
  if (D > 256) return fail(LLM_ERR_UNSUPPORTED, "pa_decode_ex: filters / weight outputs need D <= 256");
  if (T > kFilterRowMaxT)
    return fail(LLM_ERR_UNSUPPORTED, "pa_decode_ex: filters / weight outputs need T <= 2^30");
  const bool ws_form = T > kFilterMaxT;
  const size_t need = pa_decode_ex_workspace_bytes(B, H, T);
  LLM_REQUIRE(!ws_form || (workspace != nullptr && workspace_bytes >= need &&
                           reinterpret_cast<uintptr_t>(workspace) % 8 == 0),
              "pa_decode_ex: T > 8192 with filters needs an 8-byte aligned workspace of "
              "pa_decode_ex_workspace_bytes(B, H, T)");
  PaFilterArgs a{};
  a.k_pool = static_cast<const uint8_t*>(kv->k_pool);
  a.v_pool = static_cast<const uint8_t*>(kv->v_pool);
  a.page_table = kv->page_table;
  a.q = q;
  a.out = out;
  a.probs_out = opt->probs_out;
  a.scores_out = opt->scores_out;
  a.beam_ids = beam_ids;
  a.context_lens = context_lens;
  a.B = B; a.H = H; a.D = D; a.T = T; a.TS = kv->page_size;
  a.num_pages = kv->num_pages; a.num_beams = kv->num_beams; a.max_tiles = kv->max_tiles;
  a.page_stride = kv_view_page_stride(*kv) / std::max(1, kv_elem_size(kv->kv_dtype));
  a.temperature = opt->temperature;
  if (ws_form) {
    a.Tp = filter_row_stride(T);
    a.ws_key = static_cast<uint64_t*>(workspace);
    a.ws_sc = reinterpret_cast<float*>(a.ws_key + (size_t)B * H * a.Tp);
  }
  a.top_k = opt->top_k;
  a.top_p = opt->top_p;
  a.eos = opt->eos_token;
  a.eos_thr = opt->eos_threshold;
  a.shift = (a.TS & (a.TS - 1)) == 0 ? __builtin_ctz((unsigned)a.TS) : -1;
  // rows of whole 16-byte pieces, at most a wave's lanes of them, where the pools allow
  // 16-byte loads; other rows are read element by element
  const int row_bytes = D * kv_elem_size(kv->kv_dtype), pieces = row_bytes / 16;
  const bool whole = row_bytes % 16 == 0 && pieces <= 64 && (pieces & (pieces - 1)) == 0;
  const auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  a.lpt = whole && kv_view_page_stride(*kv) % 16 == 0 && aligned(kv->k_pool) && aligned(kv->v_pool)
              ? pieces : 0;
  hipStream_t st = as_stream(stream);
  const dim3 grid(B * H), block(kFilterThreads);
#define LLM_FILTER_LAUNCH(KVT)                                                  \
  do {                                                                          \
    if (ws_form)                                                                \
      hipLaunchKernelGGL((pa_filter_kernel<KVT, kWs>), grid, block, 0, st, a);   \
    else if (T <= kRankRow)                                                     \
      hipLaunchKernelGGL((pa_filter_kernel<KVT, kShort>), grid, block, 0, st, a); \
    else                                                                        \
      hipLaunchKernelGGL((pa_filter_kernel<KVT, kLds>), grid, block, 0, st, a);  \
  } while (0)
  switch (kv->kv_dtype) {
    case LLM_F16: LLM_FILTER_LAUNCH(LLM_F16); break;
    case LLM_BF16: LLM_FILTER_LAUNCH(LLM_BF16); break;
    case LLM_F32: LLM_FILTER_LAUNCH(LLM_F32); break;
    case LLM_I8: LLM_FILTER_LAUNCH(LLM_I8); break;
    default: return fail(LLM_ERR_INVALID, "pa_decode_ex: kv_dtype");
  }
#undef LLM_FILTER_LAUNCH
  LLM_HIP_RET(hipGetLastError());
  return LLM_OK;
}
