// Causal paged attention of a prompt chunk on MFMA (the reference's is_prefill
// pass: AttentionCUDA's `is_prefill` flag, attention/attention_cuda.hpp:21,
// with the maths of cpu_paged_attention_forward,
// attention_cpu/cpu_attention_kernel.cpp:37-129, per query token).
//
// m query tokens of ONE sequence sit at positions p0 .. p0+m-1 and their K/V
// are already in the sequence's pages (page-table row `row`).  Query i attends
// to positions 0 .. p0+i.  The decode kernel computes the same thing with one
// wave per (token, head), so each page is re-read once per query token; here a
// workgroup of 4 waves owns 64 consecutive queries of one head, loads every
// stage of K and V (32 keys; 64 where D is 64) into LDS ONCE, and each wave runs
//   S^T[32 keys][16 queries] = K · Q^T     (v_mfma_f32_16x16x32_f16)
//   O^T[D][16 queries]     += V^T · P^T
// with the flash online softmax (log2 units, as pa_split_kernel) in between.
//
// A stage goes from memory straight into LDS, one stage ahead, its loads shared
// out among the waves, with the pages of 64 groups of 16 keys looked up a lane each.
// The 16-byte chunks of a row are exchanged by the key so that the 16 rows of a
// fragment lie in different banks.
//
// Bound by the vector instructions of the softmax and the matrix cores, each on its own
// wave: what counts is waves to choose from and few instructions.  2048 queries x 16
// heads x 128: 61 us with stages of 64 keys, two waves a SIMD; 55 with half the LDS and
// four waves; 49 with the maximum moved only when it grew by more than 1, halves made
// by conversions in pairs, LDS offsets in the instructions and page lookups in one
// load (183 -> 141 instructions of both kinds a wave and 32 keys, 32 of them products).
//
// Orientation: keys are the MFMA row index of S^T, so the C layout of S^T
// (lane l: rows 4(l>>4)+r, column l&15) already holds, per lane, 8 keys of ONE
// query: that is the B operand of the P·V product once the 32 keys are taken
// in the k order slot(key) = 8·((key&15)>>2) + 4·(key>>4) + (key&3).  V is
// row-major and its V^T A operand, in that same key order, is two
// hardware-transposed LDS reads (ds_read_b64_tr_b16) per 16 dims.  The query is the lane's column in both
// products, so the running max / sum / rescale are per lane (the 4 lanes of a
// query agree after a 2-step max exchange).
//
// Accuracy: q (fp32, pre-scaled by sm_scale·log2e) and p (fp32) are split into
// fp16 hi + lo halves and each product is two MFMAs; K and V are fp16 already.
// Both are first scaled by a power of two (q per query to |q|max ≈ 2^14, p by
// 2^14) because the MFMA drops fp16 subnormal inputs: unscaled, the lo half
// of every p < 0.25 was lost (1e-5 .. 5e-5 output error, measured).  Scaled,
// products of fp16 pairs are exact in the fp32 accumulator and the output
// error is at the decode kernel's level (scripts/diag_prefill.py).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <type_traits>

#include "common.hpp"
#include "ln_wave.hpp"
#include "pa_decode.hpp"
#include "row_ops.hpp"

namespace llm {
namespace {

struct PaPrefillArgs {
  const float* q;
  int q_stride;  // floats between query rows
  float* out;
  int out_stride;
  const uint8_t* k_pool;
  const uint8_t* v_pool;
  size_t page_stride;     // bytes
  const int32_t* pt_row;  // page_table + row * H * max_tiles
  int H, max_tiles, num_pages;
  int p0, m;
  float qscale;  // sm_scale * log2(e)
  // key-range split (blockIdx.z = split s: tiles [s*pps, (s+1)*pps)); with
  // part_acc the unnormalised state goes to the decode layout
  // [(i*H + h)*nsplit + s][D] / [..][2] (m, l) for pa_merge_rows_internal
  int nsplit, pps;
  float* part_acc;
  float* part_ml;
  _Float16* out16;  // one pass: packed fp16 rows of H * D (a_frag_off_f16) in place of out
};

constexpr int stage_keys(int D) { return D == 64 ? 64 : 32; }
constexpr int kWaves = 4;
constexpr int kTileQueries = 16 * kWaves;  // of a workgroup
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
constexpr float kPScale = 16384.f;  // P enters the PV MFMA as p * 2^14 (hi + lo)

__device__ __forceinline__ void split_f16(float x, _Float16& hi, _Float16& lo) {
  hi = (_Float16)x;
  lo = (_Float16)(x - (float)hi);
}

// Two values' fp16 halves (the asm: the compiler makes each hi a second time for its lo).
__device__ __forceinline__ void split_pair(float x, float y, uint32_t& hi, uint32_t& lo) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x, y}, f16x2));
  asm("" : "+v"(hi));
  const f16x2 h = __builtin_bit_cast(f16x2, hi);
  lo = __builtin_bit_cast(uint32_t, f16x2{(_Float16)(x - (float)h[0]), (_Float16)(y - (float)h[1])});
}

// KEYS: of a stage; 4 workgroups' stages fill a CU's LDS where these are stage_keys(D), 2 else.
template <int D, int TS, int KEYS>
__global__ __launch_bounds__(64 * kWaves, KEYS == stage_keys(D) ? 4 : 2) void pa_prefill_kernel(PaPrefillArgs a) {
  constexpr int ROWB = 2 * D;                // bytes of a key's row
  constexpr int CPR = D / 8;                 // its 16-byte chunks
  constexpr int kStageKeys = KEYS;
  constexpr int OWN = kStageKeys / kWaves;   // keys of a stage that a wave loads, of one page
  constexpr int LOADS = OWN * ROWB / 1024;   // its loads of 1 KiB, each of K and V
  constexpr int BLOCKS = kStageKeys / 32, GROUPS = kStageKeys / 16;
  constexpr int NKK = D / 32;                // k-steps of q.k
  constexpr int ND = D / 16;                 // 16-dim tiles of the output
  constexpr int QW = 16, QT = kTileQueries;  // queries of a wave, of the workgroup
  static_assert(D % 32 == 0 && TS % 16 == 0 && 16 % OWN == 0 && OWN * ROWB % 1024 == 0, "shape");
  __shared__ u32x4 lds[2][2][kStageKeys * CPR];  // [stage][K, V][key][chunk, exchanged]

  const int lane = threadIdx.x & 63;
  const int w = wave_id_uniform();
  const int g = lane >> 4;
  const int c = lane & 15;
  // heads go round the XCDs: the tiles of a head share its K and V in one L2, and
  // every XCD has long and short ones
  const int h = blockIdx.x;
  const int qbase = ((int)gridDim.y - 1 - (int)blockIdx.y) * QT;  // the longest first
  const int q0 = qbase + w * QW;                                  // this wave's first query
  const int lastpos = a.p0 + min(qbase + QT, a.m) - 1;  // last key any query here sees
  const int wave_first = a.p0 + q0;
  const int wave_last = q0 < a.m ? a.p0 + min(q0 + QW, a.m) - 1 : -1;
  const int split = blockIdx.z;
  const int s0 = split * (a.pps * TS / kStageKeys);
  const int s1 = min(a.nsplit > 1 ? (split + 1) * (a.pps * TS / kStageKeys) : INT_MAX,
                     lastpos / kStageKeys + 1);
  // no query of this workgroup reaches this split: the merge never reads it
  if (s0 >= s1) return;
  const int32_t* pt = a.pt_row + (size_t)h * a.max_tiles;

  // Lane i: the page of the split's 16-key group `group` + i (-1: none, or past lastpos).
  auto pages_from = [&](int group) -> int {
    const int key = s0 * kStageKeys + 16 * (group + lane), tile = key / TS;
    const int pg = key <= lastpos && tile < a.max_tiles ? pt[tile] : -1;
    return pg < a.num_pages ? pg : -1;
  };
  // LDS position of chunk `ch` of key k (0..15 of a group): 16 rows that read one
  // chunk each meet 16 different bank groups, and so do 8 rows that read two
  auto exchange = [](int k, int ch) { return ch ^ (CPR == 16 ? ((k << 1) | (k >> 3)) & 15 : (k >> 1) & 7); };
  auto issue = [&](int buf, int s, int page) {  // this wave's keys of stage s
    const int key0 = s * kStageKeys + OWN * w / 16 * 16, at = OWN * w * CPR;  // (of their group)
    if (page < 0) {  // masked: V = 0, since 0 * NaN would not be 0
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        lds[buf][0][at + 64 * i + lane] = u32x4{0u, 0u, 0u, 0u};
        lds[buf][1][at + 64 * i + lane] = u32x4{0u, 0u, 0u, 0u};
      }
      return;
    }
    const size_t base = (size_t)page * a.page_stride + (size_t)(key0 % TS) * ROWB;
    const uint8_t *k = a.k_pool + base, *v = a.v_pool + base;  // of all lanes
    const uint32_t last = lastpos - key0;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const uint32_t row = OWN * w % 16 + (64 * i + lane) / CPR, ch = exchange(row, (64 * i + lane) % CPR);
      // (rows past lastpos may never have been written: the last one that was, masked)
      const uint32_t off = min(row, last) * ROWB + 16 * ch;
      load_to_lds(k + off, &lds[buf][0][at + 64 * i]);
      load_to_lds(v + off, &lds[buf][1][at + 64 * i]);
    }
  };
  constexpr unsigned ALL = (1u << GROUPS) - 1;
  const int own = OWN * w / 16;  // the group of this wave's keys
  int pages = pages_from(0), more = pages_from(64);
  unsigned long long there = __ballot(pages >= 0);
  unsigned valid = (unsigned)there & ALL;
  issue(0, s0, __builtin_amdgcn_readlane(pages, own));

  // Q^T B-operand fragments: lane holds q[qi][32kk + 8g .. +7] (pre-scaled by
  // qscale), hi + lo.  The query's values are also scaled by a power of two
  // 2^(14-e) (|q|max < 2^e) so the lo halves stay clear of fp16 subnormals,
  // which the MFMA does not keep; S is scaled back exactly after the MFMA.
  f16x8 qh[NKK], ql[NKK];
  float qinv;
  {
    const int qi = q0 + c;
    float qx[NKK][8];
    float amax = 0.f;
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      f32x4 x0 = {0.f, 0.f, 0.f, 0.f}, x1 = x0;
      if (qi < a.m) {
        const float* qp = a.q + (size_t)qi * a.q_stride + h * D + 32 * kk + 8 * g;
        x0 = *reinterpret_cast<const f32x4*>(qp);
        x1 = *reinterpret_cast<const f32x4*>(qp + 4);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        qx[kk][e] = x0[e] * a.qscale;
        qx[kk][4 + e] = x1[e] * a.qscale;
        amax = fmaxf(amax, fmaxf(fabsf(qx[kk][e]), fabsf(qx[kk][4 + e])));
      }
    }
    amax = fmaxf(amax, __shfl_xor(amax, 16, 64));
    amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
    int qe = 0;
    (void)frexpf(amax, &qe);  // amax < 2^qe (0 for amax == 0)
    qe = min(max(qe, -100), 100);
    const float qsc = ldexpf(1.f, 14 - qe);
    qinv = ldexpf(1.f, qe - 14);
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        _Float16 hi, lo;
        split_f16(qx[kk][e] * qsc, hi, lo);
        qh[kk][e] = hi;
        ql[kk][e] = lo;
      }
  }

  f32x4 O[ND];
  float mrun = kNegSentinel, mtop = kNegSentinel, lrun = 0.f;
#pragma unroll
  for (int nd = 0; nd < ND; ++nd) O[nd] = f32x4{0.f, 0.f, 0.f, 0.f};

  // V's place in LDS for 16 dims of the first block.  A operand lane l: V^T[d = 16nd +
  // (l&15)][k 8g+j] = V[key(8g+j)][d], keys 4g..4g+3 then 16+4g..16+4g+3: two transposed reads
  // of 4 V rows x 16 columns, lane 4q+p addressing row q, columns 4p..
  uint32_t vat[ND];
#pragma unroll
  for (int nd = 0; nd < ND; ++nd) {
    const int vk = 4 * g + (c >> 2), p4 = c & 3;
    vat[nd] = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) u32x4*)&lds[0][0][0] + vk * ROWB +
              16 * exchange(vk, 2 * nd + (p4 >> 1)) + 8 * (p4 & 1);
  }

  // stage s of the split, in buffer BUF: known, its LDS offsets are in the instructions
  auto stage = [&](auto BUF, int s) {
    constexpr int buf = decltype(BUF)::value;
    wait_lds_loads();
    __syncthreads();  // stage s has landed, the other buffer is read out
    const int at = (s + 1 - s0) * GROUPS % 64;  // the next one's groups
    if (at == 0) {
      pages = more;
      more = pages_from((s + 1 - s0) * GROUPS + 64);
      there = __ballot(pages >= 0);
    }
    const unsigned here_all = valid;
    valid = (unsigned)(there >> at) & ALL;
    if (s + 1 < s1) issue(buf ^ 1, s + 1, __builtin_amdgcn_readlane(pages, at + own));
#pragma unroll
    for (int kb = 0; kb < BLOCKS; ++kb) {
      const int key0 = s * kStageKeys + 32 * kb;
      if (key0 > wave_last) break;
      const unsigned here = here_all >> (2 * kb) & 3u;  // of the block's two 16-key tiles
      // S^T: two 16-key tiles
      f32x4 sc[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        sc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
        const u32x4* krow = &lds[buf][0][(32 * kb + 16 * u + c) * CPR];
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk) {
          const f16x8 kf = __builtin_bit_cast(f16x8, krow[exchange(c, 4 * kk + g)]);
          sc[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qh[kk], sc[u], 0, 0, 0);
          sc[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, ql[kk], sc[u], 0, 0, 0);
        }
      }
      float mloc = -INFINITY;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) mloc = fmaxf(mloc, sc[u][r]);
      // causal + missing-page mask
      if (key0 + 31 > wave_first || here != 3u) {
        mloc = -INFINITY;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if (!(here >> u & 1u) || key0 + 16 * u + 4 * g + r > wave_first + c)
              sc[u][r] = -INFINITY;
            mloc = fmaxf(mloc, sc[u][r]);
          }
      }
      // online softmax (per query = per lane): p = 2^(s - m), m the running maximum or up to 1
      // less (p <= 2, its scaled halves below 2^15), so that few blocks move what is summed; s
      // is scaled back in the same operation.  (The scale of the halves in the exponent as well,
      // 2^(s - m + 14), saves an instruction a value and rounds the exponent of the large p
      // to 2^-21: 1.2 to 2 times the error of the result.)
      uint32_t ph[4], pl[4];
      const float mblk = rows_max(mloc) * qinv;
      mtop = fmaxf(mtop, mblk);
      if (__any(mblk > mrun + 1.f)) {
        const float mnew = mtop;
        const float corr = __builtin_amdgcn_exp2f(mrun - mnew);
        lrun *= corr;
#pragma unroll
        for (int nd = 0; nd < ND; ++nd) O[nd] *= corr;
        mrun = mnew;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p0 = __builtin_amdgcn_exp2f(fmaf(sc[i / 2][i % 2 * 2], qinv, -mrun));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(sc[i / 2][i % 2 * 2 + 1], qinv, -mrun));
        lrun += p0;
        lrun += p1;
        split_pair(p0 * kPScale, p1 * kPScale, ph[i], pl[i]);  // clear of fp16 subnormals
      }
      const f16x8 phi = __builtin_bit_cast(f16x8, u32x4{ph[0], ph[1], ph[2], ph[3]});
      const f16x8 plo = __builtin_bit_cast(f16x8, u32x4{pl[0], pl[1], pl[2], pl[3]});
      // O^T += V^T · P^T
#pragma unroll
      for (int nd = 0; nd < ND; ++nd) {
        const uint32_t at = vat[nd] + (2 * buf + 1) * sizeof(lds[0][0]) + 32 * kb * ROWB;
        const s16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)at);
        const s16x4 y = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(at + 16 * ROWB));
        const f16x8 vf = __builtin_bit_cast(
            f16x8, s16x8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]});
        O[nd] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, phi, O[nd], 0, 0, 0);
        O[nd] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, plo, O[nd], 0, 0, 0);
      }
    }
  };
  for (int s = s0;;) {
    stage(std::integral_constant<int, 0>{}, s);
    if (++s >= s1) break;
    stage(std::integral_constant<int, 1>{}, s);
    if (++s >= s1) break;
  }
  {
    const float corr = __builtin_amdgcn_exp2f(mrun - mtop);
    lrun *= corr;
#pragma unroll
    for (int nd = 0; nd < ND; ++nd) O[nd] *= corr;
  }

  // the 4 lanes of a query hold partial sums over their keys
  lrun += __shfl_xor(lrun, 16, 64);
  lrun += __shfl_xor(lrun, 32, 64);
  const int qi = q0 + c;
  if (qi >= a.m) return;
  if (a.part_acc) {  // split partial state (unnormalised, log2 units)
    const size_t pidx = ((size_t)qi * a.H + h) * a.nsplit + split;
    float* o = a.part_acc + pidx * D + 4 * g;
#pragma unroll
    for (int nd = 0; nd < ND; ++nd)
      *reinterpret_cast<f32x4*>(o + 16 * nd) = O[nd] * (1.0f / kPScale);
    if (g == 0) *reinterpret_cast<float2*>(a.part_ml + pidx * 2) = float2{mtop, lrun};
  } else if (a.out16) {
    const float inv = 1.0f / (lrun + 1e-6f) * (1.0f / kPScale);
    _Float16* o = a.out16 + a_frag_off_f16(qi, h * D + 4 * g, a.H * D / 32);
#pragma unroll
    for (int nd = 0; nd < ND; ++nd)  // (16 dims further: 2 of a fragment's 4 groups of 8)
      *reinterpret_cast<ln_f16x4*>(o + nd / 2 * 512 + nd % 2 * 256) = ln_half4(O[nd] * inv);
  } else {
    const float inv = 1.0f / (lrun + 1e-6f) * (1.0f / kPScale);
    float* o = a.out + (size_t)qi * a.out_stride + h * D + 4 * g;
#pragma unroll
    for (int nd = 0; nd < ND; ++nd) *reinterpret_cast<f32x4*>(o + 16 * nd) = O[nd] * inv;
  }
}

template <int D, int TS>
hipError_t launch_prefill(const PaPrefillArgs& a, hipStream_t st) {
  const dim3 grid(a.H, (a.m + kTileQueries - 1) / kTileQueries, a.nsplit);
  // one pass of few workgroups: 64 keys a stage, half the barriers, as no others fill the waits
  // (16 heads of 128: 17 queries after 4,000 114 -> 100 us, 2,048 after 2,048 147 -> 134)
  const bool alone = a.nsplit == 1 && (long long)grid.x * grid.y <= 512;
  hipLaunchKernelGGL((alone ? pa_prefill_kernel<D, TS, 64> : pa_prefill_kernel<D, TS, stage_keys(D)>), grid,
                     dim3(64 * kWaves), 0, st, a);
  return hipGetLastError();
}

// The key range is cut into splits of `per` stages, the length for which the rounds of
// workgroups (4 per CU) times their length is least.  A split more counts as half a stage, a
// whole one where many rows with a long context before them write short splits, and more than 16,
// which pa_merge_row_kernel merges, as four besides.  No more than split_bound of them a query,
// and one of up to 64 keys (16 heads of 128, 64 queries: 7.4 us, in two splits 10.2).
// 32 queries a wave in place of 16 (16 heads of 128, with the merge; two waves a SIMD, of 32
// queries there can be no more): 2048 queries 72 -> 70 us, but those after 2048 more 120 -> 139,
// 1024 34 -> 36, 117 11 -> 14; heads of 64 2048 48 -> 60.
constexpr int kRound = 1024;
struct PrefillPlan {
  int nsplit, pps;
};
int split_bound(int H, int m) {
  const int nq = (m + kTileQueries - 1) / kTileQueries;
  return std::min(kRound / std::max(nq * H, 1) + 1, 128);
}
PrefillPlan prefill_plan(const pa_kv_view* kv, int p0, int m) {
  PrefillPlan p;
  const int H = kv->num_heads, kStageKeys = stage_keys(kv->head_dim);
  const int most = (p0 + m - 1) / kStageKeys + 1;
  const int bound = split_bound(H, m);
  // us by splits, heads of 128.  4 heads, 64 queries after 8,000: 12 28.5, 16 24.8, 20 26.2, 32
  // 25.5; 32 heads: 8 46.3, 16 43.7, 23 50.0.  32 heads, 128 queries after 3,000: 4 36.9, 8 35.7,
  // 14 41.9; 16 heads, 200 queries alone, whose rows have half of them: 3 12.9, 4 12.4.
  const double split = kv->head_dim == 128 && m * H >= 1500 && p0 >= m ? 1.0 : 0.5, many = 4.0;
  int best = most;
  double least = 1e30;
  for (int n = 1; n <= (p0 + m <= 64 ? 1 : std::min(bound, most)); ++n) {
    const int per = (most + n - 1) / n;
    long long wgs = 0;
    for (int q = 0; q < m; q += kTileQueries)
      wgs += ((p0 + std::min(q + kTileQueries, m) - 1) / kStageKeys + per) / per;
    const double cost = (double)((wgs * H + kRound - 1) / kRound) * per + split * (most + per - 1) / per +
                        (n > 16 ? many : 0.0);
    if (cost < least) {
      least = cost;
      best = per;
    }
  }
  p.nsplit = (most + best - 1) / best;
  p.pps = best * kStageKeys / kv->page_size;
  return p;
}

}  // namespace

bool pa_prefill_supported(const pa_kv_view* kv) {
  return kv && kv->kv_dtype == LLM_F16 && (kv->head_dim == 64 || kv->head_dim == 128) &&
         (kv->page_size == 16 || kv->page_size == 32);
}

bool pa_prefill_one_pass(const pa_kv_view* kv, int p0, int m) {
  return pa_prefill_supported(kv) && m > 0 && p0 >= 0 && prefill_plan(kv, p0, m).nsplit == 1;
}

// A plan has no more splits than split_bound and its stages allow, but fewer at one p0
// than at a shorter one (2048 queries x 16 heads: three at p0 0, one from p0 2048 on), so
// the size is of the most that any context up to this one takes.
size_t pa_prefill_ws_bytes(const pa_kv_view* kv, int p0, int m) {
  if (!pa_prefill_supported(kv) || m <= 0 || p0 < 0) return 0;
  const int most = (int)(((long long)p0 + m - 1) / stage_keys(kv->head_dim)) + 1;
  const int n = std::min(split_bound(kv->num_heads, m), most);
  if (n <= 1) return 0;
  return (size_t)m * kv->num_heads * n * (size_t)(kv->head_dim + 2) * sizeof(float);
}

int pa_prefill_internal(const pa_kv_view* kv, const float* q, int q_stride, float* out,
                        int out_stride, int row, int p0, int m, float sm_scale, void* workspace,
                        size_t workspace_bytes, hipStream_t st, const PaRowOutputs* rows) {
  LLM_REQUIRE(kv && q, "pa_prefill: NULL argument");
  if (!pa_prefill_supported(kv))
    return fail(LLM_ERR_UNSUPPORTED,
                "pa_prefill: fp16 pools with head_dim 64 or 128 and page_size 16 or 32 only");
  const int H = kv->num_heads, D = kv->head_dim, hid = H * D;
  LLM_REQUIRE(m >= 1 && p0 >= 0, "pa_prefill: need m >= 1 and p0 >= 0");
  LLM_REQUIRE(row >= 0 && row < kv->num_beams, "pa_prefill: row outside the page table");
  LLM_REQUIRE((long long)(p0 + m + kv->page_size - 1) / kv->page_size <= kv->max_tiles,
              "pa_prefill: positions past the page table's max_tiles");
  if (q_stride <= 0) q_stride = hid;
  if (out_stride <= 0) out_stride = hid;
  LLM_REQUIRE(q_stride >= hid && out_stride >= hid && q_stride % 4 == 0 && out_stride % 4 == 0,
              "pa_prefill: row strides must be >= H*D and multiples of 4");
  LLM_REQUIRE(reinterpret_cast<uintptr_t>(q) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0,
              "pa_prefill: q and out must be 16-byte aligned");
  const bool row_out = rows && (rows->q || rows->out16);
  PrefillPlan pl = prefill_plan(kv, p0, m);
  const size_t need = (size_t)m * H * pl.nsplit * (size_t)(D + 2) * sizeof(float);
  const bool split = pl.nsplit > 1 && workspace && workspace_bytes >= need &&
                     (out == nullptr || out_stride == hid) &&
                     (!row_out || rows->pack);  // the merge writes packed o_proj inputs
  const bool direct16 = !split && row_out && rows->out16 && !rows->q && !rows->keep_out && rows->pack;
  LLM_REQUIRE(out || (split && row_out) || direct16, "pa_prefill: out is NULL");
  PaPrefillArgs a{};
  a.q = q;
  a.q_stride = q_stride;
  a.out = out;
  a.out_stride = out_stride;
  a.k_pool = static_cast<const uint8_t*>(kv->k_pool);
  a.v_pool = static_cast<const uint8_t*>(kv->v_pool);
  a.page_stride = kv_view_page_stride(*kv);
  a.pt_row = kv->page_table + (size_t)row * H * kv->max_tiles;
  a.H = H;
  a.max_tiles = kv->max_tiles;
  a.num_pages = kv->num_pages;
  a.p0 = p0;
  a.m = m;
  a.qscale = sm_scale * kLog2e;
  if (split) {
    a.nsplit = pl.nsplit;
    a.pps = pl.pps;
    a.part_acc = static_cast<float*>(workspace);
    a.part_ml = a.part_acc + (size_t)m * H * pl.nsplit * D;
  } else {
    a.nsplit = 1;
    a.pps = kv->max_tiles;
    if (direct16) a.out16 = static_cast<_Float16*>(rows->out16);
  }
  hipError_t e;
  const int TS = kv->page_size;
  if (D == 64)
    e = TS == 16 ? launch_prefill<64, 16>(a, st) : launch_prefill<64, 32>(a, st);
  else
    e = TS == 16 ? launch_prefill<128, 16>(a, st) : launch_prefill<128, 32>(a, st);
  if (e != hipSuccess) return fail(LLM_ERR_HIP, std::string("pa_prefill launch: ") + hipGetErrorString(e));
  if (split)
    return pa_merge_rows_internal(a.part_acc, a.part_ml, (rows && !rows->keep_out) ? nullptr : out,
                                  rows, nullptr, p0, m, H, D, p0 + m, TS, pl.pps, pl.nsplit,
                                  kv->max_tiles, st);
  if (row_out && !direct16) {  // one pass: convert the fp32 rows into the o_proj input
    if (rows->q)
      LLM_HIP_RET(launch_quantize_rows(out, m, hid, rows->q, rows->inv_scale, st, rows->pack));
    if (rows->out16)
      LLM_HIP_RET(launch_to_f16(out, (size_t)m * hid, rows->out16, st, rows->pack ? hid : 0));
  }
  return LLM_OK;
}

}  // namespace llm

extern "C" size_t pa_prefill_workspace_bytes(const pa_kv_view* kv, int p0, int m) {
  return llm::pa_prefill_ws_bytes(kv, p0, m);
}

extern "C" int pa_prefill(const pa_kv_view* kv, const float* q, int q_stride, float* out,
                          int out_stride, int row, int p0, int m, float sm_scale, void* workspace,
                          size_t workspace_bytes, void* stream) {
  LLM_REQUIRE(out, "pa_prefill: out is NULL");
  return llm::pa_prefill_internal(kv, q, q_stride, out, out_stride, row, p0, m, sm_scale,
                                  workspace, workspace_bytes, llm::as_stream(stream));
}
