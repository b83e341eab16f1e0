// Paged decode attention for gfx950 (CDNA4): launch planning (split counts,
// forms), the split merges and the C entry points (pa_decode,
// pa_decode_grouped, pa_decode_plan).  The split kernel itself, and the design
// notes of the scan, are in pa_split.hpp; the tuning build's experiment
// kernels and A/B entry are in csrc/tune/pa_decode_tune.hip.
#include "pa_split.hpp"
#include "pa_tuning.hpp"

namespace llm {

// Split merge fused with the next consumer's input conversion: one workgroup
// per row b merges all H heads into an LDS row [H*D], then writes any of
//   out   fp32 [B][H*D]            (pa_decode's output)
//   q     int8 [B][H*D] + inv_scale[b]   (per-row quantisation of the o_proj
//         input, int8_quant.cpp:5-13,59-64 — replaces a quantize_rows launch)
//   out16 fp16 [B][H*D]            (fp16 o_proj input of the FP16 decoder)
struct PaMergeRowArgs {
  const float* part_acc;
  const float* part_ml;
  float* out;
  int8_t* q;
  float* inv_scale;
  _Float16* out16;
  const int32_t* context_lens;
  int B, H, D, T, TS, pps, nsplit, max_tiles;
  int pack;  // q / out16 in packed-A order (common.hpp a_frag_off_*)
  int ctx_p0;  // >= 0 and context_lens NULL: row b's context is ctx_p0 + b + 1 (prefill)
};

// One head's split merge (flash-decoding LSE combine) by one wave, DPL =
// output dims per lane (D / 64, at least 1).  The head's split weights (m, l),
// lane-parallel (lane holds splits lane and 64 + lane), and the partials of
// its first BATCH splits are loaded together: every address depends on the
// launch's arguments only (clamped to its nsplit), so they issue with the
// caller's context_lens load and a merge costs one memory round trip (splits
// beyond the batch: one more per 8).  The row's split count ns masks the
// values afterwards (splits past ns may hold stale bits).  Summation order
// s = 0, 1, ... (sequential) for L and for every output; split s's (l, w) come
// from lane s by readlane.  acc[j] * the returned 1 / L is the output at dim
// lane + 64 j; a head with no partial returns acc = 0.
template <int DPL, int BATCH>
struct MergeFirst {
  float m0, l0, m1, l1, v[BATCH][DPL];
  __device__ __forceinline__ void load(const float* ml, const float* pa, int nsplit, int D) {
    const int lane = lane_id(), nsl = max(nsplit - 1, 0);
    m0 = ml[2 * min(lane, nsl)], l0 = ml[2 * min(lane, nsl) + 1];
    m1 = ml[2 * min(64 + lane, nsl)], l1 = ml[2 * min(64 + lane, nsl) + 1];
#pragma unroll
    for (int s2 = 0; s2 < BATCH; ++s2)
#pragma unroll
      for (int j = 0; j < DPL; ++j)
        v[s2][j] = pa[(size_t)min(s2, nsl) * D + min(lane + 64 * j, D - 1)];
  }
};
template <int DPL, int BATCH>
__device__ __forceinline__ float merge_loaded(MergeFirst<DPL, BATCH>& f, const float* pa, int ns,
                                              int D, float (&acc)[DPL]) {
  const int lane = lane_id();
  float (&v)[BATCH][DPL] = f.v;
  const float m0 = lane < ns ? f.m0 : kNegSentinel;
  const float m1 = 64 + lane < ns ? f.m1 : kNegSentinel;
  const float l0 = lane < ns ? f.l0 : 0.f;
  const float l1 = 64 + lane < ns ? f.l1 : 0.f;
#pragma unroll
  for (int s2 = 0; s2 < BATCH; ++s2)
#pragma unroll
    for (int j = 0; j < DPL; ++j) v[s2][j] = s2 < ns ? v[s2][j] : 0.f;
#pragma unroll
  for (int j = 0; j < DPL; ++j) acc[j] = 0.f;
  const float M = ln_wave_max(fmaxf(m0, m1));
  if (ns <= 0 || M <= 0.5f * kNegSentinel) return 0.f;
  const float w0 = lane < ns ? __builtin_amdgcn_exp2f(m0 - M) : 0.f;
  const float w1 = 64 + lane < ns ? __builtin_amdgcn_exp2f(m1 - M) : 0.f;
  float L = 0.f;
#pragma unroll
  for (int s2 = 0; s2 < BATCH; ++s2)
    if (s2 < ns) {
      const float ls = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(l0), s2));
      const float ws = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w0), s2));
      L += ls * ws;
    }
  for (int s2 = BATCH; s2 < ns; ++s2) {
    const float ls = s2 < 64 ? __shfl(l0, s2, 64) : __shfl(l1, s2 - 64, 64);
    const float ws = s2 < 64 ? __shfl(w0, s2, 64) : __shfl(w1, s2 - 64, 64);
    L += ls * ws;
  }
#pragma unroll
  for (int s2 = 0; s2 < BATCH; ++s2) {
    const float ws = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w0), s2));  // 0 past ns
#pragma unroll
    for (int j = 0; j < DPL; ++j) acc[j] += v[s2][j] * ws;
  }
  for (int s0 = BATCH; s0 < ns; s0 += 8) {  // long split lists
#pragma unroll
    for (int j = 0; j < DPL; ++j) {
      const int d = lane + 64 * j;
      float u[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) u[k] = (s0 + k < ns && d < D) ? pa[(size_t)(s0 + k) * D + d] : 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int s2 = s0 + k;
        if (s2 < ns) {
          const float ws = s2 < 64 ? __shfl(w0, s2, 64) : __shfl(w1, s2 - 64, 64);
          acc[j] += u[k] * ws;
        }
      }
    }
  }
  return 1.0f / (L + 1e-6f);
}
template <int DPL, int BATCH>
__device__ __forceinline__ float merge_head(const float* ml, const float* pa, int nsplit, int ns,
                                            int D, float (&acc)[DPL]) {
  MergeFirst<DPL, BATCH> f;
  f.load(ml, pa, nsplit, D);
  return merge_loaded(f, pa, ns, D, acc);
}

// Split merge, fp32 output: one wave per (b, h), 4 per workgroup.  The first
// 16 splits' partials come in the first round trip (the 8-row C3 step merges
// 16 splits per head: 8.0 us per launch when the (m, l) and partial loads
// were issued split by split).
struct PaMergeArgs {
  const float* part_acc;
  const float* part_ml;
  float* out;
  const int32_t* context_lens;
  int B, H, D, T, TS, pps, nsplit, max_tiles;
};

// RAGGED: the split launch dealt its splits out by need (ragged_plan).
template <int DPL, bool RAGGED>
__global__ __launch_bounds__(256) void pa_merge_kernel(PaMergeArgs a) {
  const int lane = lane_id();
  const int bh = blockIdx.x * 4 + wave_id_uniform();
  if (bh >= a.B * a.H) return;
  const int b = bh / a.H;
  const float* ml = a.part_ml + (size_t)bh * a.nsplit * 2;
  const float* pa = a.part_acc + (size_t)bh * a.nsplit * a.D;
  MergeFirst<DPL, 16> first;
  first.load(ml, pa, a.nsplit, a.D);  // (of equal splits: they come while the plan is made)
  int ns;
  if constexpr (RAGGED) {
    const RaggedPlan p = ragged_plan(a.context_lens, a.B, a.T, a.TS, a.max_tiles, a.nsplit);
    const int ntiles = min((ragged_tokens(p, b) + a.TS - 1) >> __builtin_ctz(a.TS), a.max_tiles);
    if (p.unit) {
      const RowSplits r = ragged_find(p, a.B, [&](int row, int, int) { return row == b; });
      const size_t at = (size_t)r.first * a.H + (size_t)(bh % a.H) * r.count;
      ml = a.part_ml + at * 2;
      pa = a.part_acc + at * a.D;
      first.load(ml, pa, r.count, a.D);
      ns = (ntiles + p.unit - 1) / p.unit;
    } else {
      const int pps = row_pps(0, a.nsplit, ntiles);
      ns = min(a.nsplit, (ntiles + pps - 1) / pps);
    }
  } else {
    int Tb = a.context_lens ? a.context_lens[b] : a.T;
    Tb = min(max(Tb, 0), a.T);
    const int ntiles = min((Tb + a.TS - 1) / a.TS, a.max_tiles);
    const int pps = row_pps(a.pps, a.nsplit, ntiles);
    // pps < 0: every split holds a partial (beam launches: cost-balanced splits)
    ns = a.pps < 0 ? a.nsplit : min(a.nsplit, (ntiles + pps - 1) / pps);
  }
  float acc[DPL];
  const float inv = merge_loaded(first, pa, ns, a.D, acc);
  float* o = a.out + (size_t)bh * a.D;
#pragma unroll
  for (int j = 0; j < DPL; ++j) {
    const int d = lane + 64 * j;
    if (d < a.D) o[d] = acc[j] * inv;
  }
}

// Splits per first round trip of pa_merge_row_kernel's heads.
constexpr int kMergeBatch = 8;

template <int DPL>
__global__ __launch_bounds__(1024) void pa_merge_row_kernel(PaMergeRowArgs a) {
  extern __shared__ float row[];  // [H*D]
  __shared__ float sh[16];
  const int lane = lane_id();
  const int w = wave_id_uniform();
  const int nw = blockDim.x >> 6;
  const int b = blockIdx.x;
  const int hid = a.H * a.D;
  int Tb = a.context_lens ? a.context_lens[b] : a.ctx_p0 >= 0 ? a.ctx_p0 + b + 1 : a.T;
  Tb = min(max(Tb, 0), a.T);
  const int ntiles = min((Tb + a.TS - 1) / a.TS, a.max_tiles);
  const int pps = row_pps(a.pps, a.nsplit, ntiles);
  // pps < 0: every split holds a partial (beam launches: cost-balanced splits)
  const int ns = a.pps < 0 ? a.nsplit : min(a.nsplit, (ntiles + pps - 1) / pps);
  for (int h = w; h < a.H; h += nw) {
    const size_t bh = (size_t)b * a.H + h;
    float acc[DPL];
    const float inv = merge_head<DPL, kMergeBatch>(a.part_ml + bh * a.nsplit * 2,
                                                   a.part_acc + bh * a.nsplit * a.D, a.nsplit, ns,
                                                   a.D, acc);
    float* dst = row + h * a.D;
#pragma unroll
    for (int j = 0; j < DPL; ++j) {
      const int d = lane + 64 * j;
      if (d < a.D) dst[d] = acc[j] * inv;
    }
  }
  __syncthreads();
  float am = 0.f;
  // packed int8 o_proj input only (the decode step): 4 values per thread, one
  // dword store each (4 consecutive k are 4 consecutive bytes of a fragment)
  const bool quad = a.q && a.pack && !a.out && !a.out16 && hid % 64 == 0;
  if (quad) {
    for (int i4 = threadIdx.x; i4 < hid / 4; i4 += blockDim.x) {
      const f32x4 v = reinterpret_cast<const f32x4*>(row)[i4];
      am = fmaxf(am, fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
    }
  } else {
    for (int i = threadIdx.x; i < hid; i += blockDim.x) {
      const float v = row[i];
      am = fmaxf(am, fabsf(v));
      if (a.out) a.out[(size_t)b * hid + i] = v;
      if (a.out16)
        a.out16[a.pack ? a_frag_off_f16(b, i, hid >> 5) : (size_t)b * hid + i] = (_Float16)v;
    }
  }
  if (!a.q) return;
  am = ln_wave_max(am);
  if (lane == 0) sh[w] = am;
  __syncthreads();
  am = sh[0];
  for (int i = 1; i < nw; ++i) am = fmaxf(am, sh[i]);
  const float scale = 127.f / (am + 1e-6f);
  if (quad) {
    for (int i4 = threadIdx.x; i4 < hid / 4; i4 += blockDim.x)
      *reinterpret_cast<uint32_t*>(a.q + a_frag_off_i8(b, 4 * i4, hid >> 6)) =
          ln_quant4(reinterpret_cast<const f32x4*>(row)[i4], scale);
  } else {
    for (int i = threadIdx.x; i < hid; i += blockDim.x) {
      float y = roundf(__fmul_rn(row[i], scale));
      y = fminf(fmaxf(y, -128.f), 127.f);
      a.q[a.pack ? a_frag_off_i8(b, i, hid >> 6) : (size_t)b * hid + i] = (int8_t)(int)y;
    }
  }
  if (threadIdx.x == 0) a.inv_scale[b] = 1.0f / scale;
}

// The same for a prompt's rows: many of them, few splits each.  A thread takes four
// neighbouring values of QPT quads, of every split one 16-byte load, and keeps them to the
// quantisation; it works out its head's weights itself, two to four exponentials in most
// prompts.  Bound by the partials' bytes (2048 rows of 16 x 128, three splits at most, int8
// out: 22 us by a wave a head and values through LDS, all splits' places read, now 10).
template <int QPT>
__global__ __launch_bounds__(256) void pa_merge_prompt_kernel(PaMergeRowArgs a) {
  __shared__ float sh[4];
  const int b = a.pack ? packed_row(blockIdx.x, gridDim.x) : blockIdx.x;
  const int hid = a.H * a.D, step = blockDim.x;
  const int ntiles = min((min(a.ctx_p0 + b + 1, a.T) + a.TS - 1) / a.TS, a.max_tiles);
  const int ns = min(a.nsplit, (ntiles + a.pps - 1) / a.pps);
  f32x4 v[QPT];
  const auto merge = [&](auto N) {  // N: the row's splits, 0: more than the cases below
    constexpr int AT_ONCE = decltype(N)::value ? decltype(N)::value : 4;
#pragma unroll
    for (int i = 0; i < QPT; ++i) {
      const int at = 4 * (threadIdx.x + i * step), h = at / a.D;
      v[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (at >= hid) continue;
      const size_t first = ((size_t)b * a.H + h) * a.nsplit;
      const float2* ml = reinterpret_cast<const float2*>(a.part_ml) + first;
      const float* pa = a.part_acc + first * a.D + at % a.D;
      float M = kNegSentinel, L = 0.f;
      if constexpr (decltype(N)::value == 0)
#pragma unroll 4
        for (int s = AT_ONCE; s < ns; ++s) M = fmaxf(M, ml[s].x);
      f32x4 x[AT_ONCE];
      float2 st[AT_ONCE];
#pragma unroll
      for (int s = 0; s < AT_ONCE; ++s) {
        x[s] = *reinterpret_cast<const f32x4*>(pa + (size_t)s * a.D);
        st[s] = ml[s];
      }
#pragma unroll
      for (int s = 0; s < AT_ONCE; ++s) M = fmaxf(M, st[s].x);
#pragma unroll
      for (int s = 0; s < AT_ONCE; ++s) {
        const float w = __builtin_amdgcn_exp2f(st[s].x - M);
        L += st[s].y * w;
        v[i] += x[s] * w;
      }
      if constexpr (decltype(N)::value == 0)
#pragma unroll 4
        for (int s = AT_ONCE; s < ns; ++s) {
          const float w = __builtin_amdgcn_exp2f(ml[s].x - M);
          L += ml[s].y * w;
          v[i] += *reinterpret_cast<const f32x4*>(pa + (size_t)s * a.D) * w;
        }
      v[i] *= M <= 0.5f * kNegSentinel ? 0.f : 1.0f / (L + 1e-6f);
    }
  };
  switch (ns) {
    case 1: merge(std::integral_constant<int, 1>{}); break;
    case 2: merge(std::integral_constant<int, 2>{}); break;
    case 3: merge(std::integral_constant<int, 3>{}); break;
    case 4: merge(std::integral_constant<int, 4>{}); break;
    default: merge(std::integral_constant<int, 0>{});
  }
  float am = 0.f;
#pragma unroll
  for (int i = 0; i < QPT; ++i) {
    const int at = 4 * (threadIdx.x + i * step);
    if (at >= hid) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) am = fmaxf(am, fabsf(v[i][e]));
    if (a.out) *reinterpret_cast<f32x4*>(a.out + (size_t)b * hid + at) = v[i];
    if (a.out16)
      *reinterpret_cast<ln_f16x4*>(
          a.out16 + (a.pack ? a_frag_off_f16(b, at, hid >> 5) : (size_t)b * hid + at)) = ln_half4(v[i]);
  }
  if (!a.q) return;
  am = ln_wave_max(am);
  if (lane_id() == 0) sh[wave_id_uniform()] = am;
  __syncthreads();
  am = sh[0];
  for (int i = 1; i < step >> 6; ++i) am = fmaxf(am, sh[i]);
  const float scale = 127.f / (am + 1e-6f);
#pragma unroll
  for (int i = 0; i < QPT; ++i) {
    const int at = 4 * (threadIdx.x + i * step);
    if (at < hid)
      *reinterpret_cast<uint32_t*>(
          a.q + (a.pack ? a_frag_off_i8(b, at, hid >> 6) : (size_t)b * hid + at)) = ln_quant4(v[i], scale);
  }
  if (threadIdx.x == 0) a.inv_scale[b] = 1.0f / scale;
}

namespace {

constexpr int kMinPps = 8;
constexpr int kMaxWavesPerCu = 32;  // 8 per SIMD x 4 SIMDs (gfx950)

// Resident waves of the whole chip for one split-kernel instantiation
// (occupancy query x CU count), cached.  Fallback: 256 CUs x 3 waves/SIMD.
// Register stages of an instantiation: pages above 8 KiB hold a whole stage
// per page already (two would not fit the VGPR file).
template <int D, int TS, int KVT>
constexpr int split_stages() {
  return TS * D * kv_elem_bytes<KVT>() > 8192 ? 1 : 2;
}

template <int D, int TS, bool DIRECT, int KVT>
long long resident_waves() {
  static long long cached = 0;
  if (cached) return cached;
  int dev = 0, cus = 0, blocks = 0;
  constexpr int ST = split_stages<D, TS, KVT>();
  if (hipGetDevice(&dev) == hipSuccess &&
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
      hipOccupancyMaxActiveBlocksPerMultiprocessor(
          &blocks, pa_split_kernel<D, TS, DIRECT, 16384, kKvLoadAux, ST, 0, false, false, KVT>, 256,
          0) == hipSuccess &&
      cus > 0 && blocks > 0) {
    cached = (long long)cus * blocks * 4;
  } else {
    (void)hipGetLastError();
    cached = 256LL * 4 * 3;
  }
  return cached;
}

}  // namespace

// The FP16 decoder's o_proj fused into the workgroup merge (decoder.cpp
// oproj_fusable); LLM_OPROJ_FUSE=0 (tuning build) restores the o_proj GEMM.
bool oproj_fuse_on() { return pa_tuning().oproj_fuse; }
bool beam_steal_on() { return pa_tuning().beam_steal; }

namespace {

// The experiment forms of beam-group launches (pa_beam4_kernel,
// pa_beam_mfma_kernel, the steal form, ...) exist only in the tuning build
// (csrc/tune/pa_decode_tune.hip, switched by pa_tuning.hpp).  All measured
// slower than the LDS-staged BEAM form of pa_split_kernel (C4 launch with
// merge: beam4 69.2 us at 16 splits, 74.2 with two pages per register stage,
// 82.3 at 12 splits, against 67.6 us; MFMA 69.8 vs 60.8 us; steal 76-92 vs
// 65.3 us).

template <int D, int TS, int KVT>
hipError_t launch_split(const PaSplitArgs& a, bool direct, hipStream_t st, bool* beam) {
  const int waves = ((a.B + a.group - 1) / a.group) * a.group * a.H * a.nsplit;
  const dim3 grid((waves + 3) / 4), block(256);
  if constexpr (KVT != LLM_F16) {
    // other KV element types: the standard schedule (no beam-prefetch form)
    constexpr int ST = split_stages<D, TS, KVT>();
    if (a.ragged)
      hipLaunchKernelGGL((pa_split_kernel<D, TS, false, 16384, kKvLoadAux, ST, 0, false, false, KVT,
                                          true, false, false, 0, false, false, false, true>),
                         grid, block, 0, st, a);
    else if (direct)
      hipLaunchKernelGGL((pa_split_kernel<D, TS, true, 16384, kKvLoadAux, ST, 0, false, false, KVT>),
                         grid, block, 0, st, a);
    else
      hipLaunchKernelGGL((pa_split_kernel<D, TS, false, 16384, kKvLoadAux, ST, 0, false, false, KVT>),
                         grid, block, 0, st, a);
    return hipGetLastError();
  }
  constexpr int ST = split_stages<D, TS, LLM_F16>();
  if (a.wgm) {  // pa_decode_internal: group 1, 2..8 splits, not direct
    if constexpr (D <= kOprojMaxD) {
      if (a.o_acc) {
        hipLaunchKernelGGL((pa_split_kernel<D, TS, false, 16384, kKvLoadAux, ST, 0, false, false,
                                            LLM_F16, true, true, true>),
                           dim3(a.B * a.H), dim3(64 * a.nsplit), 0, st, a);
        return hipGetLastError();
      }
    }
    hipLaunchKernelGGL((pa_split_kernel<D, TS, false, 16384, kKvLoadAux, ST, 0, false, false,
                                        LLM_F16, true, true>),
                       dim3(a.B * a.H), dim3(64 * a.nsplit), 0, st, a);
    return hipGetLastError();
  }
  if (a.group == 4 && !direct && ST == 2) {
    // 8 KiB register stages: 112 VGPRs, 4 waves per SIMD.  The 16 KiB form
    // (179 VGPRs, 2 waves) spent 27 % of its wave time in issue stalls and
    // 20 % parked (SQ PMC, scripts/gpu_sq_pmc.sh); same-box A/B of the C4
    // launch: 72-74 vs 76 us (scripts/ab_attention_lib.py, -DLLM_BEAM_CHUNK=)
#ifndef LLM_BEAM_CHUNK
#define LLM_BEAM_CHUNK 8192
#define LLM_BEAM_WAVES 0
#endif
    hipError_t te;
    if (tune_launch_form(a, D, TS, grid, st, &te)) {  // tuning build: an experiment form
      *beam = true;
      return te;
    }
    hipLaunchKernelGGL((pa_split_kernel<D, TS, false, LLM_BEAM_CHUNK, kKvLoadAux, 2, LLM_BEAM_WAVES,
                                        false, true, LLM_F16, true, false, false, 0, false, true, true>),
                       grid, block, 0, st, a);
    *beam = true;
  } else if (a.ragged) {
    hipLaunchKernelGGL((pa_split_kernel<D, TS, false, 16384, kKvLoadAux, ST, 0, false, false, LLM_F16,
                                        true, false, false, 0, false, false, false, true>),
                       grid, block, 0, st, a);
  } else if (direct) {
    hipLaunchKernelGGL((pa_split_kernel<D, TS, true, 16384, kKvLoadAux, ST>), grid, block, 0, st, a);
  } else {
    hipLaunchKernelGGL((pa_split_kernel<D, TS, false, 16384, kKvLoadAux, ST>), grid, block, 0, st, a);
  }
  return hipGetLastError();
}

template <int D, int KVT>
hipError_t dispatch_ts(const PaSplitArgs& a, int TS, bool direct, hipStream_t st, bool* beam) {
  constexpr int ES = kv_elem_bytes<KVT>();
  if (TS == 16) {
    if constexpr (kv_shape_ok(D, 16, ES)) return launch_split<D, 16, KVT>(a, direct, st, beam);
  } else if (TS == 32) {
    if constexpr (kv_shape_ok(D, 32, ES)) return launch_split<D, 32, KVT>(a, direct, st, beam);
  }
  return hipErrorInvalidValue;
}

template <int D>
hipError_t dispatch_kvt(const PaSplitArgs& a, int kvt, int TS, bool direct, hipStream_t st,
                        bool* beam) {
  switch (kvt) {
    case LLM_F16: return dispatch_ts<D, LLM_F16>(a, TS, direct, st, beam);
    case LLM_BF16: return dispatch_ts<D, LLM_BF16>(a, TS, direct, st, beam);
    case LLM_F32: return dispatch_ts<D, LLM_F32>(a, TS, direct, st, beam);
    case LLM_I8: return dispatch_ts<D, LLM_I8>(a, TS, direct, st, beam);
    default: return hipErrorInvalidValue;
  }
}

int kv_dtype_bytes(int kvt) {
  switch (kvt) {
    case LLM_F16: case LLM_BF16: return 2;
    case LLM_F32: return 4;
    case LLM_I8: return 1;
    default: return 0;
  }
}

bool supported(int D, int TS, int kvt) {
  const int es = kv_dtype_bytes(kvt);
  return es > 0 && (D == 32 || D == 64 || D == 128 || D == 256) && (TS == 16 || TS == 32) &&
         kv_shape_ok(D, TS, es);
}

// Upper bound of the split count of any launch over rows of <= ntiles tiles
// (workspace sizing; host-only, no device query).
long long max_nsplit(int B, int H, int ntiles) {
  ntiles = std::max(ntiles, 1);
  const long long bh = std::max(1LL, (long long)B * H);
  const long long cap = 256LL * kMaxWavesPerCu;  // largest resident-wave count
  const long long lo = (ntiles + kMaxPps - 1) / kMaxPps;
  return std::min<long long>(
      kMaxSplits,
      std::max(lo, std::min<long long>((ntiles + kMinPps - 1) / kMinPps, lo + (cap + bh - 1) / bh + 1)));
}

// Splits per (b, h): the smallest NS that is a whole number of resident-wave
// rounds (B*H*NS ~ k * resident) with splits of <= kMaxPps pages, so every wave
// carries the same page count and the last round is not a ragged tail; never
// below kMinPps pages per split.  Small launches, where a full round would
// leave each wave under kShortPps pages, use fewer, longer splits instead,
// as long as at least kMinLaunchWaves waves remain: a split's fixed cost
// (page ids, q, its partial and its share of the merge) outweighs an idle
// part of the chip there.  Measured (scripts/sweep_attention_pps.py), round
// rule -> this rule: C2 (16 x 12 heads, 2048 tokens) 25.1 -> 21.3 us;
// 64 x 12 x 2048: 72.7 -> 66.6 us; 8 x 16 x 4096: 49.3 -> 46.1 us;
// 1 x 16 x 8192: 32.8 -> 26.4 us; 4 x 12 x 1024 unchanged (9.9 us).
constexpr int kShortPps = 32;
constexpr long long kMinLaunchWaves = 512;
// Workgroup-merge launches (PaSplitArgs::wgm) have no merge launch to feed, so
// their splits stay long: C2 (130 tiles) 3 splits, not 5.  Same-box C2 sweep
// (scripts/gpu_wgm_splits.sh, forced splits 2 / 3 / 4 / 5 / 6 / 8):
// 27.4-28.0k / 29.6-30.1k / 29.1-29.2k / 28.4k / 28.6-28.9k / 28.2-29.0k tok/s.
constexpr int kWgmShortPps = 64;
int choose_nsplit(int B, int H, int ntiles, int pps_fixed, long long resident,
                  int short_pps = kShortPps) {
  ntiles = std::max(ntiles, 1);
  if (pps_fixed > 0) {
    const int pps = std::min(pps_fixed, kMaxPps);
    return (ntiles + pps - 1) / pps;
  }
  const long long bh = std::max(1LL, (long long)B * H);
  const long long lo = (ntiles + kMaxPps - 1) / kMaxPps;
  long long ns = lo;
  for (long long k = 1; k <= 64; ++k) {
    const long long cand = (k * resident + bh - 1) / bh;
    if (cand >= lo) { ns = cand; break; }
  }
  ns = std::min<long long>(ns, std::max(1, (ntiles + kMinPps - 1) / kMinPps));
  if ((ntiles + ns - 1) / ns < short_pps)
    ns = std::min(ns, std::max<long long>((ntiles + short_pps - 1) / short_pps,
                                          (kMinLaunchWaves + bh - 1) / bh));
  ns = std::max(ns, lo);
  return (int)std::min(ns, max_nsplit(B, H, ntiles));
}

// Splits of up to 32 pairs of row and head whose whole rounds of waves make more than a workgroup merges: a merge of
// few parts costs less (steps are short beside it where T, the longest sequence held, is not filled), more waves read
// long rows sooner.  4 layers, T (held), us by 16 / 24 / 32 / 48 / 64 splits and by whole rounds (how many), alone and (in
// turns, three decoders' steps that overlap):
//  * 1 x 4 of 64 T 14,336 (12,902) 163 / 153 / 150 / 154 / 161, rounds 182 (112) (67 / 63 / 61 / 61 / 63, 69); T 20,480
//    (18,432) 190 / 171 / 164 / 163 / 166, 197 (128) (78 / 71 / 68 / 66 / 66, 74);
//  * 1 x 12 of 64 T 4,500 (4,050) 155 / 158 / 161, 161 (36); T 7,144 (6,429) 170 / 168 / 171, 177 (43) (76 / 74 / 74, 75); T
//    9,600 (1,440) 145 / 147 / 153, 153 (43), (8,640) 180 / 173 / 176, 182 (82 / 78 / 77, 79); T 32,000 (28,800) 273 / 238 / 228 / 224,
//    235 (63) (140 / 123 / 116 / 111, 113); 1 x 8 T 20,480 (18,432) 211 / 191 / 185 / 184, 186 (64) (95 / 85 / 81 / 80, 79);
//  * 1 x 8 of 128 T 7,144 (1,071) 157 / 165 / 164 / 177, 178 (56), (6,429) 206 / 198 / 197 / 208, 213 (104 / 99 / 97 / 99, 100): 16 as a step
//    alone decides; T 9,600 (8,640) 224 / 211 / 208 / 215, 228 (64) (116 / 109 / 103 / 104, 106); T 14,336 (12,902) 263 / 236 /
//    228 / 232, 241 (142 / 126 / 119 / 115, 115); T 32,000 (28,800) 400 / 332 / 303 / 285, 284 (233 / 195 / 174 / 158, 152);
//  * 1 x 16 of 128 T 7,144 (1,071) 249 / 257, 257 (32) (138 / 140, 140), (6,429) 300 / 292, 295 (174 / 166, 165); T 12,144 (6,000)
//    294 / 289, 292 (170 / 163, 162), (1,821) by 24 264, 269 (143, 145), (10,929) 325, 320 (194, 186); T 14,336 (12,902) 362 / 336, 329 (222 / 204, 197); T 32,000 (28,800) 508 / 443 / 416 / 420, 446 (63) (333 /
//    297 / 283 / 273, 283).
//  * 17 pairs and more: 2 x 16 of 128 T 14,336 (8,192) 331 / 329, 338 (28) (217 / 211, 213); of 64 16 (T 20,480 (18,500) 258, 293 (40)).
int few_pairs_splits(long long bh, int D, int tiles, int nsplit) {
  const bool wide = D > 64;
  int n;
  if (bh > 16) n = wide && tiles > 560 ? 24 : 16;
  else if (tiles <= (wide ? (bh <= 8 ? 512 : 320) : (bh <= 4 ? 900 : 416))) n = 16;
  else if (tiles <= (wide ? (bh <= 8 ? 0 : 760) : 624)) n = 24;
  else if (wide && tiles <= 640) n = 32;
  else n = bh > 8 || tiles <= (wide ? 960 : 1248) ? 48 : 64;
  return std::min(n, nsplit);
}

// The FP16 decoder's attention and what its o_proj is: `nsplit` splits that a workgroup merges and
// multiplies by the head's rows of W_o (fused), splits and a merge launch, or one split, both with an
// o_proj GEMM after them.  `nsplit` in: what the rules above give; their fused form (2..8) may become any
// of the three, the others stay what they are (the fused sums have a range, the GEMM's none).
//
// Lines from steps of 2 to 3 layers of one decoder alone, rows x heads of D, the longest sequence held T, sequences
// that fill it unless said; us a step, before -> now (with them the best fixed choice).  "In turns": steps of three
// decoders of 4 layers that overlap.
//  * a fused workgroup reads D x hidden of W_o whatever its row's length, and its 4 waves (8 where that
//    is 256 KB or more: two rounds of columns for 8) fit the chip 512 (256) times.  Past that one split of up
//    to 128 pages: 64 x 16 of 128 T 720 476 -> 422, 48 x 12 of 64 T 720 194 -> 182, T 1,920 286 -> 261; below
//    it where contexts are short for their W_o: 16 x 16 of 128 T 133 225 -> 196, 1 x 16 of 128 195 -> 176,
//    but T 320 235 -> 223 by 8 waves, one split 219 (22 pages: the line).
//  * few pairs of long rows leave CUs idle, so splits over more workgroups: 4 x 16 of 128 T 1,920 241 ->
//    216, T 8,192 with 2,048 held 246 -> 222; 16 x 4 of 64 T 8,300 180 -> 151 by 12.  Heads of 64 with 17 to
//    64 pairs do so past 8,192 tokens, as a step's sequences may be far shorter than T (T 7,144 with 1,000
//    held, in turns: 4 x 16 of 64 by 4 waves 120, 12 splits 134), more than 64 pairs of 128 never (in turns, 8 x 16
//    T 7,144 with 1,000 held and more 220, 8 splits 228).  As many as
//    few_pairs_splits says, and 12 from 33 pairs on, not 16 to 40 (in turns 4 x 12 of 64 T 14,336 with 8,192 119 -> 114, 16 x 4
//    121 -> 115, 3 x 16 with 9,000 141 -> 134; 4 x 16 T 20,480 with 18,500 259 -> 238, of 128 505 -> 491; 3 x 16 of 128 there
//    406 -> 416, alone 548 -> 517).
//    64 pairs of 128, whose W_o a fused workgroup's waves also read, gain alone and pay in turns, where the other decoders
//    fill the CUs that one leaves idle, until their rows are long: 4 layers of 4 x 16, fused -> apart, alone and (in turns): T 1,920
//    with 300 held 239 -> 235 (135.5 -> 141.2), 1,500 288 -> 265 (157.7 -> 163.7); T 7,144 with 1,000 267 -> 255
//    (147.5 -> 155.4), 3,000 343 -> 296 (190.0 -> 192.1), 6,000 455 -> 351 (260.5 -> 248.9).  A step alone decides.
//    Less than 512 KB of W_o is no load to part with for short rows: 8 x 8 of 128 T 800 with 120 held 139 -> 149 (74.9 -> 78.1), T
//    1,920 with 288 145 -> 154 (77.5 -> 81.6), 1,728 199 -> 182 (100.8 -> 106.5), T 4,500 with 675 160 -> 165 (84.3 -> 87.7),
//    4,050 285 -> 227 (142 -> 149); 4 x 8 T 800 with 120 134 -> 144 (71 -> 74): apart past 4,096 tokens there.
//    9 to 12 splits of 33 to 64 pairs stay (4 x 12 of 128 T 4,000 with 3,600 held 261, by 8 270; 600 held 212, 210).
//  * else 4 waves: 16 x 12 of 64 T 8,192 with 2,048 held 162 -> 156 (by 8), T 2,720 167 -> 161 (by 3).
//    Up to 128 pairs as before (in turns, 5 x 16 of 64 T 6,644 by 7 101.5, by 4 111.0;
//    10 x 12 T 7,644 118.5, 125.9; 12 x 16 by 8 157.1, by 4 155.4), and up to 32 KB of W_o, which one wave's
//    columns cover (64 x 4 of 64 T 1,920 175; by 4 179; in turns 16 x 4 T 6,744 with 600 held and more, by 8 76.4,
//    by 4 85.5).
struct F16Form {
  int nsplit;
  bool fused;
};
F16Form f16_step_form(long long bh, int D, int hidden, int tiles, int nsplit) {
  const long long kb = (long long)D * hidden * 2 / 1024;  // of W_o a head
  const bool fits = nsplit >= 2 && nsplit <= kWgmMaxSplits;
  const long long one = kb >= 512 ? std::max<long long>(bh > 256 ? 80 : bh > 128 ? 22 : 0, 13 * kb / 512)
                        : kb >= 256 ? (bh > 256 ? 20 : 0)
                                    : (bh > 400 ? 25 : bh > 256 ? 10 : 0);
  if (fits && tiles <= kMaxPps && (bh > 512 || tiles <= one)) return {1, false};
  const bool apart = D > 64 ? tiles > (bh > 64 ? INT_MAX : fits && kb < 512 ? 256 : 45)
                            : tiles > (bh <= 16 ? 110 : bh <= 64 ? 512 : INT_MAX);
  if (nsplit > 1 && apart) {
    int n = bh <= 32 ? (fits ? 8 : few_pairs_splits(bh, D, tiles, nsplit)) : D > 64 && fits && tiles <= 256 ? 8 : 12;
    if (!fits) n = std::min(n, nsplit);
    if ((long long)n * kMaxPps >= tiles) return {n, false};
  }
  if (!fits) return {nsplit, false};
  if (tiles <= 4 * kMaxPps && bh > (kb >= 512 ? 400 : 512) && kb >= 256) return {4, false};
  int n = kb >= 512 || (kb >= 256 && bh <= 256) ? 8 : kb <= 32 || bh <= 128 ? nsplit : 4;
  while (n < kWgmMaxSplits && (long long)n * kMaxPps < tiles) n *= 2;
  return {std::min(n, kWgmMaxSplits), true};
}

// fp32 rows that the o_proj quantises (hidden up to 2,048): splits that a workgroup merges (2..8) or a
// merge launch does.  `nsplit` in: what the rules above give; half_round's stay.  Whole rounds of waves
// make 9 to 95 splits of few pairs, most of them empty where the sequences are short of the longest held,
// T, and merged in odd batches.  Steps of 2 layers of one decoder alone, rows x heads of D, T (held), us, before ->
// now; "in turns" as above:
//  * few_pairs_splits up to 32 pairs: 1 x 4 of 64 T 7,144 (1,000) 68 -> 62, T 12,144 (6,000) 93 -> 75; 1 x 16 of 128 T 4,520
//    (4,500) 144 -> 143; from 33 pairs on 12 in place of 9 to 12, 16 in place of more than 16: 16 x 4 of 64 T 4,520
//    (4,500) 97 -> 95; 4 layers in turns, 4 x 12 T 32,000 (29,000) 275 -> 249, 3 x 16 of 128 554 -> 525;
//  * 8 up to 128: 8 x 16 of 128 T 4,520 (4,500) 243 -> 220, 32 x 4 of 64 146 -> 133; past that merged in the
//    workgroup: 16 x 12 of 64 T 8,192 (2,048) 140 -> 133, T 12,144 (6,000) 217 -> 194;
//  * 13 to 16 of 33 to 128 pairs stay: in turns, 16 x 4 of 64 T 6,744 14 splits 83.1, 16
//    86.0; 32 x 4 T 7,144 14 splits 120.5, 8 125.6; 8 x 16 of 128 209.8, 212.7 (alone the same), where 25 x 4 T 10,144
//    20 splits 147.9, 8 140.6; 3 x 16 T 12,144 24 splits 129.0, 16 122.3;
//  * 257 to 512 pairs of 64: 4 in place of 8 (32 x 12 T 8,192 (2,048) 186 -> 177; 64 x 12 275 -> 257, but in
//    turns 307 -> 313), and past 512 pairs one for up to 128 pages (64 x 12 T 720 163 -> 157, 64 x 16 of 128 303 -> 299).
//    Two and a half waves a CU of heads of 128 end unevenly where they are long: 4 layers of 40 x 16, T 1,920 (1,728) 622 ->
//    609, in turns 499 -> 543, so below three a CU up to 720 tokens.
struct F32Form {
  int nsplit;
  bool wgm;
};
F32Form f32_step_form(long long bh, int D, int tiles, int nsplit) {
  const bool wgm = nsplit <= kWgmMaxSplits;
  if (nsplit >= 2 && bh > 512 && tiles <= (D > 64 && bh < 768 ? 45 : kMaxPps)) return {1, false};
  if (wgm) return {D <= 64 && bh > 256 && bh <= 512 && tiles <= 4 * kMaxPps ? std::min(nsplit, 4) : nsplit, true};
  if (bh > 32 && bh <= 128 && nsplit > 12 && nsplit <= 16) return {nsplit, wgm};
  const int n = bh <= 32 ? few_pairs_splits(bh, D, tiles, nsplit) : bh <= 64 ? (nsplit > 16 ? 16 : 12) : 8;
  if ((long long)n * kMaxPps < tiles) return {nsplit, false};
  return {n, bh > 128};
}

template <int D, int TS, int KVT>
long long resident_for() {
  if constexpr (kv_shape_ok(D, TS, kv_elem_bytes<KVT>()))
    return resident_waves<D, TS, false, KVT>();
  return 256LL * 4 * 3;
}

template <int D>
long long resident_for_kvt(int TS, int kvt) {
  auto by_ts = [&](auto k) -> long long {
    constexpr int K = decltype(k)::value;
    return TS == 16 ? resident_for<D, 16, K>() : resident_for<D, 32, K>();
  };
  switch (kvt) {
    case LLM_BF16: return by_ts(std::integral_constant<int, LLM_BF16>{});
    case LLM_F32: return by_ts(std::integral_constant<int, LLM_F32>{});
    case LLM_I8: return by_ts(std::integral_constant<int, LLM_I8>{});
    default: return by_ts(std::integral_constant<int, LLM_F16>{});
  }
}

long long resident_waves_for(int D, int TS, int kvt) {
  auto pick = [&](auto d) -> long long {
    constexpr int DD = decltype(d)::value;
    return resident_for_kvt<DD>(TS, kvt);
  };
  switch (D) {
    case 32: return pick(std::integral_constant<int, 32>{});
    case 64: return pick(std::integral_constant<int, 64>{});
    case 128: return pick(std::integral_constant<int, 128>{});
    default: return pick(std::integral_constant<int, 256>{});
  }
}

}  // namespace

int pa_pages_per_split(int B, int H, int T, int TS, int max_tiles) {
  const int ntiles = std::max(1, std::min((T + TS - 1) / TS, max_tiles));
  const int ns = choose_nsplit(B, H, ntiles, 0, 256LL * 4 * 3);
  return (ntiles + ns - 1) / ns;
}

}  // namespace llm

using namespace llm;

extern "C" int pa_decode_pages_per_split(int B, int H, int T, int page_size, int max_tiles) {
  if (B < 0 || H <= 0 || T < 0 || page_size <= 0 || max_tiles <= 0) return -1;
  return pa_pages_per_split(B, H, T, page_size, max_tiles);
}

extern "C" size_t pa_decode_workspace_bytes(int B, int H, int D, int max_tiles,
                                            int pages_per_split) {
  if (B <= 0 || H <= 0 || D <= 0 || max_tiles <= 0) return 0;
  const size_t nsplit = pages_per_split > 0
                            ? (size_t)choose_nsplit(B, H, max_tiles, pages_per_split, 0)
                            : (size_t)max_nsplit(B, H, max_tiles);
  return (size_t)B * H * nsplit * (size_t)(D + 2) * sizeof(float);
}

int llm::pa_merge_splits_internal(const float* part_acc, const float* part_ml, float* out,
                                  const int32_t* context_lens, int B, int H, int D, int T, int TS,
                                  int pps, int nsplit, int max_tiles, hipStream_t st,
                                  bool ragged) {
  PaMergeArgs mg{part_acc, part_ml, out, context_lens, B, H, D, T, TS, pps, nsplit, max_tiles};
  const auto launch = [&](auto r) {
    constexpr bool R = decltype(r)::value;
    const dim3 grid((B * H + 3) / 4);
    if (D <= 64)
      hipLaunchKernelGGL((pa_merge_kernel<1, R>), grid, dim3(256), 0, st, mg);
    else if (D <= 128)
      hipLaunchKernelGGL((pa_merge_kernel<2, R>), grid, dim3(256), 0, st, mg);
    else
      hipLaunchKernelGGL((pa_merge_kernel<4, R>), grid, dim3(256), 0, st, mg);
  };
  if (ragged) launch(std::true_type{});
  else launch(std::false_type{});
  LLM_HIP_RET(hipGetLastError());
  return LLM_OK;
}

int llm::pa_merge_rows_internal(const float* part_acc, const float* part_ml, float* out,
                                const PaRowOutputs* rows, const int32_t* context_lens, int ctx_p0,
                                int B, int H, int D, int T, int TS, int pps, int nsplit,
                                int max_tiles, hipStream_t st) {
  PaMergeRowArgs mg{part_acc, part_ml, out, rows ? rows->q : nullptr,
                    rows ? rows->inv_scale : nullptr,
                    rows ? static_cast<_Float16*>(rows->out16) : nullptr, context_lens, B, H, D, T,
                    TS, pps, nsplit, max_tiles, rows ? rows->pack : 0, ctx_p0};
  // a prompt's rows (more splits a row than 16: one after the other they cost more than the
  // waves of a row that take a head each)
  const int quads = H * D / 4;
  if (ctx_p0 >= 0 && !context_lens && pps > 0 && nsplit <= 16 && D % 64 == 0 && quads <= 1024) {
    const int per_row = std::min((quads + 63) / 64 * 64, 256);
    const auto kernel = quads <= 256   ? pa_merge_prompt_kernel<1>
                        : quads <= 512 ? pa_merge_prompt_kernel<2>
                                       : pa_merge_prompt_kernel<4>;
    hipLaunchKernelGGL(kernel, dim3(B), dim3(per_row), 0, st, mg);
    LLM_HIP_RET(hipGetLastError());
    return LLM_OK;
  }
  // one wave per head (heads past 16 loop); a prompt's rows fill the chip by themselves,
  // and four waves each leave room for four times the rows on a CU
  const int threads = 64 * std::min(B >= 1024 ? 4 : 16, H);
  const size_t lds = (size_t)H * D * sizeof(float);
  if (D <= 64)
    hipLaunchKernelGGL(pa_merge_row_kernel<1>, dim3(B), dim3(threads), lds, st, mg);
  else if (D <= 128)
    hipLaunchKernelGGL(pa_merge_row_kernel<2>, dim3(B), dim3(threads), lds, st, mg);
  else
    hipLaunchKernelGGL(pa_merge_row_kernel<4>, dim3(B), dim3(threads), lds, st, mg);
  LLM_HIP_RET(hipGetLastError());
  return LLM_OK;
}

namespace {
template <int D, int TS>
hipError_t beam_occupancy(int* blocks) {
  hipError_t e;
  if (tune_beam_occupancy(D, TS, blocks, &e)) return e;
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(
      blocks, pa_split_kernel<D, TS, false, LLM_BEAM_CHUNK, kKvLoadAux, 2, LLM_BEAM_WAVES, false, true,
                              LLM_F16, true, false, false, 0, false, true, true>,
      256, 0);
}

// Resident waves of the beam-group kernel (0 where the plain schedule runs
// instead: pages above 8 KiB).
template <int D, int TS>
long long beam_resident_waves() {
  if constexpr (!kv_shape_ok(D, TS, 2) || split_stages<D, TS, LLM_F16>() != 2) {
    return 0;
  } else {
    static long long cached = -1;
    if (cached >= 0) return cached;
    int dev = 0, cus = 0, blocks = 0;
    cached = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
        beam_occupancy<D, TS>(&blocks) == hipSuccess &&
        cus > 0 && blocks > 0)
      cached = (long long)cus * blocks * 4;
    else
      (void)hipGetLastError();
    return cached;
  }
}

long long beam_resident_waves_for(int D, int TS) {
  auto by_ts = [&](auto d) -> long long {
    constexpr int DD = decltype(d)::value;
    return TS == 16 ? beam_resident_waves<DD, 16>() : beam_resident_waves<DD, 32>();
  };
  switch (D) {
    case 32: return by_ts(std::integral_constant<int, 32>{});
    case 64: return by_ts(std::integral_constant<int, 64>{});
    case 128: return by_ts(std::integral_constant<int, 128>{});
    default: return by_ts(std::integral_constant<int, 256>{});
  }
}
}  // namespace

int llm::pa_decode_internal(const pa_kv_view* kv, const float* q, int q_stride, float* out,
                            const int32_t* beam_ids, const int32_t* context_lens, int B, int H,
                            int D, int T, float sm_scale, int pages_per_split, void* workspace,
                            size_t workspace_bytes, hipStream_t st, const PaRowOutputs* rows,
                            int row_group, PaPlan* plan) {
  LLM_REQUIRE(kv != nullptr, "pa_decode: kv view is NULL");
  LLM_REQUIRE(B >= 0 && H > 0 && D > 0 && T >= 0, "pa_decode: bad B/H/D/T");
  if (plan) *plan = PaPlan{};
  if (B == 0) return LLM_OK;
  const bool row_out = rows && (rows->q || rows->out16);
  // the FP16 decoder's fused o_proj (PaRowOutputs::o_acc): workgroup-merge launches only
  const bool oproj = rows && rows->o_acc && !rows->q && !rows->f32_rows;
  LLM_REQUIRE(plan || (q != nullptr && (out != nullptr || row_out || oproj)), "pa_decode: q/out NULL");
  LLM_REQUIRE(!oproj || (rows->wo_heads && rows->o_x && rows->o_flag && rows->o_n > 0 &&
                         D <= kOprojMaxD && H <= 64),
              "pa_decode: fused o_proj needs W_o head slices, an output, a range flag, o_n > 0, "
              "head_dim <= 128 and at most 64 heads");
  LLM_REQUIRE(!rows || !rows->q || rows->inv_scale, "pa_decode: row quantisation needs inv_scale");
  LLM_REQUIRE(!row_out || (size_t)H * D * 4 <= 65536, "pa_decode: row outputs need H*D <= 16384");
  LLM_REQUIRE(!rows || !rows->pack || (H * D) % 64 == 0, "pa_decode: packed row outputs need H*D % 64 == 0");
  LLM_REQUIRE(kv->k_pool && kv->v_pool && kv->page_table, "pa_decode: kv pointers NULL");
  LLM_REQUIRE(kv_dtype_bytes(kv->kv_dtype) > 0,
              "pa_decode: kv_dtype must be LLM_F16, LLM_BF16, LLM_F32 or LLM_I8");
  LLM_REQUIRE(kv->num_heads == H, "pa_decode: H != kv->num_heads");
  LLM_REQUIRE(kv->head_dim == D, "pa_decode: D != kv->head_dim");
  LLM_REQUIRE(kv->num_pages > 0 && kv->num_beams > 0 && kv->max_tiles > 0,
              "pa_decode: empty kv view");
  if (!supported(D, kv->page_size, kv->kv_dtype))
    return fail(LLM_ERR_UNSUPPORTED, "pa_decode: unsupported head_dim/page_size/kv_dtype (D in "
                                     "{32,64,128,256}, page_size in {16,32}, one page of "
                                     "1..16 KiB)");
  const size_t page_stride = kv_view_page_stride(*kv);
  LLM_REQUIRE(page_stride >= (size_t)kv->page_size * D * kv_dtype_bytes(kv->kv_dtype) &&
                  page_stride % 16 == 0,
              "pa_decode: page_stride must be 0 or >= one page and a multiple of 16");
  LLM_REQUIRE((long long)kv->num_pages * (long long)page_stride < (1LL << 47),
              "pa_decode: pool too large");
  const int TS = kv->page_size;
  // tiles at or past max_tiles have no page-table entry: they are missing (masked)
  const int ntiles_max = std::max(1, std::min((T + TS - 1) / TS, kv->max_tiles));
  const int pps_fixed = pages_per_split > 0 ? std::min(pages_per_split, kMaxPps) : 0;
  const long long resident = pps_fixed <= 0 ? resident_waves_for(D, TS, kv->kv_dtype) : 0;
  // beam-group launches size their splits for the beam kernel's occupancy
  // (4 waves per SIMD against the plain kernel's 2: C4 8 splits, not 4)
  const long long resident_launch =
      pps_fixed <= 0 && row_group == 4 && kv->kv_dtype == LLM_F16
          ? std::max(resident, beam_resident_waves_for(D, TS)) : resident;
  // fp16 o_proj input only (the FP16 decoder's attention): with at most one
  // merge batch of splits per (b, h) the splits merge inside the split
  // launch's workgroup (C2: 12 merge launches per step fewer), with long splits
  // fp32 rows for a quantising consumer (the INT8 decoder's o_proj prologue)
  // merge in the workgroup too, with a split count that divides the CU's 8
  // resident waves (2 / 4 / 8 waves per workgroup: a 6-wave workgroup would
  // leave 2 of the 8 slots idle): C3 6 -> 8 splits
  const bool f32_rows = rows && rows->f32_rows && !rows->q && !rows->out16;
  const PaTuning tn = pa_tuning();
  int nsplit = choose_nsplit(B, H, ntiles_max, pps_fixed, resident_launch);
  // fp32 rows whose launch is exactly one resident round of more splits than
  // a workgroup merge holds (C3's model at 8 rows per GPU: 128 (row, head)
  // pairs x 16 splits of 33 pages = 2,048 waves): half the splits, twice as
  // long, still split + merge.  Standalone (scripts/tune_attention.py --B 8,
  // profiles/r05/attention_b8_split_sweep.txt): 85.6 -> 84.3 us, the
  // loads-only form 83.7 / 83.4 us at either count.
  const bool half_round = f32_rows && row_group == 1 && pps_fixed <= 0 &&
                          kv->kv_dtype == LLM_F16 && nsplit > kWgmMaxSplits &&
                          (long long)B * H * nsplit == resident_launch &&
                          (ntiles_max + nsplit - 1) / nsplit <= 2 * kShortPps;
  if (half_round) nsplit = (nsplit + 1) / 2;
  bool wgm_ok = ((row_out && rows->out16 && !rows->q) || oproj || f32_rows) && row_group == 1 &&
                      kv->kv_dtype == LLM_F16 && tn.wg_merge && !half_round;
  if (wgm_ok && pps_fixed <= 0 && !f32_rows) {
    const int nw = choose_nsplit(B, H, ntiles_max, 0, resident_launch, kWgmShortPps);
    if (nw >= 2 && nw <= kWgmMaxSplits) nsplit = nw;
  }
  if (wgm_ok && pps_fixed <= 0 && f32_rows && nsplit >= 2) {
    int nw = 2;
    while (nw < nsplit && nw < kWgmMaxSplits) nw *= 2;
    if (nw >= nsplit && (long long)nw * kMaxPps >= ntiles_max) nsplit = nw;
  }
  if (wgm_ok && pps_fixed <= 0 && rows->o_n > 0 && tn.wgm_splits <= 0) {
    const F16Form f = f16_step_form((long long)B * H, D, rows->o_n, ntiles_max, nsplit);
    wgm_ok = f.fused;  // (the workspace holds max_nsplit splits; a workgroup merge needs none)
    nsplit = f.fused ? f.nsplit : (int)std::min<long long>(f.nsplit, max_nsplit(B, H, ntiles_max));
  }
  if (wgm_ok && pps_fixed <= 0 && f32_rows && H * D <= 2048 && tn.wgm_splits <= 0) {
    const F32Form f = f32_step_form((long long)B * H, D, ntiles_max, nsplit);
    wgm_ok = f.wgm;
    nsplit = f.wgm ? f.nsplit : (int)std::min<long long>(f.nsplit, max_nsplit(B, H, ntiles_max));
  }
  // tuning build: forced split counts of beam-group launches and of the
  // workgroup-merge eligible ones (fp16 row outputs, dynamic splits)
  if (row_group == 4 && pps_fixed <= 0) {
    const int f = tn.beam_nsplit;
    if (f >= 2 && (long long)f * kMaxPps >= ntiles_max) nsplit = std::min(f, kMaxSplits);
  }
  if (rows && (rows->out16 || oproj || f32_rows) && !rows->q && row_group == 1 && pps_fixed <= 0) {
    const int f = tn.wgm_splits;
    if (f >= 2 && f <= kWgmMaxSplits && (long long)f * kMaxPps >= ntiles_max) nsplit = f;
  }
  // beam groups of 4 rows (fp16 pages <= 8 KiB, dynamic splits): pa_beam4_kernel,
  // one wave per (group, head, split), splits sized for its own occupancy (a
  // whole number of resident rounds over (group, head) pairs), each split
  // holding <= 128 page items; fixed pages_per_split keeps the BEAM form
  bool use_beam4 = false;
  if (row_group == 4 && pps_fixed <= 0 && kv->kv_dtype == LLM_F16 && TS * D * 2 <= 8192 &&
      tn.beam4 && !tn.beam_mfma) {
    const long long groups = (long long)((B + 3) / 4) * H;
    const long long need = (4LL * ntiles_max + kMaxPps - 1) / kMaxPps;
    long long ns = (tune_beam4_resident_for(D, TS) + groups - 1) / groups;
    ns = std::max(std::max(ns, need), 2LL);
    ns = std::min(ns, max_nsplit(B, H, ntiles_max));
    if (tn.beam4_splits >= 2) ns = std::min<long long>(tn.beam4_splits, max_nsplit(B, H, ntiles_max));
    if (ns >= need && ns >= 2) {
      use_beam4 = true;
      nsplit = (int)ns;
    }
  }
  if (nsplit > kMaxSplits || (long long)nsplit * (pps_fixed > 0 ? pps_fixed : kMaxPps) < ntiles_max)
    return fail(LLM_ERR_UNSUPPORTED,
                "pa_decode: at most 128 splits of at most 128 pages per row (raise "
                "pages_per_split, or pass 0; T <= 16384 pages)");
  const bool direct = nsplit <= 1;
  // beam groups of 4 fp16 rows with counters: dynamic tile assignment
  const bool steal_form = tn.beam_steal && row_group >= 4 && !direct &&
                          kv->kv_dtype == LLM_F16 && pps_fixed <= 0 && !use_beam4 &&
                          !tn.beam_mfma && steal_shape_ok(D, TS);
  if (plan) {
    const int group = std::max(1, std::min(row_group, 4));
    const bool wg = wgm_ok && !direct && group == 1 && nsplit <= kWgmMaxSplits;
    const bool beam = group == 4 && !direct && kv->kv_dtype == LLM_F16 &&
                      TS * D * 2 <= 8192;
    const bool steal = steal_form && rows && rows->beam_ctr;
    plan->nsplit = nsplit;
    plan->form = (direct ? LLM_PA_FORM_DIRECT : wg ? LLM_PA_FORM_WG_MERGE
                  : row_out ? LLM_PA_FORM_SPLIT_MERGE_ROW : LLM_PA_FORM_SPLIT_MERGE) |
                 (beam ? LLM_PA_FORM_BEAM : 0) | (oproj && wg ? LLM_PA_FORM_OPROJ : 0) |
                 (steal ? LLM_PA_FORM_STEAL : 0);
    return LLM_OK;
  }
  unsigned* steal_ctr = nullptr;
  if (steal_form)
    steal_ctr = rows && rows->beam_ctr ? rows->beam_ctr
                                       : tune_steal_counters(2 * (size_t)((B + 3) / 4) * H);
  LLM_REQUIRE(!direct || out != nullptr, "pa_decode: single-split launch needs the fp32 out");
  if (oproj && (direct || row_group != 1 || nsplit > kWgmMaxSplits || !wgm_ok))
    return fail(LLM_ERR_UNSUPPORTED, "pa_decode: the fused o_proj needs the workgroup-merge form");

  PaSplitArgs a{};
  a.k_pool = static_cast<const uint8_t*>(kv->k_pool);
  a.v_pool = static_cast<const uint8_t*>(kv->v_pool);
  a.page_table = kv->page_table;
  a.q = q;
  a.q_stride = q_stride;
  a.out = out;
  a.beam_ids = beam_ids;
  a.context_lens = context_lens;
  a.B = B;
  a.H = H;
  a.T = T;
  a.num_pages = kv->num_pages;
  a.num_beams = kv->num_beams;
  a.max_tiles = kv->max_tiles;
  a.page_stride = page_stride;
  a.pps = pps_fixed;
  a.nsplit = nsplit;
  a.group = std::max(1, std::min(row_group, 4));
  a.qscale = sm_scale * kLog2e;
  a.ragged = context_lens && !rows && !direct && row_group == 1 && pps_fixed <= 0 && B > 1 &&
             B <= kRaggedRows && nsplit < kRaggedSplits &&
             (ntiles_max + nsplit - 1) / nsplit >= kRaggedPages;
  const bool wgm = wgm_ok && !direct && a.group == 1 && nsplit <= kWgmMaxSplits;
  if (!direct && !wgm) {  // (the workgroup merge keeps its splits' states in LDS)
    const size_t need = (size_t)B * H * nsplit * (size_t)(D + 2) * sizeof(float);
    LLM_REQUIRE(workspace != nullptr && workspace_bytes >= need,
                "pa_decode: workspace too small (see pa_decode_workspace_bytes)");
    a.part_acc = static_cast<float*>(workspace);
    a.part_ml = a.part_acc + (size_t)B * H * nsplit * D;
  }
  a.balance16 = tn.beam_balance16;
  // beam-group workgroups in split-major order (PaSplitArgs::smaj).  Same box,
  // C4 (profiles/r06/c4_smaj_ab.txt): 12,719-12,737 against 12,604-12,617
  // tok/s; the launch's HBM bytes 1.031 -> 1.014x algorithmic
  // (profiles/pmc_attention_c4.json), the exits by dispatch slot unchanged
  a.smaj = a.group == 4 && tn.beam_smaj ? 1 : 0;
  a.beam4 = use_beam4 ? 1 : 0;
  a.steal = a.group == 4 ? steal_ctr : nullptr;
  if (wgm) {
    a.wgm = 1;
    a.out16 = static_cast<_Float16*>(rows->out16);
    a.pack = rows->pack;
    a.out = rows->keep_out || f32_rows ? out : nullptr;
    if (oproj) {
      a.o_acc = rows->o_acc;
      a.o_x = rows->o_x;
      a.wo_heads = static_cast<const _Float16*>(rows->wo_heads);
      a.o_n = rows->o_n;
      a.o_flag = rows->o_flag;
    }
  }
  // one split of fp16 pages writes the o_proj's fp16 rows itself
  const bool direct16 = direct && row_out && rows->out16 && !rows->q && !rows->keep_out &&
                        kv->kv_dtype == LLM_F16;
  if (direct16) {
    a.out16 = static_cast<_Float16*>(rows->out16);
    a.pack = rows->pack;
  }
  hipError_t e;
  bool beam = false;  // the beam kernel ran: every split holds a partial
  switch (D) {
    case 32: e = dispatch_kvt<32>(a, kv->kv_dtype, TS, direct, st, &beam); break;
    case 64: e = dispatch_kvt<64>(a, kv->kv_dtype, TS, direct, st, &beam); break;
    case 128: e = dispatch_kvt<128>(a, kv->kv_dtype, TS, direct, st, &beam); break;
    default: e = dispatch_kvt<256>(a, kv->kv_dtype, TS, direct, st, &beam); break;
  }
  if (e != hipSuccess) return fail(LLM_ERR_HIP, std::string("pa_split launch: ") + hipGetErrorString(e));
  if (wgm || direct16) return LLM_OK;
  if (row_out && !direct)
    return pa_merge_rows_internal(a.part_acc, a.part_ml, rows->keep_out ? out : nullptr, rows,
                                  context_lens, -1, B, H, D, T, TS, beam ? -1 : pps_fixed, nsplit,
                                  kv->max_tiles, st);
  if (!direct) {
    const int r = pa_merge_splits_internal(a.part_acc, a.part_ml, out, context_lens, B, H, D, T,
                                           TS, beam ? -1 : pps_fixed, nsplit, kv->max_tiles, st, a.ragged);
    if (r != LLM_OK) return r;
  }
  if (row_out) {  // single split: out is final; convert it in a row pass
    if (rows->q)
      LLM_HIP_RET(launch_quantize_rows(out, B, H * D, rows->q, rows->inv_scale, st, rows->pack));
    if (rows->out16)
      LLM_HIP_RET(launch_to_f16(out, (size_t)B * H * D, rows->out16, st, rows->pack ? H * D : 0));
  }
  return LLM_OK;
}

extern "C" int pa_decode_grouped(const pa_kv_view* kv, const float* q, float* out,
                                 const int32_t* beam_ids, const int32_t* context_lens, int B,
                                 int H, int D, int T, float sm_scale, int pages_per_split,
                                 int row_group, void* workspace, size_t workspace_bytes,
                                 void* stream) {
  LLM_REQUIRE(row_group >= 1 && row_group <= 4, "pa_decode_grouped: row_group must be in [1, 4]");
  return pa_decode_internal(kv, q, H * D, out, beam_ids, context_lens, B, H, D, T, sm_scale,
                            pages_per_split, workspace, workspace_bytes, as_stream(stream),
                            nullptr, row_group);
}

extern "C" int pa_decode_plan(const pa_kv_view* kv, int B, int H, int D, int T,
                              int pages_per_split, int row_group, int* nsplit, int* form) {
  LLM_REQUIRE(nsplit && form, "pa_decode_plan: NULL output");
  LLM_REQUIRE(row_group >= 1 && row_group <= 4, "pa_decode_plan: row_group must be in [1, 4]");
  PaPlan p;
  const int rc = pa_decode_internal(kv, nullptr, H * D, nullptr, nullptr, nullptr, B, H, D, T, 1.f,
                                    pages_per_split, nullptr, 0, nullptr, nullptr, row_group, &p);
  *nsplit = p.nsplit;
  *form = p.form;
  return rc;
}

extern "C" int pa_decode(const pa_kv_view* kv, const float* q, float* out,
                         const int32_t* beam_ids, const int32_t* context_lens, int B, int H,
                         int D, int T, float sm_scale, int pages_per_split, void* workspace,
                         size_t workspace_bytes, void* stream) {
  return pa_decode_internal(kv, q, H * D, out, beam_ids, context_lens, B, H, D, T, sm_scale,
                            pages_per_split, workspace, workspace_bytes, as_stream(stream));
}
