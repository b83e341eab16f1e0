// Shared host/device helpers for the gfx950 decode path.
#pragma once

#ifndef LLM_TUNING
#define LLM_TUNING 0  // 1: the tuning library (Makefile `tune`)
#endif

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <string>

#include "llm_decoder.h"

namespace llm {

// Integer tuning knob from the environment (dflt when unset or empty).
inline int env_int(const char* name, int dflt) {
  const char* v = std::getenv(name);
  return (v && *v) ? std::atoi(v) : dflt;
}

// Thread-local last-error message (llm_last_error()).
void set_error(const std::string& msg);
int fail(int status, const std::string& msg);

#define LLM_HIP_RET(expr)                                                        \
  do {                                                                           \
    hipError_t _e = (expr);                                                      \
    if (_e != hipSuccess)                                                        \
      return ::llm::fail(LLM_ERR_HIP, std::string(#expr " failed: ") +           \
                                          hipGetErrorString(_e));                \
  } while (0)

#define LLM_REQUIRE(cond, msg)                                                   \
  do {                                                                           \
    if (!(cond)) return ::llm::fail(LLM_ERR_INVALID, msg);                       \
  } while (0)

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// ---------------------------------------------------------------------------
// device helpers
// ---------------------------------------------------------------------------
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr float kNegSentinel = -1.0e30f;  // "minus infinity" that stays finite
constexpr float kLog2e = 1.4426950408889634f;

// Counted fixed-point accumulator of the FP16 decoder's fused o_proj
// (pa_decode.hip, workgroup merge): the H (row, head) workgroups of a row each
// add their head's product o_h . W_o[h] into one int64 per output column as
// 2^56 (an arrival count in the top bits) + the product in units of 2^-32.
// Integer addition is order-independent, so the sum is the same bits whatever
// order the heads' atomics land in (fp32 atomics would not be), and the adder
// whose returned old value counts H - 1 arrivals holds the complete sum: it
// stores the fp32 value and clears the column for the next layer.  Exact to
// 2^-33 per head for |sum| < 2^23 (8.4e6) and H <= 64.
//
// Range guard: the count bits stay intact only while |sum| < 2^23.  Each
// head's term is therefore clamped to |v| <= oacc_limit(H) = (2^23 - 1) / H,
// so H terms can never reach 2^23, and a NaN maps to the positive limit.  A
// clamped term sets *flag (a plain vector store; the decoder turns it into
// LLM_ERR_RANGE at llm_decoder_sync / the next synchronous step).  The
// column then still completes after exactly H arrivals and is cleared, so an
// out-of-range value costs that one output, never the later layers or steps.
constexpr float kOAccScale = 4294967296.f;  // 2^32
constexpr long long kOAccCount = 1LL << 56;
__host__ __device__ __forceinline__ float oacc_limit(int H) {
  return (float)((1 << 23) - 1) / (float)H;
}
__device__ __forceinline__ long long oacc_term(float v, float lim, bool& clamped) {
  const bool ok = fabsf(v) <= lim;  // false for NaN and +-inf
  clamped = !ok;
  const float c = ok ? v : (v < 0.f ? -lim : lim);
  return __float2ll_rn(c * kOAccScale) + kOAccCount;
}
__device__ __forceinline__ int oacc_count(long long v) {
  return (int)((v + (kOAccCount >> 1)) >> 56);
}
__device__ __forceinline__ float oacc_value(long long v) {
  const long long f = v - (long long)oacc_count(v) * kOAccCount;
  return (float)((double)f * (1.0 / 4294967296.0));
}

// DPP lane moves (row = 16 lanes).  ctrl must be a compile-time constant.
template <int CTRL>
__device__ __forceinline__ float mov_dpp(float x) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xF, 0xF, true));
}

// x and the x of lane l ^ 16 (l ^ 32), in some order: an exchange of rows between registers,
// no trip through LDS.
struct LanePair {
  float a, b;
};
__device__ __forceinline__ LanePair with_lane16(float x) {
  const uint32_t b = __builtin_bit_cast(uint32_t, x);
  const auto r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
  return {__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1])};
}
__device__ __forceinline__ LanePair with_lane32(float x) {
  const uint32_t b = __builtin_bit_cast(uint32_t, x);
  const auto r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return {__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1])};
}
__device__ __forceinline__ float add(LanePair p) { return p.a + p.b; }
// (fmaxf of what comes as bits takes two more instructions to quiet a NaN)
__device__ __forceinline__ float larger(LanePair p) {
  float x;
  asm("v_max_f32 %0, %1, %2" : "=v"(x) : "v"(p.a), "v"(p.b));
  return x;
}
// The largest of lanes l, l ^ 16, l ^ 32, l ^ 48 (the same lane of the wave's four rows).
__device__ __forceinline__ float rows_max(float x) { return larger(with_lane32(larger(with_lane16(x)))); }

// Sum over aligned groups of G lanes (G in {2,4,8,16,32,64}); every lane of a
// group ends with the identical total (commutative butterfly).
template <int G>
__device__ __forceinline__ float group_sum(float x) {
  if constexpr (G >= 2) x += mov_dpp<0xB1>(x);   // quad_perm [1,0,3,2]
  if constexpr (G >= 4) x += mov_dpp<0x4E>(x);   // quad_perm [2,3,0,1]
  if constexpr (G >= 8) x += mov_dpp<0x141>(x);  // row_half_mirror
  if constexpr (G >= 16) x += mov_dpp<0x140>(x); // row_mirror
  if constexpr (G >= 32) x = add(with_lane16(x));
  if constexpr (G >= 64) x = add(with_lane32(x));
  return x;
}

// Inclusive scans over the wave's lanes (row shifts, then the rows' last lanes to the
// rows behind), so lane 63 holds the total; wave_scan_max of values >= 0.
template <int CTRL, int ROWS>
__device__ __forceinline__ int lanes_before(int x) {  // 0 where there is none
  return __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xF, false);
}
__device__ __forceinline__ int wave_scan_add(int x) {
  x += lanes_before<0x111, 0xF>(x);  // row_shr 1, 2, 4, 8
  x += lanes_before<0x112, 0xF>(x);
  x += lanes_before<0x114, 0xF>(x);
  x += lanes_before<0x118, 0xF>(x);
  x += lanes_before<0x142, 0xA>(x);  // row_bcast 15 into rows 1 and 3
  return x + lanes_before<0x143, 0xC>(x);  // row_bcast 31 into rows 2 and 3
}
__device__ __forceinline__ int wave_scan_max(int x) {
  x = max(x, lanes_before<0x111, 0xF>(x));
  x = max(x, lanes_before<0x112, 0xF>(x));
  x = max(x, lanes_before<0x114, 0xF>(x));
  x = max(x, lanes_before<0x118, 0xF>(x));
  x = max(x, lanes_before<0x142, 0xA>(x));
  return max(x, lanes_before<0x143, 0xC>(x));
}

__device__ __forceinline__ float wave_max(float x) {
  x = fmaxf(x, mov_dpp<0xB1>(x));
  x = fmaxf(x, mov_dpp<0x4E>(x));
  x = fmaxf(x, mov_dpp<0x141>(x));
  x = fmaxf(x, mov_dpp<0x140>(x));
  return rows_max(x);
}

// op over lanes l, l ^ 32, l ^ 16, .. l ^ 1, in that order: exchanges between registers, no trips through
// LDS (behind lane ^ 8 lanes l and l ^ 8 hold the same, so that a rotation by 4 is an exchange
// too).
template <int CTRL>
__device__ __forceinline__ int mov_lanes(int x) {
  return __builtin_amdgcn_mov_dpp(x, CTRL, 0xF, 0xF, true);
}
template <typename T, typename Op>
__device__ __forceinline__ T wave_reduce(T v, Op op) {
  static_assert(sizeof(T) == 4);
  const auto as_int = [](T x) { return __builtin_bit_cast(int, x); };
  const auto as_t = [](int x) { return __builtin_bit_cast(T, x); };
  const LanePair p = with_lane32(__builtin_bit_cast(float, v));
  v = op(__builtin_bit_cast(T, p.a), __builtin_bit_cast(T, p.b));
  const LanePair q = with_lane16(__builtin_bit_cast(float, v));
  v = op(__builtin_bit_cast(T, q.a), __builtin_bit_cast(T, q.b));
  v = op(v, as_t(mov_lanes<0x128>(as_int(v))));  // row_ror 8, 4
  v = op(v, as_t(mov_lanes<0x124>(as_int(v))));
  v = op(v, as_t(mov_lanes<0x4E>(as_int(v))));  // quad_perm [2,3,0,1], [1,0,3,2]
  return op(v, as_t(mov_lanes<0xB1>(as_int(v))));
}
// x of lane l ^ OFF, OFF 1, 2, 4 or 8
template <int OFF>
__device__ __forceinline__ int lane_xor(int x) {
  if constexpr (OFF == 4)
    return __builtin_amdgcn_ds_swizzle(x, 4 << 10 | 31);
  else
    return mov_lanes<OFF == 1 ? 0xB1 : OFF == 2 ? 0x4E : 0x128>(x);  // quad_perm, row_ror 8
}
template <int OFF>
__device__ __forceinline__ float lane_xor(float x) {
  return __builtin_bit_cast(float, lane_xor<OFF>(__builtin_bit_cast(int, x)));
}
__device__ __forceinline__ float wave_sum(float x) {
  return wave_reduce(x, [](float a, float b) { return a + b; });
}

__device__ __forceinline__ int wave_id_uniform() {
  return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

// 16 bytes per lane from memory straight into LDS, lane l's at lds + 16 l (lds:
// the same for the whole wave).  Written as assembly so the compiler does not
// order later LDS reads behind it: a wave calls wait_lds_loads() and then the
// workgroup barrier before anyone reads what was loaded.
__device__ __forceinline__ void load_to_lds(const void* src, void* lds) {
  const uint32_t at = __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(at), "v"(src)
               : "memory", "m0");
}
// The wait (for all but the wave's last LEFT loads, and for its LDS reads) is the
// builtin: the compiler then knows that its own earlier loads are there too and
// does not wait for them among the next stage's.
template <int LEFT = 0>
__device__ __forceinline__ void wait_lds_loads() {
  static_assert(LEFT < 64);
  __builtin_amdgcn_s_waitcnt(0x0070 | (LEFT & 15) | (LEFT >> 4) << 14);  // vmcnt(LEFT), lgkmcnt(0)
  asm volatile("" ::: "memory");
}
// 16 bytes per lane written past L2.  A launch ends with its XCDs' L2s writing out what they
// hold, the next one starts after that; what is written past them meanwhile does not wait
// there (2048 x 2048 fp32 from 256 blocks of a product: 23.3 -> 18.6 us of the whole; 64
// MiB of them 46.3 -> 40.9; nontemporal stores 20.8, 46.1).  For results larger than a few
// MiB, that another launch reads.  The s_nop: the next instruction may write v's registers.
__device__ __forceinline__ void store_through(void* p, u32x4 v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ void store_through(void* p, u32x2 v) {
  asm volatile("global_store_dwordx2 %0, %1, off sc0 sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}
// The workgroup's barrier without __syncthreads' wait for the loads in flight; no access
// to memory moves over it.
__device__ __forceinline__ void barrier_only() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Offset of activation element (m, k) in MFMA A-fragment order ("packed A"):
// one contiguous 1 KiB block per (16-row tile, k-step), lane l of the block
// holding row l&15 and 16 B of k (16 int8 or 8 fp16) — the exact operand
// layout of v_mfma_i32_16x16x64_i8 / v_mfma_f32_16x16x32_f16, so the GEMM
// reads each fragment with one coalesced buffer_load_dwordx4.
// KS = k-steps per row (K/64 for int8, K/32 for fp16).  Offsets in elements.
__host__ __device__ __forceinline__ size_t a_frag_off_i8(int m, int k, int KS) {
  return ((size_t)((m >> 4) * KS + (k >> 6)) * 64 + (m & 15) + 16 * ((k & 63) >> 4)) * 16 + (k & 15);
}
__host__ __device__ __forceinline__ size_t a_frag_off_f16(int m, int k, int KS) {
  return ((size_t)((m >> 4) * KS + (k >> 5)) * 64 + (m & 15) + 16 * ((k & 31) >> 3)) * 8 + (k & 7);
}
// The row of a workgroup that writes one of `rows` packed rows: workgroups go round the 8
// XCDs, and a packed tile's 16 rows lie 16 bytes each in its lines, so that rows in their own
// order leave parts of lines in every XCD's L2 (int8 2048 x 8192: 33 MB written for 17).  128
// rows at a time an XCD gets whole tiles.
__device__ __forceinline__ int packed_row(int block, int rows) {
  const int first = block & ~127;
  return first + 128 <= rows ? first + 16 * (block & 7) + (block >> 3 & 15) : block;
}

}  // namespace llm
