// Matrix products of the layer-stack models: packing, plain products, the
// grouped-query projections and the grouped (expert) products.  The kernels are
// in mm_impl.hpp; mm_mix.hip has the epilogues of the other mixers.
#include "mm_impl.hpp"

#include <cmath>

namespace llm {
namespace {

template <typename T>
__global__ void mm_pack_kernel(const uint16_t* __restrict__ src, const int32_t* __restrict__ map,
                               int N, int K, int KS, size_t chunks, u32x4* __restrict__ dst) {
  constexpr int E = 16 / sizeof(T);
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= chunks) return;
  const int lane = idx & 63;
  const size_t blk = idx >> 6;
  const int ks = (int)(blk % KS);
  const int n = (int)(blk / KS) * 16 + (lane & 15);
  const int row = n < N ? (map ? map[n] : n) : -1;
  const int k0 = ks * 4 * E + (lane >> 4) * E;
  T v[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const uint16_t h = row >= 0 && k0 + e < K ? src[(size_t)row * K + k0 + e] : (uint16_t)0;
    if constexpr (sizeof(T) == 2)
      v[e] = __builtin_bit_cast(T, h);
    else
      v[e] = __builtin_bit_cast(T, (uint32_t)h << 16);
  }
  u32x4 o;
  __builtin_memcpy(&o, v, 16);
  dst[idx] = o;
}

}  // namespace

size_t mm_packed_bytes(int dtype, int N, int K) {
  const int ks = mm_kstep(dtype);
  return (size_t)((N + 15) / 16) * ((K + ks - 1) / ks) * 1024;
}

hipError_t mm_pack(int dtype, const uint16_t* src, const int32_t* row_map, int N, int K, void* dst,
                   hipStream_t st) {
  const int ks = mm_kstep(dtype), KS = (K + ks - 1) / ks;
  const size_t chunks = (size_t)((N + 15) / 16) * KS * 64;
  const dim3 grid((unsigned)((chunks + 255) / 256));
  if (dtype == LLM_F32)
    hipLaunchKernelGGL(mm_pack_kernel<float>, grid, dim3(256), 0, st, src, row_map, N, K, KS,
                       chunks, static_cast<u32x4*>(dst));
  else
    hipLaunchKernelGGL(mm_pack_kernel<__bf16>, grid, dim3(256), 0, st, src, row_map, N, K, KS,
                       chunks, static_cast<u32x4*>(dst));
  return hipGetLastError();
}

static KernelArgs plain_args(int dtype, const MmArgs& a) {
  KernelArgs p{};
  p.a = a;
  p.KS = (a.K + mm_kstep(dtype) - 1) / mm_kstep(dtype);
  return p;
}

// A product of few blocks takes the time of its chain of K, so slices of K fill the chip, and the reader
// of the sums, a norm, adds them up as it reads.  Priced by the form that each count of slices would take,
// of whose time K / 2048 is the product's, 0.5 us for a slice more and its sums' way to memory and
// back at 3 TB/s, and more slices only for 2 % and more.  With the norm behind it (us, weights from memory, 1 / 2 / 4 slices; the choice):
// bf16 2048 columns of K 4096: 16 rows 13.0 / 10.7 / 10.9 (2), 64 14.4 / 13.5 / 11.4 (4), 333 26.3 / 19.7 /
// 18.5 (4), 1000 32.7 / 28.4 / 30.8 (2); K 6144: 333 rows 34.2 / 24.5 / 22.3 (4); K 2048: 16 rows 9.0 / 8.2 /
// 8.1 (2), 333 16.1 / 15.3 / 16.7 (2), 1400 24.8 / 26.4 / 31.2 (1); 1024 columns of K 1024: 1000 rows 13.3 /
// 14.6 / 17.7 (1).  Over 1 to 2011 rows and 1024 to 4096 columns and K 0.88 of the time in bf16 (the best
// count each: 0.86), 0.93 in fp32 (0.91).
template <typename T>
static int parts_of(KernelArgs p) {
  int best = 1;
  float least = 0.f;
  for (int parts = 1; parts <= kMmMostParts; parts *= 2) {
    if (parts > 1 && (p.KS / parts < 24 || p.a.M * parts > kMmPartRows)) break;
    p.a.parts = parts;
    const float us = form_of<T, kStore>(p).us;
    if (us == 0.f) break;
    const float all = kFixedUs + (us - kFixedUs) * (float)p.a.K / (2048.f * (float)parts) +
                      (float)(parts - 1) * (0.5f + 1.33e-6f * (float)p.a.M * (float)p.a.N);
    if (parts > 1 && all >= 0.98f * least) continue;
    best = parts;
    least = all;
  }
  return best;
}

int mm_parts(int dtype, int M, int N, int K) {
  MmArgs a;
  a.M = M;
  a.N = N;
  a.K = K;
  const KernelArgs p = plain_args(dtype, a);
  return dtype == LLM_F32 ? parts_of<float>(p) : parts_of<__bf16>(p);
}

template <typename T>
static float whole_us(KernelArgs p, int M, int N) {
  if (M == 0) return 0.f;
  p.a.M = M;
  p.a.N = N;
  const float us = form_of<T, kStore>(p).us;
  if (us == 0.f) return NAN;  // not priced
  return kFixedUs + (us - kFixedUs) * (float)p.a.K / 2048.f;
}

// By mm's prices: a launch more is in them, the rows' pages and rotations are not (2048 rows x 2560 columns
// x 2048 to pages 39 us, priced 28; their 512 columns of keys and values 15.6 and one row's queries 5.7, priced
// 12.1 and 4.7; a scan's 2011 x 8192 60, priced 53; 4096 of its columns 34.8 and three rows' 6.9, priced 27 and 4.7).
bool mm_apart(int dtype, int M, int N, int K, int rows, int cols) {
  if (cols % 16 != 0 || cols >= N) return false;  // (a column tile of packed weights holds 16)
  MmArgs a;
  a.K = K;
  const KernelArgs p = plain_args(dtype, a);
  const auto us = [&](int m, int n) {
    return dtype == LLM_F32 ? whole_us<float>(p, m, n) : whole_us<__bf16>(p, m, n);
  };
  return us(M, N - cols) + us(rows, cols) < us(M, N);
}

hipError_t mm(int dtype, const MmArgs& a, hipStream_t st) {
  const KernelArgs p = plain_args(dtype, a);
  return dtype == LLM_F32 ? launch<float, kStore>(p, st) : launch<__bf16, kStore>(p, st);
}

hipError_t mm_qkv(int dtype, const MmArgs& a, const MmQkv& e, hipStream_t st) {
  if (a.rows && a.N > (e.H + e.G) * e.D) return hipErrorInvalidValue;  // (value columns go by rows side by side)
  KernelArgs p = plain_args(dtype, a);
  p.q = e;
  return dtype == LLM_F32 ? launch<float, kQkv>(p, st) : launch<__bf16, kQkv>(p, st);
}

int mm_group_tile_rows(int M, int top, int experts) {
  const long long rows = (long long)M * top / experts;  // of an expert, on average
  return M <= 64 || rows < 24 ? 16 : rows < 192 ? 64 : 128;
}

hipError_t mm_grouped_in(int dtype, const MmGrouped& g, int w_nt, hipStream_t st) {
  return dtype == LLM_F32 ? launch_grouped<float, kGroupIn>(g, w_nt, st)
                          : launch_grouped<__bf16, kGroupIn>(g, w_nt, st);
}

hipError_t mm_grouped_out(int dtype, const MmGrouped& g, int w_nt, hipStream_t st) {
  return dtype == LLM_F32 ? launch_grouped<float, kGroupOut>(g, w_nt, st)
                          : launch_grouped<__bf16, kGroupOut>(g, w_nt, st);
}

}  // namespace llm
