// Kernels of the layer-stack models' matrix products on gfx950 MFMA; mm.hip and
// mm_mix.hip instantiate them per epilogue.
//
//   bf16: v_mfma_f32_16x16x32_bf16      fp32: v_mfma_f32_16x16x4_f32
//
// Two kernels.  Decode rows stream: a block owns 16 MT rows x 16 NT columns, its
// 8 waves split K and load A (row-major rows, 64 bytes per row and k-step) and W
// (packed 1 KiB fragments) straight into registers, so every weight byte of the
// product is in flight at once.  More rows go through LDS in blocks of 64 x 32 to
// 128 x 256, both operands loaded from memory straight into LDS.
// Grouped rows take either form; a tile list (built by the routing kernel) names
// the group and rows of each row of the grid.
// A and W share the k order inside a fragment, so the sum is exact whatever the
// hardware's own order; C: column = lane & 15, row = 4 (lane >> 4) + reg.
//
// Epilogues work on column pairs (2i, 2i + 1), which sit in neighbouring lanes:
// rotation partners and (gate, up) pairs are packed side by side, so a pair is
// one DPP move away and no product needs a second launch to finish it.
#pragma once

#include <algorithm>

#include "block_product.hpp"
#include "common.hpp"
#include "mm.hpp"

namespace llm {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

enum Epi {
  kStore, kQkv, kGroupIn, kGroupOut,                                    // mm.hip
  kSplit, kGlu, kSoftplus, kConv, kLatent, kHeads, kExpand              // mm_mix.hip
};

template <typename T>
struct Kind;
template <>
struct Kind<__bf16> {
  static constexpr bool BF16 = true;
  static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <>
struct Kind<float> {
  static constexpr bool BF16 = false;
  static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
    const f32x4 x = __builtin_bit_cast(f32x4, a), y = __builtin_bit_cast(f32x4, b);
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[j], y[j], c, 0, 0, 0);
    return c;
  }
};

struct KernelArgs {
  MmArgs a;
  int KS;
  MmQkv q;
  MmGrouped g;
  MmSplit split;
  MmConv conv;
  MmLatent lat;
  MmHeads heads;
  MmPageRows page_rows;
  GluParams glu;
  const float* bias;
};

// Where a plain product goes.  A captured head's rows have another place at every step (16 rows of
// 32,768 logits: 26 us into device memory and a copy of 38 over the bus behind it, 51 as the
// blocks' own stores to the host's memory).
__device__ __forceinline__ float* stored_to(const KernelArgs& p) {
  float* c = p.a.C_at ? *p.a.C_at : nullptr;
  return (c ? c : p.a.C) + blockIdx.z * p.a.c_part;
}

__device__ __forceinline__ float glu(float gate, float up, const GluParams& p) {
  const float g = fminf(gate, p.limit);
  const float u = fminf(fmaxf(up, -p.limit), p.limit);
  return g / (1.f + expf(-p.alpha * g)) * (u + p.up_bias);
}

// log(1 + e^v) = max(v, 0) + log1p(e), e = e^-|v|; log1p(e) = 2 atanh(s) with
// s = e / (2 + e) <= 1/3, whose series needs no case for small or large v
__device__ __forceinline__ float softplus(float v) {
  const float a = -fabsf(v), t = a * kLog2e;
  const float lo = fmaf(a, kLog2e, -t);  // what rounding took from the exponent
  const float p = __builtin_amdgcn_exp2f(t);
  const float e = fmaf(p, lo * 0.6931472f, p);
  const float s = e * __builtin_amdgcn_rcpf(2.f + e), q = s * s;
  float r = 1.f / 15.f;
  r = fmaf(r, q, 1.f / 13.f);
  r = fmaf(r, q, 1.f / 11.f);
  r = fmaf(r, q, 1.f / 9.f);
  r = fmaf(r, q, 1.f / 7.f);
  r = fmaf(r, q, 1.f / 5.f);
  r = fmaf(r, q, 1.f / 3.f);
  r = fmaf(r, q, 1.f);
  return fmaxf(v, 0.f) + 2.f * s * r;
}

template <typename T>
__device__ __forceinline__ void put_pair(T* p, float v0, float v1) {
  typedef T pair_t __attribute__((ext_vector_type(2)));
  pair_t v;
  v[0] = (T)v0;
  v[1] = (T)v1;
  *reinterpret_cast<pair_t*>(p) = v;
}

// What a block of rows and columns works on: set once from the launch arguments
// or the tile list.
template <typename T>
struct Block {
  static constexpr bool kSome = false;
  const T* A = nullptr;
  const char* W = nullptr;
  int lda = 0, M = 0, N = 0, KS = 0, m0 = 0;
  size_t w_tile = 0;  // bytes from a column tile of W to the next
  bool shared = false;
  GluParams glu;
};
// One of MmArgs::rows.  A kernel of its own: the look-up costs the others registers (bf16 kSplit streams
// 82 -> 87, 110 -> 120, 130 -> 136, and 5.8 -> 6.2 us for 64 rows x 96 columns of a decode step).
template <typename T>
struct SomeBlock : Block<T> {
  static constexpr bool kSome = true;
};
template <typename T, bool SOME>
using BlockOf = std::conditional_t<SOME, SomeBlock<T>, Block<T>>;

template <typename T, int EPI>
__device__ __forceinline__ Block<T> block_of(const KernelArgs& p, int row_block, int by) {
  Block<T> b;
  if constexpr (EPI == kGroupIn || EPI == kGroupOut) {
    const MmTile t = p.g.tiles[by];
    const MmGroup g = p.g.groups[t.group];
    b.shared = t.group >= p.g.n_routed;
    b.m0 = t.row0;
    b.M = t.row0 + t.rows;
    if constexpr (EPI == kGroupIn) {
      b.A = static_cast<const T*>(p.g.h);
      b.lda = p.g.ldh;
      b.W = static_cast<const char*>(g.w_in);
      b.N = g.n_in;
      b.KS = g.ks_in;
      b.glu = g.glu;
    } else {
      b.A = static_cast<const T*>(b.shared ? p.g.act_shared : p.g.act);
      b.lda = b.shared ? p.g.lds : p.g.lda;
      b.W = static_cast<const char*>(g.w_out);
      b.N = g.n_out;
      b.KS = g.ks_out;
    }
  } else {
    b.A = static_cast<const T*>(p.a.A);
    b.W = static_cast<const char*>(p.a.W);
    b.lda = p.a.lda;
    b.M = p.a.M;
    b.N = p.a.N;
    b.KS = p.KS;
    b.m0 = by * row_block;
    b.glu = p.glu;
    if constexpr (EPI == kHeads) {
      b.A += blockIdx.z * p.heads.a_head;
      b.W += blockIdx.z * p.heads.w_head;
    }
    if constexpr (EPI == kStore) {
      b.w_tile = (size_t)p.KS * 1024;
      if (p.a.parts > 1) {
        const int z = blockIdx.z, k0 = z * p.KS / p.a.parts;
        b.A += (size_t)k0 * (64 / sizeof(T));
        b.W += (size_t)k0 * 1024;
        b.KS = (z + 1) * p.KS / p.a.parts - k0;
      }
      return b;
    }
  }
  b.w_tile = (size_t)b.KS * 1024;
  return b;
}

// Products of which only some rows may be wanted (MmArgs::rows).
template <int EPI>
constexpr bool some_rows() {
  return EPI == kQkv || EPI == kLatent || EPI == kSplit;
}

// Row m of A (the last one for rows past it).
template <typename T, int EPI, typename B>
__device__ __forceinline__ const char* a_row(const KernelArgs& p, const B& b, int m) {
  m = min(m, b.M - 1);
  if constexpr (EPI == kGroupIn) {
    if (!b.shared) m = p.g.perm[m] / p.g.top;
  }
  if constexpr (EPI == kHeads) {
    if (p.heads.rows) m = p.heads.rows[m];
  }
  if constexpr (B::kSome) m = p.a.rows[m];
  if constexpr (EPI == kExpand) {
    const MmPageRows& r = p.page_rows;
    const int pos = r.pos[m];
    int page = r.table[(size_t)r.slot[m] * r.max_tiles + min(pos / kPageTokens, r.max_tiles - 1)];
    page = min(max(page, 0), r.num_pages - 1);
    return static_cast<const char*>(r.pool) + (size_t)page * r.page_stride +
           (size_t)(pos % kPageTokens) * r.row * sizeof(T);
  }
  return reinterpret_cast<const char*>(b.A + (size_t)m * b.lda);
}

template <int EPI>
struct History {};
template <>
struct History<kConv> {  // of the pair's two channels: earlier inputs, taps, bias
  float v[2][kMmConvTaps - 1], w[2][kMmConvTaps], bias[2];
};

// What an epilogue needs of a row, and of a column pair (n, n + 1): found once
// per row and column of a block's tiles.
template <int EPI>
struct RowOf {
  static constexpr bool PAGED = EPI == kQkv || EPI == kExpand;
  int m = -1;             // -1: no such row
  int at = 0, entry = 0;  // paged: place in the page, page-table entry of head 0 (-1: none)
  int pos = 0;
  int out = 0;            // kGroupOut: the row's place in the output, its weight
  float weight = 1.f;

  __device__ __forceinline__ RowOf() {}
  template <typename B>
  __device__ __forceinline__ RowOf(const KernelArgs& p, const B& b, int row) {
    if (row >= b.M) return;
    m = row;
    if constexpr (B::kSome) m = p.a.rows[row];
    if constexpr (PAGED) {
      const MmQkv& e = p.q;
      pos = e.pos[m];
      const int tile = pos / kPageTokens;
      at = pos % kPageTokens;
      entry = tile < e.max_tiles ? e.slot[m] * e.G * e.max_tiles + tile : -1;
    }
  }
  // of lane l
  __device__ __forceinline__ RowOf from(int l) const {
    RowOf r;
    r.m = __shfl(m, l, 64);
    if constexpr (PAGED) {
      r.at = __shfl(at, l, 64);
      r.entry = __shfl(entry, l, 64);
      r.pos = __shfl(pos, l, 64);
    }
    if constexpr (EPI == kGroupOut) {
      r.out = __shfl(out, l, 64);
      r.weight = __shfl(weight, l, 64);
    }
    return r;
  }
  // kGroupOut.  The stream kernel's rows do it in Target::find, behind one branch with the
  // rest: behind one of its own the compiler waits for the weight, and so for the first
  // loads of A and W, before it issues the next (fp32, a row: 18.0 us, now 14.1).
  template <typename T>
  __device__ __forceinline__ void look_up(const KernelArgs& p, const Block<T>& b) {
    if constexpr (EPI == kGroupOut) {
      out = b.shared ? p.g.M * p.g.top + m : p.g.perm[m];
      if (!b.shared) weight = p.g.weight[out];
    }
  }
};
template <int EPI>
struct ColOf {
  int n = -1;  // -1: no such column
  int part = 0, head = 0, d = 0;

  __device__ __forceinline__ ColOf() {}
  template <typename T>
  __device__ __forceinline__ ColOf(const KernelArgs& p, const Block<T>& b, int col) {
    if (col >= b.N) return;
    n = col;
    if constexpr (RowOf<EPI>::PAGED) {  // query, key, value
      const MmQkv& e = p.q;
      const int nq = e.H * e.D, nk = e.G * e.D;
      part = n < nq ? 0 : n < nq + nk ? 1 : 2;
      const int i = n - (part == 0 ? 0 : part == 1 ? nq : nq + nk), size = part == 2 ? e.Dv : e.D;
      head = i / size;
      d = i - head * size;
    } else if constexpr (EPI == kLatent) {  // query, projected down
      const MmLatent& e = p.lat;
      const int hd = e.D + e.rot;
      part = n >= e.H * hd;
      if (part) {
        d = n - e.H * hd;
      } else {
        head = n / hd;
        d = n - head * hd;
      }
    }
  }
};

template <typename T>
__device__ __forceinline__ T* page_at(const MmQkv& e, void* pool, int entry, int head) {
  const int page = e.table[(size_t)entry + (size_t)head * e.max_tiles];
  return page >= 0 && page < e.num_pages
             ? reinterpret_cast<T*>(static_cast<char*>(pool) + (size_t)page * e.page_stride)
             : nullptr;
}

// Where a column pair of a row goes, and what it still needs: found before the
// sums are there, so the loads behind it (page, angle, assignment) overlap the
// weight stream.
template <typename T, int EPI>
struct Target {
  History<EPI> past;
  void* p0 = nullptr;  // NULL: nothing to write
  void* p1 = nullptr;  // the second column's place where it is not next to the first
  float cs = 1.f, sn = 0.f;  // rotation; kGroupOut: cs is the weight

  template <bool LOOKED_UP = false>
  __device__ __forceinline__ void find(const KernelArgs& p, const Block<T>& b, const RowOf<EPI>& r,
                                       const ColOf<EPI>& c) {
    const int m = r.m, n = c.n;
    if (m < 0 || n < 0) return;
    if constexpr (EPI == kStore) {
      float* d = stored_to(p) + (size_t)m * p.a.ldc + n;
      p0 = d;
      p1 = n + 1 < b.N ? d + 1 : nullptr;
    } else if constexpr (EPI == kGroupIn) {
      T* d = static_cast<T*>(b.shared ? p.g.act_shared : p.g.act);
      p0 = d + (size_t)m * (b.shared ? p.g.lds : p.g.lda) + (n >> 1);
    } else if constexpr (EPI == kGroupOut) {
      RowOf<EPI> at = r;
      if constexpr (!LOOKED_UP) at.look_up(p, b);
      cs = at.weight;
      float* d = p.g.out + (size_t)at.out * p.g.ldo + n;
      p0 = d;
      p1 = n + 1 < b.N ? d + 1 : nullptr;
    } else if constexpr (EPI == kSplit) {
      const MmSplit& e = p.split;
      if (n < e.n_t) p0 = static_cast<T*>(e.t) + (size_t)m * e.ldt + n;
      else p0 = e.f + (size_t)m * e.ldf + (n - e.n_t);
    } else if constexpr (EPI == kGlu) {
      p0 = static_cast<T*>(p.split.t) + (size_t)m * p.split.ldt + (n >> 1);
    } else if constexpr (EPI == kSoftplus) {
      p0 = p.a.C + (size_t)m * p.a.ldc + n;
      cs = p.bias[n];
      sn = p.bias[n + 1];
    } else if constexpr (EPI == kHeads) {
      const MmHeads& e = p.heads;
      const int row = e.rows ? e.rows[m] : m;
      T* d = static_cast<T*>(e.C) + (size_t)row * e.ldc + (size_t)blockIdx.z * e.c_head + n;
      p0 = d;
      p1 = n + 1 < b.N ? d + 1 : nullptr;
    } else if constexpr (EPI == kLatent) {
      const MmLatent& e = p.lat;
      const bool turned = !c.part && c.d >= e.D;
      T* q = static_cast<T*>(e.q) + ((size_t)m * e.H + c.head) * e.ldq + c.d;
      float* down = e.down + (size_t)m * e.ldd + c.d;
      p0 = c.part ? static_cast<void*>(down) : static_cast<void*>(q);
      if (turned) {
        const float2 t = e.turn[(size_t)m * (e.rot >> 1) + ((c.d - e.D) >> 1)];
        cs = t.x;
        sn = t.y;
        p1 = static_cast<T*>(e.q_lat) + ((size_t)m * e.H + c.head) * e.ld_lat + e.lat_rot + (c.d - e.D);
      }
    } else if constexpr (EPI == kConv) {
      const MmConv& e = p.conv;
      if (n >= e.gate) {
        p0 = static_cast<T*>(e.z) + (size_t)m * e.ldz + (n - e.gate);
        return;
      }
      p0 = static_cast<T*>(e.x) + (size_t)m * e.ldx + n;
      T* h = static_cast<T*>(e.history) + (size_t)e.slot[m] * (e.taps - 1) * e.ldw + n;
      p1 = h;
      const int pos = e.pos[m];
#pragma unroll
      for (int k = 0; k < kMmConvTaps; ++k) {
        float2 w = {0.f, 0.f};
        if (k < e.taps) w = *reinterpret_cast<const float2*>(e.w + (size_t)k * e.ldw + n);
        past.w[0][k] = w.x;
        past.w[1][k] = w.y;
        if (k == kMmConvTaps - 1) break;
#pragma unroll
        for (int j = 0; j < 2; ++j)
          past.v[j][k] = k < e.taps - 1 && pos >= e.taps - 1 - k ? (float)h[(size_t)k * e.ldw + j] : 0.f;
      }
      past.bias[0] = e.bias[n];
      past.bias[1] = e.bias[n + 1];
    } else {
      const MmQkv& e = p.q;
      if (c.part == 0) {
        turn(e, m, c.d);
        p0 = static_cast<T*>(e.q) + ((size_t)m * e.H + c.head) * e.Dp + c.d;
        return;
      }
      if (r.entry < 0) return;
      if (c.part == 1) {
        turn(e, m, c.d);
        T* page = page_at<T>(e, e.k_pool, r.entry, c.head);
        if (page) p0 = page + (size_t)r.at * e.Dp + c.d;
        return;
      }
      const int slot = v_page_slot(r.at, Kind<T>::BF16);
      T* page = page_at<T>(e, e.v_pool, r.entry, c.head);
      if (page) p0 = page + (size_t)c.d * kPageTokens + slot;
      if (c.d + 1 < e.Dv) {
        if (page) p1 = page + (size_t)(c.d + 1) * kPageTokens + slot;
      } else if (c.head + 1 < e.G) {  // (not the second half of the last pair)
        page = page_at<T>(e, e.v_pool, r.entry, c.head + 1);
        if (page) p1 = page + slot;
      }
    }
  }

  __device__ __forceinline__ void put(const KernelArgs& p, const Block<T>& b, int n, float v0,
                                      float v1) const {
    if constexpr (EPI == kStore || EPI == kGroupOut) {
      if constexpr (EPI == kGroupOut) {
        v0 *= cs;
        v1 *= cs;
      } else if (p.a.softcap > 0.f) {
        v0 = p.a.softcap * tanhf(v0 / p.a.softcap);
        v1 = p.a.softcap * tanhf(v1 / p.a.softcap);
      }
      if (p0) *static_cast<float*>(p0) = v0;
      if (p1) *static_cast<float*>(p1) = v1;
    } else if constexpr (EPI == kGroupIn || EPI == kGlu) {
      if (p0) *static_cast<T*>(p0) = (T)glu(v0, v1, b.glu);
    } else if constexpr (EPI == kSplit) {
      if (!p0) return;
      if (n < p.split.n_t) put_pair(static_cast<T*>(p0), v0, v1);
      else put_pair(static_cast<float*>(p0), v0, v1);
    } else if constexpr (EPI == kSoftplus) {
      if (p0) put_pair(static_cast<float*>(p0), softplus(v0 + cs), softplus(v1 + sn));
    } else if constexpr (EPI == kHeads) {
      if (p0) *static_cast<T*>(p0) = (T)v0;
      if (p1) *static_cast<T*>(p1) = (T)v1;
    } else if constexpr (EPI == kLatent) {
      if (!p0) return;
      if (n >= p.lat.H * (p.lat.D + p.lat.rot)) {
        put_pair(static_cast<float*>(p0), v0, v1);
      } else {
        const float t0 = v0 * cs - v1 * sn, t1 = v1 * cs + v0 * sn;
        put_pair(static_cast<T*>(p0), t0, t1);
        if (p1) put_pair(static_cast<T*>(p1), t0, t1);
      }
    } else if constexpr (EPI == kConv) {
      if (!p0) return;
      if (!p1) {
        put_pair(static_cast<T*>(p0), v0, v1);
        return;
      }
      const MmConv& e = p.conv;
      const float now[2] = {(float)(T)v0, (float)(T)v1};
      float o[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        float s = past.bias[j];
#pragma unroll
        for (int k = 0; k < kMmConvTaps; ++k) {
          if (k < e.taps - 1 && k < kMmConvTaps - 1) s += past.v[j][k] * past.w[j][k];
          if (k == e.taps - 1) s += now[j] * past.w[j][k];
        }
        o[j] = s / (1.f + expf(-s));
      }
      put_pair(static_cast<T*>(p0), o[0], o[1]);
      T* h = static_cast<T*>(p1);
#pragma unroll
      for (int k = 0; k < kMmConvTaps - 1; ++k) {
        if (k + 2 < e.taps && k + 2 < kMmConvTaps)
          put_pair(h + (size_t)k * e.ldw, past.v[0][k + 1], past.v[1][k + 1]);
        else if (k + 2 == e.taps)
          put_pair(h + (size_t)k * e.ldw, now[0], now[1]);
      }
    } else {
      if (n < (p.q.H + p.q.G) * p.q.D) {
        if (p0) put_pair(static_cast<T*>(p0), v0 * cs - v1 * sn, v1 * cs + v0 * sn);
      } else {
        if (p0) *static_cast<T*>(p0) = (T)v0;
        if (p1) *static_cast<T*>(p1) = (T)v1;
      }
    }
  }

 private:
  __device__ __forceinline__ void turn(const MmQkv& e, int m, int d) {
    if (d >= e.rot) return;
    const float2 t = e.turn[(size_t)m * (e.rot >> 1) + (d >> 1)];
    cs = t.x;
    sn = t.y;
  }
};

template <typename T>
__device__ __forceinline__ void put_eight(T* p, const float (&v)[8]) {
  constexpr int E = 16 / sizeof(T);
  typedef T chunk_t __attribute__((ext_vector_type(E)));
#pragma unroll
  for (int k = 0; k < 8; k += E) {
    chunk_t o;
#pragma unroll
    for (int e = 0; e < E; ++e) o[e] = (T)v[k + e];
    // half of fp32's 32 bytes at a time would reach memory as parts of lines
    if constexpr (E == 8) store_through(p + k, __builtin_bit_cast(u32x4, o));
    else *reinterpret_cast<chunk_t*>(p + k) = o;
  }
}
template <typename T>
__device__ __forceinline__ void put_four(T* p, f32x4 v) {
  typedef T four_t __attribute__((ext_vector_type(4)));
  four_t o;
#pragma unroll
  for (int k = 0; k < 4; ++k) o[k] = (T)v[k];
  if constexpr (sizeof(T) == 2) store_through(p, __builtin_bit_cast(u32x2, o));
  else store_through(p, __builtin_bit_cast(u32x4, o));
}
// rows of ld elements that all start at 16 bytes
template <typename T>
__device__ __forceinline__ bool whole(const void* p, size_t ld) {
  return ((reinterpret_cast<uintptr_t>(p) | ld * sizeof(T)) & 15) == 0;
}

// Where columns n .. n + 7 (n a multiple of 8) of a row go in stores of 16 bytes, and
// what they still need.  ok: sizes and places allow it; else they go pair by pair.
template <typename T, int EPI>
struct Eight {
  bool ok = false;
  void* p0 = nullptr;  // NULL: nothing to write
  void* p1 = nullptr;
  bool turned = false;
  float2 turn[4];

  __device__ __forceinline__ void find(const KernelArgs& p, const Block<T>& b, const RowOf<EPI>& r,
                                       const ColOf<EPI>& c) {
    const int m = r.m, n = c.n;
    ok = true;
    if (m < 0 || n < 0) return;
    ok = n + 8 <= b.N;
    if constexpr (EPI == kGroupIn) {
      const int ld = b.shared ? p.g.lds : p.g.lda;
      T* d = static_cast<T*>(b.shared ? p.g.act_shared : p.g.act);
      ok = ok && whole<T>(d, ld);
      p0 = d + (size_t)m * ld + (n >> 1);
    } else if constexpr (EPI == kGlu) {
      ok = ok && whole<T>(p.split.t, p.split.ldt);
      p0 = static_cast<T*>(p.split.t) + (size_t)m * p.split.ldt + (n >> 1);
    } else if constexpr (EPI == kHeads) {
      const MmHeads& e = p.heads;
      ok = ok && whole<T>(e.C, e.ldc) && whole<T>(nullptr, e.c_head);
      const int row = e.rows ? e.rows[m] : m;
      p0 = static_cast<T*>(e.C) + (size_t)row * e.ldc + (size_t)blockIdx.z * e.c_head + n;
    } else if constexpr (EPI == kLatent) {
      const MmLatent& e = p.lat;
      ok = ok && ((e.D | e.rot) & 7) == 0 && whole<T>(e.q, e.ldq) && whole<float>(e.down, e.ldd);
      if (c.part) {
        p1 = e.down + (size_t)m * e.ldd + c.d;
        return;
      }
      p0 = static_cast<T*>(e.q) + ((size_t)m * e.H + c.head) * e.ldq + c.d;
      if (c.d < e.D) return;
      ok = ok && whole<T>(e.q_lat, e.ld_lat) && whole<T>(nullptr, e.lat_rot);
      p1 = static_cast<T*>(e.q_lat) + ((size_t)m * e.H + c.head) * e.ld_lat + e.lat_rot + (c.d - e.D);
      if (ok) angles(e.turn + (size_t)m * (e.rot >> 1) + ((c.d - e.D) >> 1));
    } else if constexpr (EPI == kQkv || EPI == kExpand) {
      const MmQkv& e = p.q;
      ok = ok && c.part < 2 && ((e.D | e.rot | e.Dp) & 7) == 0;
      if (!ok) return;
      if (c.d < e.rot) angles(e.turn + (size_t)m * (e.rot >> 1) + (c.d >> 1));
      if (c.part == 0) {
        p0 = static_cast<T*>(e.q) + ((size_t)m * e.H + c.head) * e.Dp + c.d;
      } else if (r.entry >= 0) {
        T* page = page_at<T>(e, e.k_pool, r.entry, c.head);
        if (page) p0 = page + (size_t)r.at * e.Dp + c.d;
      }
    } else {
      ok = false;
    }
  }

  __device__ __forceinline__ void put(const KernelArgs& p, const Block<T>& b, int n, float (&v)[8]) const {
    if constexpr (EPI == kGroupIn || EPI == kGlu) {
      if (!p0) return;
      typedef T half_t __attribute__((ext_vector_type(4)));
      half_t o;
#pragma unroll
      for (int k = 0; k < 4; ++k) o[k] = (T)glu(v[2 * k], v[2 * k + 1], b.glu);
      *static_cast<half_t*>(p0) = o;
    } else if constexpr (EPI == kHeads) {
      if (p0) put_eight(static_cast<T*>(p0), v);
    } else if constexpr (EPI == kLatent) {
      if (!p0) {
        if (p1) put_eight(static_cast<float*>(p1), v);
        return;
      }
      rotate(v);
      put_eight(static_cast<T*>(p0), v);
      if (p1) put_eight(static_cast<T*>(p1), v);
    } else if constexpr (EPI == kQkv || EPI == kExpand) {
      if (!p0) return;
      rotate(v);
      put_eight(static_cast<T*>(p0), v);
    }
  }

 private:
  __device__ __forceinline__ void angles(const float2* t) {
    turned = true;
#pragma unroll
    for (int k = 0; k < 4; ++k) turn[k] = t[k];
  }
  __device__ __forceinline__ void rotate(float (&v)[8]) const {
    if (!turned) return;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float v0 = v[2 * k], v1 = v[2 * k + 1];
      v[2 * k] = v0 * turn[k].x - v1 * turn[k].y;
      v[2 * k + 1] = v1 * turn[k].x + v0 * turn[k].y;
    }
  }
};

// Rows of a block that begin a sequence's: found before the product, for the value columns.
template <int ROWS>
struct Starts {
  unsigned long long at[ROWS / 64];
  int rows = 0, sequences = 0;

  template <typename T>
  __device__ __forceinline__ Starts(const MmQkv& e, const Block<T>& b) {
    rows = min(ROWS, b.M - b.m0);
#pragma unroll
    for (int h = 0; h < ROWS / 64; ++h) {
      const int r = 64 * h + lane_id();
      at[h] = __ballot(r < rows && (r == 0 || e.slot[b.m0 + r] != e.slot[b.m0 + r - 1]));
      sequences += __popcll(at[h]);
    }
  }
};

struct NoStarts {
  template <typename T>
  __device__ __forceinline__ NoStarts(const MmQkv&, const Block<T>&) {}
};

// Value columns [c0, c1) of a block's sums: they lie token by token in their pages.
// Rows of a few sequences: four tokens of a page that lie together are one store,
// sixteen lanes a page's line.  A thread's tokens stay the same over its columns, whose pages
// are looked up together and before the stores: one by one, each look-up waited for the
// store before it (2011 x 4096 x 512, half of it values: 37 us, now 29.5).
// Rows of many: a row per thread, so that its page is looked up once for the columns it takes.
template <typename T, int EPI, int ROWS, int COLS, int STRIDE, int THREADS>
__device__ __forceinline__ void emit_values(const KernelArgs& p, const Block<T>& b, const float* sums,
                                            const Starts<ROWS>& starts, int first_col, int c0, int c1) {
  const MmQkv& e = p.q;
  if (starts.rows <= 0 || c0 >= c1) return;
  if (starts.sequences > 4) {
    const int r = threadIdx.x % ROWS;
    const RowOf<EPI> row(p, b, b.m0 + r);
    if (row.m < 0 || row.entry < 0) return;
#pragma unroll 4
    for (int col = c0 + threadIdx.x / ROWS; col < c1; col += THREADS / ROWS) {
      const ColOf<EPI> c(p, b, col);
      T* page = page_at<T>(e, e.v_pool, row.entry, c.head);
      if (page)
        page[(size_t)c.d * kPageTokens + v_page_slot(row.at, Kind<T>::BF16)] =
            (T)sums[r * STRIDE + col - first_col];
    }
    return;
  }
  typedef T quad_t __attribute__((ext_vector_type(4)));
  constexpr int ACROSS = THREADS / 16, PER = COLS / ACROSS;
  static_assert(COLS % ACROSS == 0);
#pragma unroll
  for (int h = 0; h < ROWS / 64; ++h) {
    for (unsigned long long left = starts.at[h]; left; left &= left - 1) {
      const int s0 = 64 * h + __ffsll(left) - 1;  // the sequence's rows: [s0, s1)
      const unsigned long long after = left & (left - 1);
      int s1 = after ? 64 * h + __ffsll(after) - 1 : starts.rows;
      if (!after && h + 1 < ROWS / 64 && starts.at[ROWS / 64 - 1])
        s1 = 64 * (h + 1) + __ffsll(starts.at[ROWS / 64 - 1]) - 1;
      const int pos0 = e.pos[b.m0 + s0], slot = e.slot[b.m0 + s0], off = pos0 & 3;
      for (int r0 = s0 + 4 * (threadIdx.x & 15) - off; r0 - 4 * (int)(threadIdx.x & 15) < s1; r0 += 64) {
        const int pos = pos0 + r0 - s0, tile = pos / kPageTokens;
        const bool here = r0 < s1 && tile < e.max_tiles;
        T* to[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j) {
          const int col = c0 + threadIdx.x / 16 + j * ACROSS;
          to[j] = nullptr;
          if (!here || col >= c1) continue;
          const ColOf<EPI> c(p, b, col);
          T* page = page_at<T>(e, e.v_pool, slot * e.G * e.max_tiles + tile, c.head);
          if (page) to[j] = page + (size_t)c.d * kPageTokens + v_page_slot(pos % kPageTokens, Kind<T>::BF16);
        }
#pragma unroll
        for (int j = 0; j < PER; ++j) {
          if (!to[j]) continue;
          const float* v = sums + r0 * STRIDE + (c0 + (int)threadIdx.x / 16 + j * ACROSS - first_col);
          if (r0 >= s0 && r0 + 4 <= s1) {
            quad_t o;
#pragma unroll
            for (int k = 0; k < 4; ++k) o[k] = (T)v[k * STRIDE];
            *reinterpret_cast<quad_t*>(to[j]) = o;
          } else {
#pragma unroll
            for (int k = 0; k < 4; ++k)
              if (r0 + k >= s0 && r0 + k < s1) to[j][k] = (T)v[k * STRIDE];
          }
        }
      }
    }
  }
}

// Columns of a row that a thread finishes: 16 bytes of fp32 or of the element type, which
// sixteen of (gate, up) make; pairs where a channel's history comes along.
template <int EPI>
constexpr int columns_each(int rows, int cols) {
  return EPI == kConv ? 2
         : EPI == kStore || EPI == kGroupOut || EPI == kSoftplus || EPI == kSplit ? 4
         : (EPI == kGroupIn || EPI == kGlu) && 1024 / cols <= rows ? 16
                                                                    : 8;
}

// A wave's ROWS x COLS finished sums, row by row in LDS -> the epilogue.  Stores are whole
// lines of a row, 64 columns of it by neighbouring lanes (straight from the accumulators a
// pair of columns a lane: bf16 2048 x 12288 x 2048 with fp32 results 101.5 us, now 95;
// 2011 rows of gate and up with their activation 108, now 105; the products alone 77), and a thread's rows
// have one set of columns, whose bias, head and place are found once.  All that is loaded
// is loaded before the first store: a load behind stores is waited for together with them.
template <typename T, int EPI, int ROWS, int COLS, int STRIDE, typename B>
__device__ __forceinline__ void emit_wave(const KernelArgs& p, const B& b, const float* sums,
                                          const RowOf<EPI>& row, int m0, int n0) {
  constexpr int E = columns_each<EPI>(ROWS, COLS), ACROSS = COLS / E, STEP = 64 / ACROSS, PER = ROWS / STEP;
  static_assert(64 % ACROSS == 0 && PER >= 1);
  const int lane = lane_id(), r0 = lane / ACROSS, c0 = lane % ACROSS * E, n = n0 + c0;
  int end = b.N;  // of the columns that go by rows; the others are values
  if constexpr (RowOf<EPI>::PAGED) end = min(b.N, (p.q.H + p.q.G) * p.q.D);
  RowOf<EPI> r[EPI == kConv ? 1 : PER];
  if constexpr (EPI != kConv) {
#pragma unroll
    for (int i = 0; i < PER; ++i) r[i] = row.from(r0 + i * STEP);
  }
  if (n >= end) return;
  sums += r0 * STRIDE + c0;
  if constexpr (EPI == kConv) {
    constexpr int BATCH = PER < 4 ? PER : 4;
    const ColOf<EPI> c(p, b, n);
#pragma unroll 1
    for (int i0 = 0; i0 < PER; i0 += BATCH) {
      Target<T, EPI> t[BATCH];
#pragma unroll
      for (int i = 0; i < BATCH; ++i) t[i].find(p, b, RowOf<EPI>(p, b, m0 + r0 + (i0 + i) * STEP), c);
#pragma unroll
      for (int i = 0; i < BATCH; ++i) {
        const float* s = sums + (i0 + i) * STEP * STRIDE;
        t[i].put(p, b, n, s[0], s[1]);
      }
    }
    return;
  }
  if constexpr (EPI == kSplit) {
    const MmSplit& e = p.split;
    const bool left = n < e.n_t, four = (e.n_t & 3) == 0 && n + 4 <= b.N;
    const bool vec = four && (left ? ((reinterpret_cast<uintptr_t>(e.t) | e.ldt * sizeof(T)) &
                                      (4 * sizeof(T) - 1)) == 0
                                   : whole<float>(e.f, e.ldf));
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int m = r[i].m;
      if (m < 0) continue;
      const f32x4 v = *reinterpret_cast<const f32x4*>(sums + i * STEP * STRIDE);
      T* t = static_cast<T*>(e.t) + (size_t)m * e.ldt + n;
      float* f = e.f + (size_t)m * e.ldf + (n - e.n_t);
      if (!vec) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (n + k >= b.N) break;
          if (n + k < e.n_t) t[k] = (T)v[k];
          else f[k] = v[k];
        }
      } else if (!left) {
        store_through(f, __builtin_bit_cast(u32x4, v));
      } else {
        put_four(t, v);
      }
    }
  } else if constexpr (E == 4) {
    float* C = EPI == kGroupOut ? p.g.out : EPI == kStore ? stored_to(p) : p.a.C;
    const size_t ldc = EPI == kGroupOut ? p.g.ldo : p.a.ldc;
    const bool vec = whole<float>(C, ldc) && n + 4 <= b.N;
    float bias[4];
    if constexpr (EPI == kSoftplus)
#pragma unroll
      for (int k = 0; k < 4; ++k) bias[k] = p.bias[min(n + k, b.N - 1)];
    const auto put = [&](int row, f32x4 v) {
      float* to = C + row * ldc + n;
      if (vec) {
        store_through(to, __builtin_bit_cast(u32x4, v));
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (n + k < b.N) to[k] = v[k];
      }
    };
    if (EPI == kStore && p.a.softcap > 0.f) {  // a model's head: apart, tanhf's code is long
#pragma unroll 1
      for (int i = 0; i < PER; ++i) {
        const int row = m0 + r0 + i * STEP;
        if (row >= b.M) break;
        f32x4 v = *reinterpret_cast<const f32x4*>(sums + i * STEP * STRIDE);
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = p.a.softcap * tanhf(v[k] / p.a.softcap);
        put(row, v);
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (r[i].m < 0) continue;
      f32x4 v = *reinterpret_cast<const f32x4*>(sums + i * STEP * STRIDE);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if constexpr (EPI == kGroupOut) v[k] *= r[i].weight;
        else if constexpr (EPI == kSoftplus) v[k] = softplus(v[k] + bias[k]);
      }
      put(EPI == kGroupOut ? r[i].out : r[i].m, v);
    }
  } else if constexpr (E == 16) {  // gate and up
    const size_t ld = EPI == kGlu ? p.split.ldt : b.shared ? p.g.lds : p.g.lda;
    T* act = static_cast<T*>(EPI == kGlu ? p.split.t : b.shared ? p.g.act_shared : p.g.act);
    const bool vec = whole<T>(act, ld) && n + 16 <= b.N;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (r[i].m < 0) continue;
      T* to = act + r[i].m * ld + (n >> 1);
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; k += 2) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(sums + i * STEP * STRIDE + 2 * k);
        v[k] = glu(x[0], x[1], b.glu);
        v[k + 1] = glu(x[2], x[3], b.glu);
      }
      if (vec) {
        put_eight(to, v);
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (n + 2 * k < b.N) to[k] = (T)v[k];
      }
    }
  } else {
    const ColOf<EPI> c(p, b, n);
    Eight<T, EPI> t[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) t[i].find(p, b, r[i], c);
    bool rest = false;  // rows that go pair by pair
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (r[i].m < 0) continue;
      const float* s = sums + i * STEP * STRIDE;
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; k += 4) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(s + k);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[k + e] = x[e];
      }
      if (t[i].ok) t[i].put(p, b, n, v);
      else rest = true;
    }
    if (!rest) return;
#pragma unroll 1
    for (int i = 0; i < PER; ++i) {
      const RowOf<EPI> at(p, b, m0 + r0 + i * STEP);
      Eight<T, EPI> e;
      e.find(p, b, at, c);
      if (at.m < 0 || e.ok) continue;
      const float* s = sums + i * STEP * STRIDE;
#pragma unroll 1
      for (int k = 0; k < 8 && n + k < end; k += 2) {
        Target<T, EPI> g;
        g.find(p, b, at, ColOf<EPI>(p, b, n + k));
        g.put(p, b, n + k, s[k], s[k + 1]);
      }
    }
  }
}

// Decode rows (and short grouped tiles): a block owns 16 MT rows x 16 NT columns
// and its WK waves split K, adding through LDS in a fixed order.  K is summed in PARTS parts,
// PARTS / WK of them by a wave one after the other: a wave that streams more of K sums it no
// further in one piece, and the bits do not depend on how many waves there are.
template <typename T, int EPI, int MT, int NT, int WK, int PARTS, bool SOME = false>
__global__ __launch_bounds__(64 * WK, MT * NT == 1 ? 4 : 2) void mm_stream_kernel(KernelArgs p) {
  if constexpr (EPI == kGroupIn || EPI == kGroupOut)
    if ((int)blockIdx.y >= *p.g.n_tiles) return;
  constexpr int U = MT * NT >= 4 ? 2 : 4;  // k-steps per load batch
  const int lane = lane_id();
  const int w = wave_id_uniform();
  const BlockOf<T, SOME> b{block_of<T, EPI>(p, 16 * MT, blockIdx.y)};
  const int ntiles = (b.N + 15) >> 4;
  const int nt0 = (int)blockIdx.x * NT;
  if (nt0 >= ntiles) return;  // (groups differ in width)

  const char* ap[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) ap[i] = a_row<T, EPI>(p, b, b.m0 + 16 * i + (lane & 15)) + 16 * (lane >> 4);
  const char* bp[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
    bp[j] = b.W + min(nt0 + j, ntiles - 1) * b.w_tile + lane * 16;

  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Neighbouring blocks start at different k ranges, so they do not all pull
  // the same A lines at once.
  const int wr = (w + (int)blockIdx.x) % WK;
  const int ks0 = wr * b.KS / WK, ks1 = (wr + 1) * b.KS / WK;
  constexpr int OWN = PARTS / WK;
  static_assert(PARTS % WK == 0, "whole parts a wave");
  __shared__ float red[PARTS][MT * NT][4][64];
  int part = wr * OWN;  // the one being summed
  auto put_part = [&] {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[part][i * NT + j][r][lane] = acc[i][j][r];
  };
  auto end_parts = [&](int k) {  // (a wave's last part ends with the wave)
    while (part < wr * OWN + OWN - 1 && (part + 1) * b.KS / PARTS <= k) {
      put_part();
      ++part;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  struct Batch {
    u32x4 a[U][MT], b[U][NT];
  };
  const bool nt_load = p.a.w_nt;
  auto load = [&](Batch& x, int ks) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = ks + u;
      if (k < ks1) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const u32x4* src = reinterpret_cast<const u32x4*>(bp[j] + (size_t)k * 1024);
          x.b[u][j] = nt_load ? __builtin_nontemporal_load(src) : *src;
        }
#pragma unroll
        for (int i = 0; i < MT; ++i)
          x.a[u][i] = *reinterpret_cast<const u32x4*>(ap[i] + (size_t)k * 64);
      } else {
#pragma unroll
        for (int j = 0; j < NT; ++j) x.b[u][j] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
        for (int i = 0; i < MT; ++i) x.a[u][i] = u32x4{0u, 0u, 0u, 0u};
      }
    }
  };
  auto mul = [&](const Batch& x, int ks) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if constexpr (OWN > 1) end_parts(ks + u);
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = Kind<T>::mma(x.a[u][i], x.b[u][j], acc[i][j]);
    }
  };
  // thread t finishes column pairs t, t + THREADS, ...: 8 pairs a row, 128 a tile
  constexpr int PAIRS = MT * NT * 128, THREADS = 64 * WK, EPT = (PAIRS + THREADS - 1) / THREADS;
  Target<T, EPI> target[EPT];
  Batch x, y;
  if (ks0 < ks1) load(x, ks0);
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    const int pr = threadIdx.x + e * THREADS, t = pr >> 7;
    if (pr < PAIRS)
      target[e].find(p, b, RowOf<EPI>(p, b, b.m0 + 16 * (t / NT) + ((pr >> 3) & 15)),
                     ColOf<EPI>(p, b, (nt0 + t % NT) * 16 + (pr & 7) * 2));
  }
  if (ks0 < ks1) {
    for (int ks = ks0;;) {
      if (ks + U < ks1) load(y, ks + U);
      mul(x, ks);
      ks += U;
      if (ks >= ks1) break;
      if (ks + U < ks1) load(x, ks + U);
      mul(y, ks);
      ks += U;
      if (ks >= ks1) break;
    }
  }

  if constexpr (OWN > 1) end_parts(b.KS);
  put_part();
  __syncthreads();
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    const int pr = threadIdx.x + e * THREADS;
    if (pr >= PAIRS) break;
    const int t = pr >> 7, row = (pr >> 3) & 15, col = (pr & 7) * 2;
    float2 s = {0.f, 0.f};
#pragma unroll
    for (int k = 0; k < PARTS; ++k) {
      const float2 v = *reinterpret_cast<const float2*>(&red[k][t][row & 3][(row >> 2) * 16 + col]);
      s.x += v.x;
      s.y += v.y;
    }
    target[e].put(p, b, (nt0 + t % NT) * 16 + col, s.x, s.y);
  }
}

// blocks of 16 NB columns in n columns
__host__ __device__ __forceinline__ int group_across(int n, int NB) { return (n + 16 * NB - 1) / (16 * NB); }

// The tile of this workgroup; false: there is none for it.
template <int EPI, int NB>
__device__ __forceinline__ bool tile_of(const KernelArgs& p, TileAt& tile) {
  int id = blockIdx.y * gridDim.x + blockIdx.x;
  if constexpr (EPI == kGroupIn || EPI == kGroupOut) {
    // the shared expert's tiles (the last of the list, the most columns or k-steps)
    // go first; each kind is dealt out over the XCDs by itself
    const int across = group_across(p.g.shared_n, NB), shared = p.g.shared_tiles * across;
    const int routed = *p.g.n_tiles - p.g.shared_tiles;
    if (id < shared) {
      tile = xcd_tile(id, across, p.g.shared_tiles);
      tile.y += routed;
    } else {
      id -= shared;
      const int nx = group_across(p.g.routed_n, NB);
      if (id >= routed * nx) return false;
      tile = xcd_tile(id, nx, routed);
    }
  } else {
    tile = xcd_tile(id, gridDim.x, gridDim.y);
  }
  return true;
}

// A block of 16 MB rows x 16 NB columns, WM x WN waves (block_product.hpp).  Two waves a SIMD in
// the bounds, for the blocks of four waves (gemm_impl.hpp, gemm_block_kernel).
template <typename T, int EPI, int MB, int NB, int WM, int WN, int ST, bool SOME = false>
__global__ __launch_bounds__(64 * WM * WN, 2) void mm_block_kernel(KernelArgs p) {
  constexpr int MT = MB / WM, NT = NB / WN;
  __shared__ u32x4 lds[ST][2 * (MB + NB)][64];
  TileAt tile;
  if (!tile_of<EPI, NB>(p, tile)) return;
  const int lane = lane_id();
  const int w = wave_id_uniform();
  const BlockOf<T, SOME> b{block_of<T, EPI>(p, 16 * MB, tile.y)};
  const int ntiles = (b.N + 15) >> 4;
  const int nt0 = tile.x * NB, KS = b.KS;
  const int wm = w / WN, wn = w % WN;
  const int m0 = 16 * wm * MT, n0 = 16 * wn * NT;
  RowOf<EPI> row(p, b, b.m0 + m0 + lane % (16 * MT));
  if (row.m >= 0) row.look_up(p, b);
  constexpr bool VALUES = RowOf<EPI>::PAGED && !SOME;
  std::conditional_t<VALUES, Starts<16 * MB>, NoStarts> starts(p.q, b);
  f32x4 acc[MT][NT];
  block_product<false, !Kind<T>::BF16, MB, NB, WM, WN, ST>(
      lds, acc, KS, b.m0 + 16 * wm * MT < b.M,
      [&](int r) { return a_row<T, EPI>(p, b, b.m0 + r); },
      [&](int t) { return b.W + min(nt0 + t, ntiles - 1) * b.w_tile; },
      [](u32x4 x, u32x4 y, f32x4 c) { return Kind<T>::mma(x, y, c); });
  // (block_product has read all of LDS before its last barrier)
  constexpr int STRIDE = 16 * NB + 4;
  static_assert(sizeof(lds) >= sizeof(float) * 16 * MB * STRIDE);
  float* sums = reinterpret_cast<float*>(&lds[0][0][0]);
  spread_sums<STRIDE>(acc, sums, m0, n0);
  emit_wave<T, EPI, 16 * MT, 16 * NT, STRIDE>(p, b, sums + m0 * STRIDE + n0, row, b.m0 + m0, 16 * nt0 + n0);
  if constexpr (VALUES) {
    const int first = max(16 * nt0, (p.q.H + p.q.G) * p.q.D), last = min(16 * (nt0 + NB), b.N);
    if (first >= last) return;
    __syncthreads();
    emit_values<T, EPI, 16 * MB, 16 * NB, STRIDE, 64 * WM * WN>(p, b, sums, starts, 16 * nt0, first, last);
  }
}

// Epilogues that strips take: a wave alone on its SIMD waits for every load and transcendental of
// the others (2011 x 4096 x 512 to pages 28.7 us by blocks, 44 by strips; x 4096 x 128 with softplus
// 16.4, 22; queries to be turned 38.4, 40.9).
template <typename T, int EPI>
constexpr bool by_strips() {
  return Kind<T>::BF16 && (EPI == kStore || EPI == kSplit || EPI == kGlu || EPI == kHeads || EPI == kGroupIn ||
                           EPI == kGroupOut);
}

// A block of 16 MB rows x 16 NT WAVES columns by strips (block_product.hpp, strip_product).  A
// wave's sums leave a quarter of its rows at a time through its part of LDS, by one copy of the
// epilogue to which they are handed down: a launch finds its code in no cache (2011 x 2048 x 2048
// amid a model, a copy for each quarter 35 KB: 27.5 us; one, 12 KB: 20.4; blocks of eight waves
// 25.5).
template <typename T, int EPI, int MB, int NT, int WAVES, int ST, int AHEAD, bool SOME = false>
__global__ __launch_bounds__(64 * WAVES, 2) void mm_strip_kernel(KernelArgs p) {
  constexpr int NB = NT * WAVES, SR = MB / 4, STRIDE = 16 * NT + 4;
  __shared__ u32x4 lds[ST][2 * MB][64];
  static_assert(by_strips<T, EPI>() && sizeof(lds) >= sizeof(float) * WAVES * 16 * SR * STRIDE);
  TileAt tile;
  if (!tile_of<EPI, NB>(p, tile)) return;
  const int w = wave_id_uniform();
  const BlockOf<T, SOME> b{block_of<T, EPI>(p, 16 * MB, tile.y)};
  const int ntiles = (b.N + 15) >> 4, nt0 = tile.x * NB + w * NT, KS = b.KS;
  f32x4 acc[MB][NT];
  strip_product<MB, NT, WAVES, ST, AHEAD>(
      lds, acc, KS, [&](int r) { return a_row<T, EPI>(p, b, b.m0 + r); },
      [&](int j) { return b.W + min(nt0 + j, ntiles - 1) * b.w_tile; },
      [](u32x4 x, u32x4 y, f32x4 c) { return Kind<T>::mma(x, y, c); });
  if (16 * nt0 >= b.N) return;
  float* sums = reinterpret_cast<float*>(&lds[0][0][0]) + w * 16 * SR * STRIDE;
  strip_rows<SR>(acc, [&](int i0, const f32x4(&part)[SR][NT]) {
    const int m0 = b.m0 + 16 * i0;
    if (m0 >= b.M) return false;
    RowOf<EPI> row(p, b, m0 + lane_id() % (16 * SR));
    if (row.m >= 0) row.look_up(p, b);
    spread_sums<STRIDE>(part, sums, 0, 0);
    emit_wave<T, EPI, 16 * SR, 16 * NT, STRIDE>(p, b, sums, row, m0, 16 * nt0);
    return true;
  });
}

template <int EPI>
int heads_of(const KernelArgs& p) {  // and parts of K
  return EPI == kHeads ? p.heads.heads : EPI == kStore ? p.a.parts : 1;
}

template <typename T, int EPI, int MT, int NT, int WK = 8, int PARTS = WK>
hipError_t stream(const KernelArgs& p, int row_blocks, int N, hipStream_t st) {
  const dim3 grid(((N + 15) / 16 + NT - 1) / NT, row_blocks, heads_of<EPI>(p));
  const auto go = [&](void (*kernel)(KernelArgs)) {
    hipLaunchKernelGGL(kernel, grid, dim3(64 * WK), 0, st, p);
    return hipGetLastError();
  };
  if constexpr (some_rows<EPI>())
    if (p.a.rows) return go(mm_stream_kernel<T, EPI, MT, NT, WK, PARTS, true>);
  return go(mm_stream_kernel<T, EPI, MT, NT, WK, PARTS>);
}

template <int EPI>
dim3 block_grid(const KernelArgs& p, int row_blocks, int N, int NB) {
  if constexpr (EPI == kGroupIn || EPI == kGroupOut)
    return dim3((p.g.max_tiles - p.g.shared_tiles) * group_across(p.g.routed_n, NB) +
                p.g.shared_tiles * group_across(p.g.shared_n, NB));
  return dim3(group_across(N, NB), row_blocks, heads_of<EPI>(p));
}

template <typename T, int EPI, int MB, int NB, int WM, int WN, int ST>
hipError_t blocks(const KernelArgs& p, int row_blocks, int N, hipStream_t st) {
  const auto go = [&](void (*kernel)(KernelArgs)) {
    hipLaunchKernelGGL(kernel, block_grid<EPI>(p, row_blocks, N, NB), dim3(64 * WM * WN), 0, st, p);
    return hipGetLastError();
  };
  if constexpr (some_rows<EPI>())
    if (p.a.rows) return go(mm_block_kernel<T, EPI, MB, NB, WM, WN, ST, true>);
  return go(mm_block_kernel<T, EPI, MB, NB, WM, WN, ST>);
}

template <typename T, int EPI, int MB, int NT, int WAVES, int ST, int AHEAD>
hipError_t strips(const KernelArgs& p, int row_blocks, int N, hipStream_t st) {
  const auto go = [&](void (*kernel)(KernelArgs)) {
    hipLaunchKernelGGL(kernel, block_grid<EPI>(p, row_blocks, N, NT * WAVES), dim3(64 * WAVES), 0, st, p);
    return hipGetLastError();
  };
  if constexpr (some_rows<EPI>())
    if (p.a.rows) return go(mm_strip_kernel<T, EPI, MB, NT, WAVES, ST, AHEAD, true>);
  return go(mm_strip_kernel<T, EPI, MB, NT, WAVES, ST, AHEAD>);
}

// How a product runs, and about how long at K = 2048 (us; 0: not told), kFixedUs of it whatever K is.
struct Form {
  using Go = hipError_t (*)(const KernelArgs&, int, int, hipStream_t);
  Go go = nullptr;
  int row_blocks = 0;
  float us = 0.f;
};
constexpr float kFixedUs = 2.f;

// Rounds of stream blocks, priced by a block's column tiles and the rows it reads (128 column tiles, us of
// bf16 / fp32: 16 rows 4.7 / 8, 48 to 64 rows 5.5 / 12).
template <typename T>
inline float stream_us(int groups, float tiles) {
  return kFixedUs + (float)((groups + 255) / 256) * (Kind<T>::BF16 ? 1.8f : 4.5f) * tiles;
}

// A block form, the blocks of it a CU holds (by their LDS), and the time of a round of them at
// K = 2048 with one, two and three a CU (us, weights from memory).  A product takes the form
// whose rounds take least.  Two blocks of 64 x 128 a CU hide each other's first loads and last
// stores, so there are two depths of them: 2048 x 2560 28.7 us (four stages, one a CU: 33.8),
// 1000 x 2048 12.3 (three stages: 13.2).  2048 x 12288: 3 rounds of 128 x 256, 97 us with the
// activation (128 x 128: 119); 2048 x 2048: one round of 128 x 128, 17.1 us (128 x 256 leaves
// half the chip idle: 26.4); 700 x 2048: 64 x 128, 12.0 us (128 x 128: 17.3).  By strips 128 x 256
// and 128 x 128 where a CU has two of them (with weights and code from memory, two a CU, K 256 / 512 /
// 1024 / 2048 / 4096: 128 x 256 19.6 / 24.6 / 35.9 / 62.6 / 112 us, two rounds of blocks 20.8 / 28.4 / 40.6
// / 65.7 / 120; 128 x 128 11.0 / 15.0 / 21.5 / 34.6 / 67.4, blocks 13.1 / 17.2 / 25.4 / 40.7 / 70.2), and
// alone from K 1024 on (128 x 128 7.4 / 9.1 / 12.2 / 19.3 / 33.1, blocks 6.6 / 8.6 / 12.7 / 20.3 / 35.1).
// fp32 blocks are
// bound by the matrix cores and take the time of their area, the small ones, of which a CU
// holds several, the time between two rounds: 2048 x 2048: two rounds of 64 x 128, 140 us
// (128 x 128: 158); 700 x 6144: five of 64 x 64, 185 us (64 x 128: 207).  Of other K the order
// is nearly the same: over 65 to 2048 rows and 1024 to 12288 columns of bf16 the form so chosen is
// on average 0.1 to 0.3 % off the best from K 1024 to 8192, 0.8 % at 512, 2.3 % at 256.
template <typename T, int EPI>
Form block_form(const KernelArgs& p, int min_mb, int max_mb, int N) {
  Form best;
  const bool long_k = (EPI == kGroupIn || EPI == kGroupOut ? p.g.min_ks : EPI == kStore ? p.KS / p.a.parts : p.KS) >= 32;
  const auto consider = [&](int mb, int nb, int per, const float (&bf16)[3], float fp32,
                            Form::Go go, bool strip = false) {
    if (mb < min_mb || mb > max_mb) return;
    const int y = (p.a.M + 16 * mb - 1) / (16 * mb);
    const dim3 g = block_grid<EPI>(p, y, N, nb);
    const int groups = g.x * g.y * g.z;
    if (strip && groups <= 256 && !long_k) return;
    const float cost = Kind<T>::BF16 ? rounds_us(groups, per, bf16) : (float)((groups + 255) / 256) * fp32;
    if (best.go && cost >= best.us) return;
    best = Form{go, y, cost};
  };
  consider(4, 2, 3, {10.8f, 12.1f, 15.6f}, 21.5f, blocks<T, EPI, 4, 2, 4, 1, 4>);
  consider(4, 4, 3, {13.3f, 15.4f, 20.4f}, 37.f, blocks<T, EPI, 4, 4, 2, 2, 3>);
  consider(4, 8, 1, {12.1f}, 70.f, blocks<T, EPI, 4, 8, 2, 4, 4>);
  if constexpr (Kind<T>::BF16) consider(4, 8, 2, {12.6f, 20.1f}, 0.f, blocks<T, EPI, 4, 8, 2, 4, 3>);
  consider(4, 16, 1, {18.7f}, 160.f, blocks<T, EPI, 4, 16, 2, 4, 3>);
  consider(8, 8, 1, {17.6f}, 156.f, blocks<T, EPI, 8, 8, 4, 2, 3>);
  consider(8, 16, 1, {28.f}, 293.f, blocks<T, EPI, 8, 16, 2, 4, 3>);
  if constexpr (by_strips<T, EPI>()) {
    consider(8, 8, 2, {17.f, 31.f}, 0.f, strips<T, EPI, 8, 2, 4, 4, 8>, true);
    consider(8, 16, 2, {27.f, 53.f}, 0.f, strips<T, EPI, 8, 4, 4, 4, 4>, true);
  }
  return best;
}

template <typename T, int EPI>
Form form_of(const KernelArgs& p) {
  const int M = p.a.M, N = p.a.N;
  const int ntiles = (N + 15) / 16;
  // A model's head: blocks of two tiles read A half as often, which counts once A's rows are
  // many beside a block's weights; four waves of two parts each stream more of K (us by one
  // tile and eight waves / two and four).  16 rows, K 1024: 1000 tiles 10.0 / 9.0, 2048 18.6 /
  // 15.0, 4000 33.9 / 26.4; K 2048: 16.9 / 14.7, 31.7 / 26.3, 59.2 / 49.0; K 4096: 31.2 / 30.7,
  // 60.1 / 58.0, 114 / 103.  8 rows: 2048 tiles 15.3 / 14.1, 26.1 / 25.5, 47.5 / 56.0; 12 rows
  // of K 4096 53.5 / 57.8.  One row: 13.4 / 13.8, 24.3 / 24.5, 44.5 / 53.7.  512 tiles of 16
  // rows: 6.0 / 6.2, 9.4 / 8.9, 16.7 / 17.0.
  if constexpr (EPI == kStore && Kind<T>::BF16)
    if (M <= 16 && M > (p.KS > 64 ? 14 : 8) && p.KS <= 128 && ntiles >= 1000)
      return Form{stream<T, EPI, 1, 2, 4, 8>, 1};
  if (M <= 16) return Form{stream<T, EPI, 1, 1>, 1, stream_us<T>(ntiles * heads_of<EPI>(p), 1.5f)};
  if constexpr (EPI == kSplit) {
    // Narrow products: the fewest column tiles a block that are one round, as a block takes the time of
    // its chain of K whatever its width allows (K 4096, 160 columns, us by 1 / 2 / 3 / 5 tiles and 16 rows, 5
    // and 32: 333 rows 7.8 / 8.7 / 9.4 / 11.4, 15.0; 700 12.5 / 9.8 / 9.8 / 11.6, 15.1; 2011 25.4 / 23.1 /
    // 18.3 / 12.5, 15.5; K 2048, 96 columns: 333 4.8, 8.7; 1400 9.6 / 9.1 / 6.1 / 7.6, 9.5); past that all
    // columns in two blocks of 32 rows, so a row is read twice.
    if (M > 64 && ntiles <= 10) {
      const int rb = (M + 15) / 16;
      const auto one_round = [&](int nt) { return (ntiles + nt - 1) / nt * rb <= 256; };
      if (one_round(1)) return Form{stream<T, EPI, 1, 1>, rb};
      if (one_round(2)) return Form{stream<T, EPI, 1, 2>, rb};
      if (one_round(3)) return Form{stream<T, EPI, 1, 3>, rb};
      if (one_round(5)) return Form{stream<T, EPI, 1, 5>, rb};
      if ((M + 31) / 32 * 2 < 1024) return Form{stream<T, EPI, 2, 5>, (M + 31) / 32};
    }
  }
  // Blocks once the smallest of them are more than half a round, else streams:
  // 64 x 6144 x 1024 5.1 us as blocks (streams 5.3), 64 x 2048 x 6144 10.7 as
  // streams (blocks 15.4), 128 x 2048 x 6144 16.3 as streams (blocks 17.5).
  if (M > 32 && (M + 63) / 64 * ((N + 31) / 32) * heads_of<EPI>(p) > 128)
    return block_form<T, EPI>(p, 4, 8, N);
  // The stream form with the fewest rounds of workgroups, a round priced by its
  // column tiles and the rows it reads.
  struct Tiles {
    int mt, nt;
    float rows;
    Form::Go go;
  };
  static constexpr Tiles forms[] = {{1, 1, 0.5f, stream<T, EPI, 1, 1>},
                                    {1, 2, 0.5f, stream<T, EPI, 1, 2>},
                                    {2, 2, 1.5f, stream<T, EPI, 2, 2>},
                                    {2, 3, 1.5f, stream<T, EPI, 2, 3>}};
  Form best;
  for (const Tiles& f : forms) {
    const int rb = (M + 16 * f.mt - 1) / (16 * f.mt);
    const float us = stream_us<T>((ntiles + f.nt - 1) / f.nt * rb * heads_of<EPI>(p), (float)f.nt + f.rows);
    if (!best.go || us < best.us) best = Form{f.go, rb, us};
  }
  return best;
}

template <typename T, int EPI>
hipError_t launch(const KernelArgs& p, hipStream_t st) {
  const Form f = form_of<T, EPI>(p);
  return f.go(p, f.row_blocks, p.a.N, st);
}

template <typename T, int EPI>
hipError_t launch_grouped(const MmGrouped& g, int w_nt, hipStream_t st) {
  KernelArgs p{};
  p.g = g;
  p.a.w_nt = w_nt;
  if (g.tile_rows > 16) {
    const Form f = block_form<T, EPI>(p, g.tile_rows / 16, g.tile_rows / 16, g.max_n);
    return f.go(p, f.row_blocks, g.max_n, st);
  }
  // bf16: at least eight k-steps a wave (an expert's output product of 32 k-steps over 37 tiles
  // 26 us by eight waves, 20.5 by four; of 16 over 52 15.2, 10.5 by two), the sums in as many
  // parts as by eight.  Two waves a workgroup are too few in flight while a CU has but two or
  // three workgroups: 16 k-steps 4.0 us by eight waves, 4.7 by two over 64 x 5 workgroups, 4.1
  // and 5.1 over 64 x 9, 6.0 and 5.3 over 64 x 13.
  if constexpr (Kind<T>::BF16) {
    const bool few = g.max_tiles * ((g.max_n + 15) / 16) <= 640;
    if (g.min_ks >= 32 && g.min_ks < 64) return stream<T, EPI, 1, 1, 4, 8>(p, g.max_tiles, g.max_n, st);
    if (g.min_ks < 32 && !few)
      return g.min_ks >= 16 ? stream<T, EPI, 1, 1, 2, 8>(p, g.max_tiles, g.max_n, st)
                            : stream<T, EPI, 1, 1, 2, 4>(p, g.max_tiles, g.max_n, st);
  }
  return g.min_ks >= 16 ? stream<T, EPI, 1, 1>(p, g.max_tiles, g.max_n, st)
                        : stream<T, EPI, 1, 1, 4>(p, g.max_tiles, g.max_n, st);
}

}  // namespace
}  // namespace llm
