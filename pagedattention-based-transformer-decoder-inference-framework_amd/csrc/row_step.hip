// All layers of a decode step of a small INT8 decoder in one launch: a workgroup is a row.
//
// At hidden 256 a layer's five launches (LayerNorm with q|k|v, attention, output product, LayerNorm
// with fc1, quantising with fc2) wait for one another and for the launch, 4.7 us each, while its weights are
// 786 KB, 6 us at the 64 bytes a clock that one CU reads from its L2.  So one workgroup of sixteen waves goes
// through the layers by itself: what passes from one step to the next lies in LDS, nine barriers a layer, and
// each step's weights are loaded into registers before the barrier in front of it, with no wait for them there.
// Rows share nothing but their XCD's copy of the weights.  A layer takes 11 to 12 us at 113 tokens (launches
// 23.5), 1.1 us of them the attention's, and 4 at 400: half the weights' way, half instructions, of which
// every one of four waves on a SIMD costs the others its turn.  So LayerNorms and the merge are one wave's
// (done again by all sixteen 16 us a layer); weights two steps ahead cost the step in between what they save
// (25 -> 27 us a step of two layers), other workgroups that pull them into L2 ahead nothing.
//
// Arithmetic is the launches': LayerNorm and quantising by ln_wave.hpp, products summed exactly in int32 and
// scaled by sa * sw, fp32 softmax with q pre-scaled to log2 units; only the attention's sums have another
// order.
#include "row_step.hpp"

#include "ln_wave.hpp"

namespace llm {
namespace {

constexpr int kWaves = 16, HID = kRowStepHidden, INTER = 4 * HID;
constexpr int kTable = 64 * kWaves;  // page ids held in LDS, one a thread; further ones are read where they are needed

// LDS is written, loads from memory stay in flight
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

__device__ __forceinline__ int rows_sum(int x) {  // of lanes l, l ^ 16, l ^ 32, l ^ 48
  auto r = __builtin_amdgcn_permlane16_swap((uint32_t)x, (uint32_t)x, false, false);
  x = (int)(r[0] + r[1]);
  r = __builtin_amdgcn_permlane32_swap((uint32_t)x, (uint32_t)x, false, false);
  return (int)(r[0] + r[1]);
}

// A wave's T column tiles of a product of KS k-steps: weights, column scales and biases.
template <int T, int KS, bool BIAS>
struct Weights {
  u32x4 w[T][KS];
  float scale[T], bias[T];

  // (not earlier than it stands: there are registers for one step's weights)
  __device__ __forceinline__ void load(const RowProduct& p, int layer, int wave, uint32_t lane) {
    __builtin_amdgcn_sched_barrier(0);
    constexpr int N = 16 * T * kWaves;
    const char* src = reinterpret_cast<const char*>(p.w + (size_t)layer * p.stride + (size_t)wave * T * KS * 1024);
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int k = 0; k < KS; ++k) w[t][k] = *reinterpret_cast<const u32x4*>(src + (t * KS + k) * 1024 + lane * 16);
    const size_t n = (size_t)layer * N + wave * T * 16;
    const char* sp = reinterpret_cast<const char*>(p.scale + n);
    const char* bp = reinterpret_cast<const char*>(p.bias + n);
#pragma unroll
    for (int t = 0; t < T; ++t) {
      scale[t] = *reinterpret_cast<const float*>(sp + t * 64 + (lane & 15) * 4);
      if constexpr (BIAS) bias[t] = *reinterpret_cast<const float*>(bp + t * 64 + (lane & 15) * 4);
    }
  }

  // column (wave T + t) 16 + (lane & 15) of a row of int8 in LDS with scale sa
  __device__ __forceinline__ void times(const uint8_t* a, float sa, float (&y)[T]) const {
#pragma clang fp contract(off)  // scaled, then the bias added: rounded twice, as the launches do
    int s[T] = {};
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const u32x4 x = *reinterpret_cast<const u32x4*>(a + 64 * k + 16 * (lane_id() >> 4));
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) s[t] = __builtin_amdgcn_sdot4((int)x[e], (int)w[t][k][e], s[t], false);
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
      y[t] = (float)rows_sum(s[t]) * (sa * scale[t]);
      if constexpr (BIAS) y[t] = y[t] + bias[t];
    }
  }
};

// A wave's row of 256 values at ln_wave.hpp's places -> int8 in LDS; its scale
__device__ __forceinline__ float quantise(const LnRow<1>& v, float largest, uint8_t* to) {
  const float scale = 127.f / (largest + 1e-6f);
  *reinterpret_cast<uint32_t*>(to + 4 * lane_id()) = ln_quant4(v.v[0], scale);
  return 1.0f / scale;
}

// TAP: the rows of int8 go to the taps too.  The same code; behind a branch it costs every step scalar registers
// (24.5 -> 25.7 us for 2 layers).
template <int D, bool TAP>
__global__ __launch_bounds__(64 * kWaves) void row_step_kernel(RowStep a) {
  constexpr int H = HID / D, PER = kWaves / H;      // waves of a head
  constexpr int ACROSS = D / 8, TOKENS = 64 / ACROSS;  // lanes of a token, tokens of a load
  __shared__ __align__(16) float x[HID], gains[2 * HID], q[HID], part_o[kWaves][D], part_ml[kWaves][2], largest[kWaves];
  __shared__ __align__(16) _Float16 kv[2 * HID];  // the new token's keys, values
  __shared__ __align__(16) uint8_t ints[INTER];
  __shared__ float ints_scale;
  __shared__ int32_t pages[kTable];
  const int w = wave_id_uniform(), m = blockIdx.x;
  int lane = lane_id();
  const int pos = a.pos[m], tile = pos >> a.page_shift, in_page = pos & ((1 << a.page_shift) - 1);
  const int held = min(kTable / H, min(tile + 1, a.max_tiles));  // tiles of a head whose pages LDS holds

  Weights<3 * HID / 16 / kWaves, HID / 64, false> wqkv;
  Weights<HID / 16 / kWaves, HID / 64, false> wo;
  Weights<INTER / 16 / kWaves, HID / 64, true> w1;
  Weights<HID / 16 / kWaves, INTER / 64, true> w2;
  // A LayerNorm's gains and biases: loaded by the first 512 threads a step ahead, then put into LDS.
  const auto gain_of = [&](const float* g, const float* b, int layer) {
    const char* p = reinterpret_cast<const char*>((w < HID / 64 ? g : b - HID) + (size_t)layer * HID);
    return w < 2 * HID / 64 ? *reinterpret_cast<const float*>(p + (uint32_t)(w * 256 + lane * 4)) : 0.f;
  };
  const auto put_gain = [&](float g) {
    if (w < 2 * HID / 64) gains[w * 64 + lane] = g;
  };
  // A row of int8 (of HID, by wave 0) and its scale to the taps.
  const auto tap = [&](int layer, int stage, float sa) {
    if constexpr (!TAP) return;
    const size_t slot = (size_t)layer * 4 + stage;
    *reinterpret_cast<uint32_t*>(a.tap_q + slot * a.tap_stride + a_frag_off_i8(m, 4 * lane_id(), HID / 64)) =
        *reinterpret_cast<const uint32_t*>(ints + 4 * lane_id());
    if (lane_id() == 0) a.tap_s[slot * a.tap_rows + m] = sa;
  };
  const auto normalise = [&](int layer, int stage) {  // x -> ints, by wave 0
    if (w != 0) return;
    LnRow<1> v, gain, shift;
    v.v[0] = *reinterpret_cast<const f32x4*>(&x[4 * lane_id()]);
    gain.v[0] = *reinterpret_cast<const f32x4*>(&gains[4 * lane_id()]);
    shift.v[0] = *reinterpret_cast<const f32x4*>(&gains[HID + 4 * lane_id()]);
    const float sa = quantise(v, ln_wave_compute(v, gain, shift, HID, a.eps), ints);
    if (lane_id() == 0) ints_scale = sa;
    tap(layer, stage, sa);
  };
  put_gain(gain_of(a.ln1_g, a.ln1_b, 0));
  if (w == kWaves - 1) {
    LnRow<1> v;
    ln_wave_load_f16(ln_embed_row(a.emb, a.tok, m, a.V, HID), HID / 4, true, v);
    *reinterpret_cast<f32x4*>(&x[4 * lane]) = v.v[0];
  }
  lds_barrier();

  for (int l = 0; l < a.L; ++l) {
    // Addresses are made where they are used (kept over the layers they take 50 registers).
    asm volatile("" : "+v"(lane));
    const int32_t* table = a.page_table + ((size_t)l * a.beams + m) * H * a.max_tiles;
    const int at = w % PER * 64 + lane;  // of the head's tiles (before the weights: what follows is waited for with them)
    const int page_id = at < held ? table[(size_t)(w / PER) * a.max_tiles + at] : -1;
    wqkv.load(a.qkv, l, w, lane);
    pages[w * 64 + lane] = page_id < a.num_pages ? page_id : -1;
    normalise(l, 0);
    lds_barrier();

    {  // q | k | v
      constexpr int T = 3 * HID / 16 / kWaves;
      static_assert(T <= 4, "a tile for a sixteen of lanes");
      float y[T];
      wqkv.times(ints, ints_scale, y);
      float mine = y[0];  // the lane's column of its sixteen's tile
#pragma unroll
      for (int t = 1; t < T; ++t) mine = (lane >> 4) == t ? y[t] : mine;
      const int n = w * T * 16 + lane;
      if (lane < 16 * T) {
        if (n < HID) q[n] = mine;
        else kv[n - HID] = (_Float16)mine;
      }
    }
    wo.load(a.o, l, w, lane);
    const float gain = gain_of(a.ln2_g, a.ln2_b, l);
    lds_barrier();

    // (a look-up past LDS would be waited for together with the weights on their way.  Rows that row_step_ok admits are
    // never so long, but the device's position can be past the host's count: replays of a captured step)
    const auto page_of = [&](int head, int t, bool in_lds) {
      const int i = t >> a.page_shift;
      if (in_lds) return pages[head * (64 * PER) + i];
      if (i >= a.max_tiles) return -1;
      const int page = table[(size_t)head * a.max_tiles + i];
      return page < a.num_pages ? page : -1;
    };
    // Attention: a head's waves take its tokens in turn, ACROSS lanes a token; lanes of different tokens
    // keep maxima and sums of their own until the end.  The new token comes out of LDS.
    {
      const int head = w / PER, part = w % PER, d = lane % ACROSS * 8;
      float qs[8], o[8] = {}, mx = kNegSentinel, sum = 0.f;
      const float qscale = a.attn_scale * kLog2e;
#pragma unroll
      for (int e = 0; e < 8; ++e) qs[e] = q[head * D + d + e] * qscale;
      const auto score = [&](const f16x8& k) {
        float s = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) s = fmaf(qs[e], (float)k[e], s);
        return group_sum<ACROSS>(s);
      };
      constexpr int U = 4;  // tokens of a lane in flight
      const auto attend = [&](int t0, bool in_lds) {
        f16x8 k[U], vv[U];
        bool ok[U];
        int page[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int t = t0 + u * PER * TOKENS + lane / ACROSS;
          page[u] = t < pos ? page_of(head, t, in_lds) : -1;
          ok[u] = page[u] >= 0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int t = t0 + u * PER * TOKENS + lane / ACROSS;
          const size_t at = (size_t)max(page[u], 0) * a.page_stride + (t & ((1 << a.page_shift) - 1)) * D + d;
          k[u] = *reinterpret_cast<const f16x8*>(a.k_pool + at);
          vv[u] = *reinterpret_cast<const f16x8*>(a.v_pool + at);
        }
        float s[U], top = mx;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          s[u] = score(k[u]);
          s[u] = ok[u] ? s[u] : kNegSentinel;
          top = fmaxf(top, s[u]);
        }
        const float f = __builtin_amdgcn_exp2f(mx - top);
        mx = top;
        sum *= f;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] *= f;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const float p = ok[u] ? __builtin_amdgcn_exp2f(s[u] - mx) : 0.f;
          sum += p;
          if (!ok[u]) vv[u] = f16x8{};  // (0 times what is no number)
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = fmaf(p, (float)vv[u][e], o[e]);
        }
      };
      int t0 = part * TOKENS;
      if (tile < held) {
        for (; t0 < pos; t0 += U * PER * TOKENS) attend(t0, true);
      } else {
        for (; t0 < pos; t0 += U * PER * TOKENS) attend(t0, false);
      }
      if (part == 0 && tile < a.max_tiles) {
        const float s = score(*reinterpret_cast<const f16x8*>(&kv[head * D + d]));
        const f16x8 vn = *reinterpret_cast<const f16x8*>(&kv[HID + head * D + d]);
        if (lane < ACROSS) {
          const float top = fmaxf(mx, s), f = __builtin_amdgcn_exp2f(mx - top), p = __builtin_amdgcn_exp2f(s - top);
          mx = top;
          sum = fmaf(sum, f, p);
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = fmaf(o[e], f, p * (float)vn[e]);
        }
      }
      float top = mx;
      if constexpr (ACROSS <= 4) top = fmaxf(top, lane_xor<4>(top));
      if constexpr (ACROSS <= 8) top = fmaxf(top, lane_xor<8>(top));
      top = rows_max(top);
      const float f = __builtin_amdgcn_exp2f(mx - top);
      const auto all = [&](float s) {  // over the lanes of other tokens
        s *= f;
        if constexpr (ACROSS <= 4) s += lane_xor<4>(s);
        if constexpr (ACROSS <= 8) s += lane_xor<8>(s);
        return add(with_lane32(add(with_lane16(s))));
      };
      sum = all(sum);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = all(o[e]);
      if (lane < ACROSS) {
#pragma unroll
        for (int e = 0; e < 8; ++e) part_o[w][d + e] = o[e];
        if (lane == 0) {
          part_ml[w][0] = top;
          part_ml[w][1] = sum;
        }
      }
    }
    put_gain(gain);
    w1.load(a.fc1, l, w, lane);
    if (w == kWaves - 1) {  // the new token into its page (a load behind a store waits for it too)
      const int which = lane / (HID / 8), n = lane % (HID / 8) * 8;
      static_assert(2 * HID / 8 == 64, "a wave's");
      const int page = tile < held ? page_of(n / D, pos, true) : page_of(n / D, pos, false);
      if (page >= 0)
        *reinterpret_cast<f16x8*>((which ? a.v_pool : a.k_pool) + (size_t)page * a.page_stride +
                                  (size_t)in_page * D + n % D) = *reinterpret_cast<const f16x8*>(&kv[which * HID + n]);
    }
    lds_barrier();

    if (w == 0) {  // merge
      const int head = 4 * lane / D, d = 4 * lane % D;
      float top = kNegSentinel, sum = 0.f;
#pragma unroll
      for (int p = 0; p < PER; ++p) top = fmaxf(top, part_ml[head * PER + p][0]);
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int p = 0; p < PER; ++p) {
        const float f = __builtin_amdgcn_exp2f(part_ml[head * PER + p][0] - top);
        sum += f * part_ml[head * PER + p][1];
        o += f * *reinterpret_cast<const f32x4*>(&part_o[head * PER + p][d]);
      }
      const float inv = 1.0f / (sum + 1e-6f);
      float most = 0.f;
      LnRow<1> v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v.v[0][e] = o[e] * inv;
        most = fmaxf(most, fabsf(v.v[0][e]));
      }
      const float sa = quantise(v, ln_wave_max(most), ints);
      if (lane == 0) ints_scale = sa;
      tap(l, 1, sa);
    }
    lds_barrier();

    {  // output product
      float y[1];
      wo.times(ints, ints_scale, y);
      if (lane < 16) x[w * 16 + lane] = y[0];
    }
    lds_barrier();

    normalise(l, 2);
    const float next_gain = gain_of(a.ln1_g, a.ln1_b, min(l + 1, a.L - 1));
    lds_barrier();

    // fc1: a column a lane
    constexpr int T1 = INTER / 16 / kWaves;
    static_assert(T1 == 4, "a tile for each sixteen of lanes");
    float h;
    {
      float y[T1];
      w1.times(ints, ints_scale, y);
      h = y[0];
#pragma unroll
      for (int t = 1; t < T1; ++t) h = (lane >> 4) == t ? y[t] : h;
      h = fmaxf(h, 0.f);
      const float most = ln_wave_max(h);
      if (lane == 0) largest[w] = most;
    }
    w2.load(a.fc2, l, w, lane);
    lds_barrier();
    put_gain(next_gain);
    const float scale = 127.f / (ln_wave_max(largest[lane & 15]) + 1e-6f);
    const uint8_t mine = (uint8_t)ln_quant4(f32x4{h, 0.f, 0.f, 0.f}, scale);
    ints[w * 64 + lane] = mine;
    if constexpr (TAP) {
      const size_t slot = (size_t)l * 4 + 3;
      a.tap_q[slot * a.tap_stride + a_frag_off_i8(m, w * 64 + lane, INTER / 64)] = (int8_t)mine;
      if (w == 0 && lane == 0) a.tap_s[slot * a.tap_rows + m] = 1.0f / scale;
    }
    lds_barrier();

    {  // fc2
      float y[1];
      w2.times(ints, 1.0f / scale, y);
      if (lane < 16) x[w * 16 + lane] = y[0];
    }
    lds_barrier();
  }
  if (w == 0) *reinterpret_cast<f32x4*>(a.x + (size_t)m * HID + 4 * lane) = *reinterpret_cast<const f32x4*>(&x[4 * lane]);
  if (w == 1) *reinterpret_cast<f32x4*>(a.q + (size_t)m * HID + 4 * lane) = *reinterpret_cast<const f32x4*>(&q[4 * lane]);
}

}  // namespace

// Up to 8 rows of up to 512 tokens: a row's attention on one CU takes 2.9 us a layer for 256 tokens, that of
// splits over the chip nearly the same time whatever they are, and of more rows the launches take longer only
// from 16 on.  One decoder with a logits' place, 16 steps and a prompt of 113 tokens before them, 2 layers: 1,065 -> 845 us;
// 8 rows of 400 tokens, 4 layers, 20 steps 4,020 -> 3,585; 2 heads of 128 1,084 -> 890, 8 of 32 1,038 -> 864.
// Three decoders in turns, 4 layers: 64 rows from 100 tokens on 159 -> 168, 16 from 600 83 -> 86 (not by this
// rule), one from 500 48.5 -> 108 with no bound on the tokens.
bool row_step_ok(int hidden, int inter, int D, int page_size, int rows, int longest) {
  return hidden == HID && inter == INTER && (D == 32 || D == 64 || D == 128) && (page_size == 16 || page_size == 32) &&
         rows >= 1 && rows <= 8 && longest <= 512;
}

hipError_t row_step(const RowStep& a, hipStream_t st) {
  if (a.rows < 1 || a.rows > a.beams || a.L < 1 || a.page_shift < 0) return hipErrorInvalidValue;
  const auto go = [&](void (*kernel)(RowStep)) {
    hipLaunchKernelGGL(kernel, dim3(a.rows), dim3(64 * kWaves), 0, st, a);
    return hipGetLastError();
  };
  switch (a.D) {
    case 32: return go(a.tap_q ? row_step_kernel<32, true> : row_step_kernel<32, false>);
    case 64: return go(a.tap_q ? row_step_kernel<64, true> : row_step_kernel<64, false>);
    case 128: return go(a.tap_q ? row_step_kernel<128, true> : row_step_kernel<128, false>);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace llm
