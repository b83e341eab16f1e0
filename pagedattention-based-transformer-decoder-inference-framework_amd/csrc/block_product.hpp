// The product of a block of 16 MB rows and 16 NB columns on MFMA, both operands
// through LDS: the prompt-sized products of the layer-stack models (mm_impl.hpp) and
// of the dense decoders (gemm_impl.hpp).
#pragma once

#include <type_traits>

#include "common.hpp"

namespace llm {

// Workgroups go round the XCDs in turn.  Block id -> tile of an nx wide grid, in a
// walk whose neighbours are the blocks of one XCD: they share rows of A and columns
// of W in its L2, eight row blocks at a time.
struct TileAt {
  int x = 0, y = 0;
};
__device__ __forceinline__ TileAt xcd_tile(int id, int nx, int ny) {
  const int total = nx * ny, xcd = id & 7, each = total >> 3, more = total & 7;
  const int t = xcd * each + min(xcd, more) + (id >> 3);
  const int group = t / (8 * nx), r = t - group * 8 * nx, rows = min(8, ny - 8 * group);
  return {r / rows, 8 * group + r % rows};
}

// WM x WN waves.  A k-step is 64 bytes of every row and column (32 bf16 / fp16, 64
// int8, 16 fp32), a fragment of 16 of them 1 KiB.  Both operands go from memory
// straight into LDS, ST stages of two k-steps in flight; while a wave multiplies one
// k-step it reads the fragments of the next.  It waits for its own loads of a stage
// alone; the barrier then makes them everyone's and frees the stage that was read
// before.  The loads are spread among the matrix instructions: issued together they
// hold up the wave while the matrix cores run dry.
// The matrix instruction takes W as its first operand: a lane's sums are four neighbouring
// columns, 4 (lane >> 4) on, of row 16 i + (lane & 15) of A.
// W is packed, fragment after fragment (w_tile(t): the first of column tile t).  A is
// packed alike (A_PACKED; a_at(t): the first fragment of row tile t) or row-major
// (a_at(r): row r).  Row-major, a load takes 8 rows x 128 bytes, whole cache lines (16
// rows x 64 bytes, the fragment itself, took 1.7 times as long per byte); the 16-byte
// chunks of a row are exchanged by (row / 2) so that a fragment's 16 rows lie in
// different banks.  Addresses past the operands' ends are the callers' to avoid.
// Bound by the matrix cores waiting at the barriers: 2048 x 2048 x 6144 48.6 us, 1060
// TFLOP/s (113 us with two k-steps loaded and waited for together in 128 x 128 blocks
// of four waves); 2048 x 12288 x 2048 101 us (143), 700 x 2048 x 2048 12.3 us (32).
//
// PARTS: K in eight parts, each summed from zero and then added to the parts before it.
// One fp32 sum over all of K is off by 2 to 3 times as much as the streams' eight waves'
// (fp16, K 8192: 5.7e-7 of the result, so 2.1e-7, streams 2.1e-7; an fp32 stack's prompt of
// 100 tokens 1.5e-6, so 8.3e-7): a wave's registers hold both, and it costs fp16 products
// 3 to 10 % (2048 x 6144 x 2048 74.0 -> 78.7 us, the 64-row streams 321), fp32 ones nothing.
// Not for bf16, whose operands' rounding hides it, nor for int8, whose sums are exact.
//
// here: whether any of the wave's rows exist (the others load and wait).  When it
// returns, nobody reads LDS any more.
template <bool A_PACKED, bool PARTS, int MB, int NB, int WM, int WN, int ST, typename Acc, typename A,
          typename W, typename Mma>
__device__ __forceinline__ void block_product(u32x4 (&lds)[ST][2 * (MB + NB)][64],
                                              Acc (&acc)[MB / WM][NB / WN], int KS, bool here,
                                              const A& a_at, const W& w_tile, const Mma& mma) {
  constexpr int WAVES = WM * WN, MT = MB / WM, NT = NB / WN;
  constexpr int LOADS = 2 * (MB + NB) / WAVES;  // of a wave and stage, 1 KiB each
  static_assert(2 * (MB + NB) % WAVES == 0);
  const int lane = lane_id(), w = wave_id_uniform();
  const int wm = w / WN, wn = w % WN, stages = KS >> 1;

  // load l of a stage: A (l < 2 MB), eight rows or a k-step of a tile, then the two
  // k-steps of each of W's column tiles
  const char* src[LOADS];
  const int l0 = w * LOADS;
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int l = l0 + i;
    if (l >= 2 * MB) {
      src[i] = w_tile((l >> 1) - MB) + (l & 1) * 1024 + lane * 16;
    } else if constexpr (A_PACKED) {
      src[i] = a_at(l >> 1) + (l & 1) * 1024 + lane * 16;
    } else {
      const int r = 8 * l + (lane >> 3);
      src[i] = a_at(r) + 16 * ((lane & 7) ^ ((r >> 1) & 7));
    }
  }
  auto issue = [&](int st, int i) {
    load_to_lds(src[i], lds[st][l0 + i]);
    src[i] += !A_PACKED && l0 + i < 2 * MB ? 128 : 2048;
  };
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = Acc{0, 0, 0, 0};
  struct Frags {
    u32x4 a[MT], c[NT];
  };
  const int ar = lane & 15;  // row-major: this lane's row of a fragment, its chunks of the two k-steps
  const int at0 = 8 * ar + ((lane >> 4) ^ (ar >> 1)), at1 = at0 ^ 4;
  auto read = [&](Frags& f, int st, int u) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const u32x4* tile = &lds[st][2 * (wm * MT + i)][0];
      f.a[i] = A_PACKED ? tile[u * 64 + lane] : tile[u ? at1 : at0];
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) f.c[j] = lds[st][2 * (MB + wn * NT + j) + u][lane];
  };
  // multiplies, with loads [FROM, TO) of stage st among the products
  auto mul = [&](const Frags& f, int st, auto from, auto to) {
    constexpr int FROM = decltype(from)::value, TO = decltype(to)::value, N = MT * NT;
#pragma unroll
    for (int t = 0; t < N; ++t) {
      if constexpr (TO > FROM) {
#pragma unroll
        for (int i = FROM; i < TO; ++i)
          if ((i - FROM) * N / (TO - FROM) == t) {
            issue(st, i);
            __builtin_amdgcn_sched_barrier(0);
          }
      }
      const int i = t / NT, j = t % NT;
      acc[i][j] = mma(f.c[j], f.a[i], acc[i][j]);
    }
  };
  Acc sum[PARTS ? MT : 1][PARTS ? NT : 1];
  if constexpr (PARTS) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) sum[i][j] = Acc{0, 0, 0, 0};
  }
  // (PARTS) the part so far to the sum of parts
  auto part = [&] {
    if constexpr (PARTS) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          sum[i][j] += acc[i][j];
          acc[i][j] = Acc{0, 0, 0, 0};
        }
    }
  };
  const int every = PARTS ? max((stages + 4) / 8, 1) : 1;  // stages of a part
  int left = every;
  const std::integral_constant<int, 0> zero;
  const std::integral_constant<int, LOADS / 2> half;
  const std::integral_constant<int, LOADS> all;
  if (stages > 0) {
#pragma unroll
    for (int s = 0; s < ST; ++s)
      if (s < stages) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) issue(s, i);
      }
    Frags x, y;
    if (stages >= ST) wait_lds_loads<(ST - 1) * LOADS>();
    else wait_lds_loads<0>();
    barrier_only();
    if (here) {
      read(x, 0, 0);
      read(y, 0, 1);
      mul(x, 0, zero, zero);
    }
    int st = 0;
    auto landed = [&](int s) {  // stage s + 1 is there for everyone, stage s read out
      if (s + ST <= stages) wait_lds_loads<(ST - 2) * LOADS>();
      else wait_lds_loads<0>();
      barrier_only();
    };
    landed(0);
    int s = 0;
    for (; s + ST < stages; ++s) {
      const int now = st;
      st = st + 1 == ST ? 0 : st + 1;
      if (here) {
        read(x, st, 0);
        mul(y, now, zero, half);
        read(y, st, 1);
        mul(x, now, half, all);
      } else {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) issue(now, i);
      }
      if (PARTS && --left == 0) {
        part();
        left = every;
      }
      landed(s + 1);
    }
    for (; s + 1 < stages; ++s) {
      st = st + 1 == ST ? 0 : st + 1;
      if (here) {
        read(x, st, 0);
        mul(y, 0, zero, zero);
        read(y, st, 1);
        mul(x, 0, zero, zero);
      }
      if (PARTS && --left == 0) {
        part();
        left = every;
      }
      landed(s + 1);
    }
    if (here) mul(y, 0, zero, zero);
  }
  if (KS & 1) {  // the last k-step of an odd number, from memory
    Frags f;
    const size_t at = (size_t)(KS - 1) * 1024 + lane * 16;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int t = wm * MT + i;
      const char* p = A_PACKED ? a_at(t) + at : a_at(16 * t + ar) + (size_t)(KS - 1) * 64 + 16 * (lane >> 4);
      f.a[i] = *reinterpret_cast<const u32x4*>(p);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) f.c[j] = *reinterpret_cast<const u32x4*>(w_tile(wn * NT + j) + at);
    mul(f, 0, zero, zero);
  }
  if constexpr (PARTS) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] += sum[i][j];
  }
}

// A strip's loads (strip_product) in the order of its code: those that a wave has issued behind A's of
// stage `at` + 1 when it waits for these in stage `at`.  Stages behind the last whole AHEAD / 2 load no W.
constexpr int strip_behind(int ST, int LOADS, int NT, int AHEAD, int stages, int at) {
  int n = 0, there = 0;
  const auto a = [&](int s, int loads) {
    n += loads;
    if (s == at + 1) there = n;
  };
  a(0, LOADS);
  n += NT;
  for (int s = 1; s < ST - 1; ++s) a(s, LOADS);
  a(ST - 1, LOADS / 2);
  n += (AHEAD - 1) * NT;
  for (int s = 0;; ++s) {
    const int w = s < stages / (AHEAD / 2) * (AHEAD / 2) ? NT : 0;
    a(s + ST - 1, LOADS / 2);
    n += w;
    if (s == at) return n - there;
    a(s + ST, LOADS / 2);
    n += w;
  }
}
// How many may still fly there, with W's loads in the stage and without.
constexpr int strip_left(int ST, int LOADS, int NT, int AHEAD, bool w) {
  return (ST - 2) * LOADS + (!w ? 0 : AHEAD < 2 * ST - 3 ? AHEAD : 2 * ST - 3) * NT;
}
constexpr bool strip_waits(int ST, int LOADS, int NT, int AHEAD) {
  for (int stages = 1; stages <= 4 * AHEAD; ++stages)
    for (int s = 0; s < stages; ++s)
      if (strip_left(ST, LOADS, NT, AHEAD, s < stages / (AHEAD / 2) * (AHEAD / 2)) >
          strip_behind(ST, LOADS, NT, AHEAD, stages, s))
        return false;
  return true;
}

// The same product by waves side by side, each of all 16 MB rows and 16 NT columns of its own:
// a wave alone reads its columns of W, so they come from memory straight into its registers,
// AHEAD k-steps ahead, and LDS holds A alone, ST stages of two k-steps.  Of a k-step a wave reads
// MB KiB from LDS for MB NT products (128 x 256: 32 KiB a block, the form above 64 KiB and W's
// 16 KiB written besides), and the block takes 64 KiB of LDS in place of 147: two a CU, whose
// first loads and last stores each other's products hide.  A fragment of A is read for the
// next k-step right behind its last product.  Sums are added in the order of the form above:
// the same bits.
// Amid a model, its code cold: 2011 x 12288 x 2048 bf16 with its activation 100 us, now
// 87; 2011 x 2048 x 2048 to 6144 40, 34; 32 experts' gate and up of 2048 tokens 146, 131.  The first
// uses the matrix cores for 62 % of the time that a CU is busy, at 1.85 GHz (kernels without products
// run at 2.3 to 2.4; products alone, out of registers, reach 2.0 PFLOP/s).
// AHEAD k-steps of W: the compiler waits for them as if A's loads between were none, so that 4 are
// 2 and 8 are 3.5; 128 x 128 alone on a CU needs the 8 (2011 x 2048 x 6144 58.7 us, 53.1), 128 x 256 has
// registers for 4.
// A is row-major, a_at as above; w_at(j): the wave's column tile j.  When it returns, nobody reads LDS any more.
template <int MB, int NT, int WAVES, int ST, int AHEAD, typename Acc, typename A, typename W, typename Mma>
__device__ __forceinline__ void strip_product(u32x4 (&lds)[ST][2 * MB][64], Acc (&acc)[MB][NT], int KS,
                                              const A& a_at, const W& w_at, const Mma& mma) {
  constexpr int LOADS = 2 * MB / WAVES;  // of A by a wave and stage
  static_assert(2 * MB % WAVES == 0 && LOADS % 2 == 0 && MB >= 2 + LOADS / 2 && ST >= 3 &&
                AHEAD >= 4 && AHEAD % 2 == 0 && (ST - 1) * LOADS + AHEAD * NT < 64 &&
                strip_waits(ST, LOADS, NT, AHEAD));
  const int lane = lane_id(), w = wave_id_uniform(), stages = KS >> 1, last = stages - 1;
  const int ar = lane & 15;  // as above
  const int at0 = 8 * ar + ((lane >> 4) ^ (ar >> 1)), at1 = at0 ^ 4;
  const char* src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int r = 8 * (w * LOADS + i) + (lane >> 3);
    src[i] = a_at(r) + 16 * ((lane & 7) ^ ((r >> 1) & 7));
  }
  const char* wp[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) wp[j] = w_at(j);
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = Acc{0, 0, 0, 0};
  if (stages > 0) {
    // loads [from, to) of stage s; behind the end the last one again, which nobody reads
    auto load_a = [&](int s, int slot, int from, int to) {
      const size_t at = (size_t)min(s, last) * 128;
#pragma unroll
      for (int i = 0; i < LOADS; ++i)
        if (i >= from && i < to) load_to_lds(src[i] + at, lds[slot][w * LOADS + i]);
    };
    u32x4 a[MB], b[AHEAD][NT];
    auto load_w = [&](int k, u32x4 (&f)[NT]) {
      const size_t at = (size_t)min(k, 2 * last + 1) * 1024;
#pragma unroll
      for (int j = 0; j < NT; ++j) f[j] = *reinterpret_cast<const u32x4*>(wp[j] + at + lane * 16);
    };
    auto read_a = [&](int i, int slot, int u) {
      const u32x4* tile = &lds[slot][2 * i][0];
      a[i] = tile[u ? at1 : at0];
    };
    load_a(0, 0, 0, LOADS);
    load_w(0, b[0]);
#pragma unroll
    for (int s = 1; s < ST - 1; ++s) load_a(s, s, 0, LOADS);
    load_a(ST - 1, ST - 1, 0, LOADS / 2);
#pragma unroll
    for (int k = 1; k < AHEAD; ++k) load_w(k, b[k]);
    __builtin_amdgcn_sched_barrier(0);
    wait_lds_loads<(ST - 1) * LOADS - LOADS / 2 + AHEAD * NT>();  // stage 0: what was issued behind it may fly
    barrier_only();
#pragma unroll
    for (int i = 0; i < MB; ++i) read_a(i, 0, 0);
    int slot = 0, before = ST - 1;  // of stage s, of stage s - 1
    // tail: W is there for all stages that are left; none of it is loaded
    auto stage = [&](auto tail, int s, u32x4 (&b0)[NT], u32x4 (&b1)[NT]) {
      constexpr bool TAIL = decltype(tail)::value;
#pragma unroll
      for (int i = 0; i < MB; ++i) {  // the other half of the loads into the slot that was freed last
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = mma(b0[j], a[i], acc[i][j]);
        read_a(i, slot, 1);
        if (i < LOADS / 2) load_a(s + ST - 1, before, LOADS / 2 + i, LOADS / 2 + i + 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (!TAIL) load_w(2 * s + AHEAD, b0);
      __builtin_amdgcn_sched_barrier(0);
      before = slot;
      slot = slot + 1 == ST ? 0 : slot + 1;
#pragma unroll
      for (int i = 0; i < MB; ++i) {
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = mma(b1[j], a[i], acc[i][j]);
        if (i == 1) {
          // The reads of stage s are done, the wave's loads of stage s + 1 there.  Behind them it has
          // issued stages s + 2 .. s + ST - 1 and 2 ST - 3 k-steps of W (s = 0: AHEAD, s = 1: more); in the
          // tail fewer of W, of which it counts none
          __builtin_amdgcn_sched_barrier(0);
          wait_lds_loads<strip_left(ST, LOADS, NT, AHEAD, !TAIL)>();
          barrier_only();
          read_a(0, slot, 0);
          read_a(1, slot, 0);
        } else if (i > 1) {
          read_a(i, slot, 0);
          if (i - 2 < LOADS / 2) load_a(s + ST, before, i - 2, i - 1);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (!TAIL) load_w(2 * s + AHEAD + 1, b1);
      __builtin_amdgcn_sched_barrier(0);
    };
    int s = 0;
    for (; s + AHEAD / 2 <= stages; s += AHEAD / 2) {
#pragma unroll
      for (int i = 0; i < AHEAD / 2; ++i) stage(std::false_type(), s + i, b[2 * i], b[2 * i + 1]);
    }
#pragma unroll
    for (int i = 0; i < AHEAD / 2 - 1; ++i)
      if (s + i < stages) stage(std::true_type(), s + i, b[2 * i], b[2 * i + 1]);
    wait_lds_loads<0>();
    barrier_only();
  }
  if (KS & 1) {  // the last k-step of an odd number, from memory
    const size_t at = (size_t)(KS - 1) * 1024 + lane * 16;
    u32x4 b[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) b[j] = *reinterpret_cast<const u32x4*>(wp[j] + at);
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const char* p = a_at(16 * i + ar) + (size_t)(KS - 1) * 64 + 16 * (lane >> 4);
      const u32x4 a = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] = mma(b[j], a, acc[i][j]);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
}

// The sums of strips, SR row tiles at a time from tile i0 on, to `emit(i0, part)`, of which there is
// one copy: they move down to the first registers.  It says whether to go on.
template <int SR, int MB, int NT, typename Acc, typename Emit>
__device__ __forceinline__ void strip_rows(const Acc (&acc)[MB][NT], const Emit& emit) {
  static_assert(MB % SR == 0);
  Acc part[MB / SR][SR][NT];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) part[i / SR][i % SR][j] = acc[i][j];
#pragma unroll 1
  for (int i0 = 0; i0 < MB; i0 += SR) {
    if (!emit(i0, part[0])) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // read before the next ones come
#pragma unroll
    for (int s = 0; s + 1 < MB / SR; ++s)
#pragma unroll
      for (int i = 0; i < SR; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) part[s][i][j] = part[s + 1][i][j];
  }
}

// us of `groups` blocks of which a CU holds `per` at once: at[n - 1] with n on every CU,
// launch included.  A round of workgroups follows the one before, the last one with as many
// a CU as are left.
inline float rounds_us(long long groups, int per, const float (&at)[3]) {
  const long long all = 256LL * per, full = groups / all, left = groups % all;
  return (float)full * at[per - 1] + (left ? at[(left + 255) / 256 - 1] : 0.f);
}

// A wave's sums into the block's LDS, row by row: row m0 + 16 i + .., column n0 + 16 j + .. of
// rows of STRIDE (a multiple of 4, not of 64: 16 lanes' 16 bytes lie in different banks).  What
// the wave then reads of its own rows and columns it need not wait for others for.
template <int STRIDE, int MT, int NT, typename Acc, typename E>
__device__ __forceinline__ void spread_sums(const Acc (&acc)[MT][NT], E* sums, int m0, int n0) {
  E* to = sums + (m0 + (lane_id() & 15)) * STRIDE + n0 + 4 * (lane_id() >> 4);
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) *reinterpret_cast<Acc*>(to + 16 * i * STRIDE + 16 * j) = acc[i][j];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

}  // namespace llm
