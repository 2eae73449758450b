// A block of a matrix product of many rows: bfloat16 in and out, float32 accumulate on MFMA (gemm_dense.hip: one matrix;
// gemm_stream.hip: groups' matrices).
//
// A block of four wavefronts, one a SIMD, takes FM * 32 rows of X by FN * 32 of W, a wavefront a quarter of it: FM x FN fragments of
// 16 x 16.  Both operands come through shared memory, brought by the load unit itself (a kilobyte an instruction: eight rows of
// 64 k, their 16-byte pieces swizzled by which piece a lane fetches, so that reading fragments meets no bank twice).  X's and
// W's halves of a stage of 64 k lie in a ring each, of RX and RW halves: as many as shared memory holds, so that a stage's
// loads have one to two stages' time.
//
// With one wavefront a SIMD nothing hides what it does between two products, and a product of fragments takes sixteen cycles:
// so whatever else there is (reading the next step's fragments, asking for a later stage's rows, places and addresses) is
// dealt out to single products, a few instructions to each at most.  One barrier a stage, in the middle of its first step: by then the
// stage's fragments are all in registers and the next stage's rows have come.  The loop has no tail of its own: loads behind the
// last stage are asked for with a buffer of no bytes, which the load unit answers by itself.
//
// 16 x 16 x 32 products and not 32 x 32 x 16: the chip slows down under load, and with random operands the wide ones
// stop at 1.85 PFLOP/s where these reach 2.10 (registers only, no memory).
#pragma once
#include <type_traits>
#include "common.h"
#include "gate_act.h"

namespace jle {
namespace dense {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;

constexpr int BK = 64;             // k of a stage (two MFMA steps)
constexpr uint32_t kUnit = 4096;   // bytes of 32 rows of a stage: a load instruction of every wavefront

template <int N, int I = 0, typename F>
__device__ __forceinline__ void each(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    each<N, I + 1>(f);
  }
}

// Where the halves of a stage lie.
struct Place {
  uint32_t x0, x1, w0, w1;
};

// 32 rows of X or W that a stage's places take: the half whose place it is and which rows in it, for the stage `ahead` of this one
struct Unit {
  bool w;
  int half, u, ahead;
};

template <int FM, int FN, int RX, int RW>
struct Ring {
  static constexpr uint32_t XB = FM * 2048, WB = FN * 2048;  // bytes of half a stage
  static constexpr uint32_t W0 = RX * XB;                    // W's ring lies behind X's
  static constexpr uint32_t bytes = W0 + RW * WB;
  static_assert((RX % 2 == 0 || FM % 2 == 0) && (RW % 2 == 0 || FN % 2 == 0), "rings of whole stages, or halves of whole units");
  static_assert(RX >= 4 && RX <= 6 && RW >= 4 && RW <= 6, "");

  static __device__ __forceinline__ uint32_t step(uint32_t at, uint32_t by, uint32_t begin, uint32_t end) {
    return at + by == end ? begin : at + by;
  }
  static __device__ __forceinline__ Place after(const Place& a) {
    Place b;
    b.x0 = RX % 2 == 0 ? step(a.x0, 2 * XB, 0, W0) : step(a.x1, XB, 0, W0);
    b.x1 = RX % 2 == 0 ? b.x0 + XB : step(b.x0, XB, 0, W0);
    b.w0 = RW % 2 == 0 ? step(a.w0, 2 * WB, W0, bytes) : step(a.w1, WB, W0, bytes);
    b.w1 = RW % 2 == 0 ? b.w0 + WB : step(b.w0, WB, W0, bytes);
    return b;
  }
  // Unit j of the ones that a stage's places take, the earlier stage's first.  With an odd ring a place takes the other
  // half of a later stage; with an even one the same, and the units of both halves follow each other.
  static constexpr Unit unit(int j) {
    int n = 0;
    for (int ahead = 2; ahead <= 3; ++ahead) {
      for (int i = 0; i < FM; ++i) {
        const int half = RX % 2 == 0 ? 0 : i / (FM / 2);
        if ((RX + half) / 2 == ahead && n++ == j) return Unit{false, half, RX % 2 == 0 ? i : i % (FM / 2), ahead};
      }
      for (int i = 0; i < FN; ++i) {
        const int half = RW % 2 == 0 ? 0 : i / (FN / 2);
        if ((RW + half) / 2 == ahead && n++ == j) return Unit{true, half, RW % 2 == 0 ? i : i % (FN / 2), ahead};
      }
    }
    return Unit{false, 0, 0, 0};
  }
  // Which of the later stage's units it is.
  static constexpr int of_stage(Unit v) {
    if (v.w) return RW % 2 == 0 ? v.u : (v.half ^ 1) * (FN / 2) + v.u;
    return RX % 2 == 0 ? v.u : (v.half ^ 1) * (FM / 2) + v.u;
  }
};

// What a block works on: `rows` rows of the result from m0 on, its columns from n0 on.
struct DenseBlock {
  const bf16_t* X;
  const bf16_t* W;
  bf16_t* Y;
  const bf16_t* bias;  // [N], or null
  const int* a_rows;   // TILED: the row of X of every row of the result, or null: its own
  const float* scale;  // TILED: a factor for every row of the result, or null
  int act;             // TILED and not GATED: max(., 0)^2 of the rounded sums
  int m0, rows, n0;
  int N, K;            // columns of Y
};

// TILED: W in the streaming layout, whose kilobytes (16 rows of 32 k) are fragments as a wavefront reads them.  GATED: gate rows
// first, silu(gate) * up of the sums.
template <int FM, int FN, int RX, int RW, bool GATED, bool TILED>
__device__ __forceinline__ void dense_block(const DenseBlock& p, unsigned char* smem) {
  using R = Ring<FM, FN, RX, RW>;
  static_assert(!GATED || (TILED && FN % 2 == 0), "a wavefront has a gate's fragments and their up's");
  constexpr int U = FM + FN, MF = FM * FN;
  constexpr uint32_t KX = BK * 2, KW = TILED ? BK * 32 : BK * 2;  // bytes from one stage to the next
  // Of a step's MF products: the reads of fragments are dealt out to the first SPAN; the barrier is behind product BP of a
  // stage's first step, eight behind the last read; from there on a load every STEP products.
  constexpr int SPAN = U > MF * 3 / 8 ? U : MF * 3 / 8, BP = SPAN + 8 < MF ? SPAN + 8 : MF - 2;
  constexpr int STEP = (2 * MF - BP - 2) / (U - 1);
  static_assert((U - 1) * SPAN / U < BP && STEP >= 1, "");
  constexpr int YOUNGER = (RX - 4) * FM / 2 + (RW - 4) * FN / 2;  // loads on their way behind those for the next stage
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int r = lane & 15, g = lane >> 4;
  const int wm = wave & 1, wn = wave >> 1;
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem + (uint32_t)(wave * 1024);
  const int m0 = p.m0, n0 = p.n0;
  const int nstage = p.K / BK;
  const int* const a_rows = TILED ? p.a_rows : nullptr;
  const uint64_t xa = (uint64_t)(uintptr_t)(a_rows != nullptr ? p.X : p.X + (size_t)m0 * p.K);
  const uint64_t wa = (uint64_t)(uintptr_t)(p.W + (size_t)n0 * p.K);
  auto same = [](uint32_t v) __attribute__((always_inline)) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
  uint32_t x_lo = same((uint32_t)xa), x_hi = same((uint32_t)(xa >> 32)), w_lo = same((uint32_t)wa), w_hi = same((uint32_t)(wa >> 32));
  asm volatile("s_nop 4" : "+s"(x_lo), "+s"(x_hi), "+s"(w_lo), "+s"(w_hi));  // (before a load reads what vector instructions wrote)
  // what this lane fetches: a piece of a row; rows behind the last one: the last one, not stored
  const uint32_t piece = (uint32_t)(((lane & 7) ^ (lane >> 3)) * 16);
  uint32_t xsrc[FM], wsrc[FN];
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int row = min(32 * i + 8 * wave + (lane >> 3), p.rows - 1);
    xsrc[i] = (uint32_t)(a_rows != nullptr ? a_rows[m0 + row] : row) * (uint32_t)(p.K * 2) + piece;
  }
#pragma unroll
  for (int i = 0; i < FN; ++i) {
    if constexpr (TILED) {  // a wavefront brings a fragment: 16 rows of one of the stage's two steps
      int row = 32 * i + 16 * (wave >> 1);
      if constexpr (GATED) {  // every half: FN * 8 rows of the gate and their rows of up
        const int in = row % (FN * 16), at = in % (FN * 8);
        row = min(row / (FN * 16) * (FN * 8) + at, p.N - 16 - n0) + (in >= FN * 8 ? p.N : 0);
      } else {
        row = min(row, p.N - 16 - n0);
      }
      wsrc[i] = (uint32_t)row * (uint32_t)(p.K * 2) + (uint32_t)((wave & 1) * 1024 + lane * 16);
      continue;
    }
    wsrc[i] = (uint32_t)min(32 * i + 8 * wave + (lane >> 3), p.N - 1 - n0) * (uint32_t)(p.K * 2) + piece;
  }
  auto load = [&](bool w, uint32_t live, uint32_t src, uint32_t k) __attribute__((always_inline)) {
    const u32x4 rsrc = {w ? w_lo : x_lo, w ? w_hi : x_hi, live, 0x00020000u};
    asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(src), "s"(rsrc), "s"(k) : "memory");
  };
  // all bytes, or none: of a stage behind the last one
  auto live = [&](int s) __attribute__((always_inline)) { return (uint32_t)__builtin_amdgcn_readfirstlane((s - nstage) >> 31); };

  f32x4 acc[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 fx[2][FM], fw[2][FN];
  const uint32_t off = (uint32_t)(r * 128 + ((g ^ (r & 7)) * 16));  // (second step: bit 6 the other way)
  const uint32_t offw = TILED ? (uint32_t)(lane * 16) : off;
  constexpr uint32_t W2 = TILED ? 1024 : 64;  // (W's second step: this bit the other way)
  // fragment I in the order in which the products need them: W's first one, X's, the rest of W's
  auto read = [&](auto SET, auto I, uint32_t x, uint32_t w) __attribute__((always_inline)) {
    constexpr int set = decltype(SET)::value, i = decltype(I)::value;
    if constexpr (i == 0 || i > FM) {
      constexpr int n = i == 0 ? 0 : i - FM;
      fw[set][n] = *reinterpret_cast<const bf16x8*>(smem + w + n * 2048);
    } else {
      fx[set][i - 1] = *reinterpret_cast<const bf16x8*>(smem + x + (i - 1) * 2048);
    }
  };

  // the first stages, as far as the rings hold them
  each<3>([&](auto S) __attribute__((always_inline)) {
    constexpr int s = decltype(S)::value;
    const uint32_t bytes = live(s);
    each<FM>([&](auto V) __attribute__((always_inline)) {
      constexpr int u = decltype(V)::value;
      if constexpr (2 * s + (u * 2 < FM ? 0 : 1) < RX) {
        asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0" ::"s"(lds0), "n"(2 * s * R::XB + u * kUnit) : "memory", "scc");
        load(false, bytes, xsrc[u], s * KX);
      }
    });
    each<FN>([&](auto V) __attribute__((always_inline)) {
      constexpr int u = decltype(V)::value;
      if constexpr (2 * s + (u * 2 < FN ? 0 : 1) < RW) {
        asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0" ::"s"(lds0), "n"(R::W0 + 2 * s * R::WB + u * kUnit) : "memory", "scc");
        load(true, bytes, wsrc[u], s * KW);
      }
    });
  });
  // (with odd halves of an even ring the units of a stage are together: FM * RX / 2 in all)
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(RX * FM / 2 + RW * FN / 2 - U) : "memory");
  Place here = {0, R::XB, R::W0, R::W0 + R::WB}, next = here;
  // where this wavefront's fragments lie: this stage's second step's, the next one's first
  uint32_t x1 = (wm ? R::XB : 0) + (off ^ 64), w1 = (wn ? R::W0 + R::WB : R::W0) + (offw ^ W2), x0 = x1 ^ 64, w0 = w1 ^ W2;
  each<U>([&](auto I) __attribute__((always_inline)) { read(std::integral_constant<int, 0>{}, I, x0, w0); });
  uint32_t to_x0 = 0, to_x1 = 0, to_w0 = 0, to_w1 = 0, live2 = 0, live3 = 0, k2 = KX, k3 = 2 * KX, kw2 = KW, kw3 = 2 * KW;
  for (int s = 0; s < nstage; ++s) {
    each<2 * MF>([&](auto I) __attribute__((always_inline)) {
      constexpr int at = decltype(I)::value, q = at / MF, i = at % MF;
      constexpr int a = i / FM, b = (a & 1) ? FM - 1 - i % FM : i % FM;  // (one operand stays from product to product)
      constexpr int late = at - BP - 1;
      constexpr bool loads = late >= 0 && late % STEP == 0 && late / STEP < U;
      constexpr Unit v = R::unit(loads ? late / STEP : 0);
      if constexpr (at == 0) to_x0 = lds0 + here.x0, to_w0 = lds0 + here.w0;
      if constexpr (at == 1) to_x1 = lds0 + here.x1, to_w1 = lds0 + here.w1;
      if constexpr (at == 2) k2 += KX, k3 += KX;
      if constexpr (at == 5 && TILED) kw2 += KW, kw3 += KW;
      if constexpr (at == 3) live2 = live(s + 2);
      if constexpr (at == 4) live3 = live(s + 3);
      if constexpr (at == BP - 3) next = R::after(here);
      if constexpr (at == BP - 2) x0 = (wm ? next.x1 : next.x0) + off, w0 = (wn ? next.w1 : next.w0) + offw;
      if constexpr (at == 2 * MF - 2) x1 = x0 ^ 64, w1 = w0 ^ W2;
      if constexpr (loads)
        asm volatile("s_add_u32 m0, %0, %1" ::"s"(v.w ? (v.half ? to_w1 : to_w0) : (v.half ? to_x1 : to_x0)), "n"(v.u * kUnit)
                     : "memory", "scc");
      // (as assembly: the compiler gives the builtin's result other registers than its addend's, and copies)
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[a][b]) : "v"(fw[q][a]), "v"(fx[q][b]));
      if constexpr (loads)
        load(v.w, v.ahead == 2 ? live2 : live3, v.w ? wsrc[R::of_stage(v) % FN] : xsrc[R::of_stage(v) % FM], TILED && v.w ? (v.ahead == 2 ? kw2 : kw3) : (v.ahead == 2 ? k2 : k3));
      constexpr int ri = (i * U + SPAN - 1) / SPAN;  // the fragment that is read here, if one is
      if constexpr (ri < U && ri * SPAN / U == i)
        read(std::integral_constant<int, q ^ 1>{}, std::integral_constant<int, ri>{}, q == 0 ? x1 : x0, q == 0 ? w1 : w0);
      if constexpr (at == BP) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(YOUNGER) : "memory");
      __builtin_amdgcn_sched_barrier(0);
    });
    here = next;
  }
  // (the last products' results are there after the wait for the barrier and sixteen cycles more)
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier\n\ts_nop 15" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);

  // accumulators: element e of [i][j] in lane (g, r) = row 4 g + e of W's fragment i, row r of X's fragment j.  Through shared memory, so
  // that rows of Y are written by whole lines, and past the caches (256 blocks' results at once are as large as they: 4,096 rows
  // of 4,096 with a k of 64 14.5 -> 9.6 us)
  constexpr int OUT = GATED ? FN * 8 : FN * 16;  // columns of Y of a wavefront
  constexpr int PITCH = OUT * 2 + 16;            // (rows begin in other banks)
  unsigned char* mine = smem + wave * FM * 16 * PITCH;
#pragma unroll
  for (int j = 0; j < FM; ++j) {
    const float sc = TILED && p.scale != nullptr ? p.scale[m0 + min(wm * FM * 16 + j * 16 + r, p.rows - 1)] : 1.f;
#pragma unroll
    for (int i = 0; i < OUT / 16; ++i) {
      float y[4];
      if constexpr (GATED) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float gate = acc[i][j][e] * sc, up = acc[i + FN / 2][j][e] * sc;
          y[e] = gate_act<0>(gate) * up;
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          y[e] = TILED ? acc[i][j][e] * sc : acc[i][j][e];
          if (TILED && p.act) y[e] = relu2(Num<bf16_t>::round(y[e]));
        }
        if (!TILED && p.bias != nullptr) {
          const int n = min(n0 + wn * OUT + i * 16 + 4 * g, p.N - 4);
          const uint2 c = *reinterpret_cast<const uint2*>(p.bias + n);
          y[0] += __uint_as_float(c.x << 16);
          y[1] += __uint_as_float(c.x & 0xffff0000u);
          y[2] += __uint_as_float(c.y << 16);
          y[3] += __uint_as_float(c.y & 0xffff0000u);
        }
      }
      *reinterpret_cast<uint2*>(mine + (j * 16 + r) * PITCH + i * 32 + g * 8) = uint2{pack_bf16(y[0], y[1]), pack_bf16(y[2], y[3])};
    }
  }
  constexpr int LANES = OUT / 8;  // a row, 16 bytes each
#pragma unroll 4
  for (int i = lane; i < FM * 16 * LANES; i += 64) {
    const int row = i / LANES, c = i % LANES;
    const u32x4 v = *reinterpret_cast<const u32x4*>(mine + row * PITCH + c * 16);
    const int t = wm * FM * 16 + row, n = n0 + wn * OUT + c * 8;
    if (t < p.rows && n < p.N) __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(p.Y + (size_t)(m0 + t) * p.N + n));
  }
}

// Bytes of shared memory of a block: its rings, or its part of the result.
template <int FM, int FN, int RX, int RW, bool GATED>
constexpr uint32_t dense_bytes() {
  constexpr uint32_t out = 4 * FM * 16 * ((GATED ? FN * 16 : FN * 32) + 16), ring = Ring<FM, FN, RX, RW>::bytes;
  return ring > out ? ring : out;
}

}  // namespace dense
}  // namespace jle
