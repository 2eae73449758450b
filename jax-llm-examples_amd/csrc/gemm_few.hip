// Matrix product of up to a few tens of rows (a decode step of up to 64 requests, the experts of such a step): bfloat16 in, float32
// accumulate on MFMA.
//
//   Y[t, n] = scale[t] * sum_k X[arow(t), k] * W[g(t)][n, k]     (plain; optionally max(., 0)^2 of the rounded sum)
//   Y[t, f] = act(s * gate) * (s * up),  gate/up = rows f and F + f of W[g(t)]   (SWIGLU, s = scale[t])
//
// The cost is reading W once, and with more than a few rows reading X again for every block: as B operands straight from
// memory, 16 rows at a time a long way apart, that took longer than the weights (gemm_skinny.hip: 2,048 x 2,048 with 8 rows
// 6.5 us, with 64 13.1).  Here both come through shared memory, brought by the load unit itself in whole lines of 128 bytes
// (a kilobyte an instruction, no register waits for it): a wavefront has a ring of its own, of stages of 64 k of its block's
// rows of W and X, and takes every fourth stage of k.  No wavefront waits for another until the four add up their sums, so
// the only thing that bounds it is how much is on its way: 48 to 128 KiB of rings a block.  Weights are asked for with loads
// that the caches need not keep.  Either layout of W (row-major, or tiles of 16 rows x 32 k of a kilobyte) is read by whole
// lines; sums and their order are the same.
// In microseconds, weights not in the caches (gigabytes of other reads between two of the same W), this and what it is taken
// instead of: gemm_skinny up to 8 rows, the library from 9 on:
//   2,048 x 2,048    1 row 4.8 | 6.6     8 rows 4.9 | 6.8     16 rows 5.2 | 11.9    32 rows 5.2 | 12.0    64 rows 6.2 | 12.4
//   2,048 x 4,096    1 row 7.0 | 7.8     8 rows 7.2 | 8.1     16 rows 7.7 | 15.5    32 rows 7.6 | 13.1    64 rows 9.5 | 15.0
//   4,096 x 4,096    1 row 7.9 | 10.0    8 rows 8.0 | 10.6    16 rows 8.5 | 16.9    32 rows 10.5 | 14.9   64 rows 12.5 | 16.8
//   4,096 x 14,336   1 row 22.8 | 31.3   8 rows 22.3 | 31.1   16 rows 24.7 | 38.1   32 rows 31.6 | 41.3   64 rows 38.9 | 51.5
//   5,120 x 5,120    1 row 12.3 | 13.0   8 rows 13.3 | 13.5   16 rows 14.6 | 19.6   32 rows 17.8 | 21.7   64 rows 23.8 | 24.7
//   7,168 x 5,120    1 row 14.3 | 15.3   8 rows 14.9 | 17.7   16 rows 16.0 | 23.6   32 rows 19.3 | 24.8   64 rows 25.1 | 27.2
//   10,304 x 2,048   1 row 10.0 | 10.3   8 rows 10.2 | 11.7   16 rows 10.8 | 18.0   32 rows 12.3 | 18.0   64 rows 15.0 | 18.9
//   14,336 x 4,096   1 row 21.9 | 22.7   8 rows 21.9 | 24.3   16 rows 22.1 | 38.9   32 rows 23.4 | 37.6   64 rows 27.7 | 37.1
// 8 groups of 4,096 x 2,048 with 128 rows 29.0 -> 24.6, of 2,048 x 4,096 37.7 -> 26.1, of 4,096 x 7,168 89.7 -> 79.7; gate
// and up of 4,096 x 2,048, 9 groups with 42 rows 47.5 -> 44.8, 8 with 128 51.4 -> 43.4 (gemm_skinny -> this).
#include "common.h"
#include "rows.h"

using namespace jle;

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

namespace {

constexpr int kLine = 64;           // k of a stage
constexpr int kPiece = 16 * 128;    // bytes of 16 rows of a stage
constexpr int kWaves = 4;           // wavefronts of a block

struct FewArgs {
  const bf16_t* X;
  const bf16_t* W;
  void* Y;
  const int* offsets;  // null: one group
  const int* a_rows;
  const float* scale;
  const bf16_t* W_last;
  int M, Nout, K, groups, tiled, tiled_last, slots, act;
};

// load_to_lds16 for bytes that nobody reads again: the caches need not keep them
__device__ __forceinline__ void load_to_lds16_once(const void* base, uint32_t byte_off, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt\n" ::"v"(byte_off), "s"(base), "s"(lds_addr) : "memory");
}

// waits until at most N of this wavefront's loads are on their way
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <typename OutT>
__device__ __forceinline__ float rounded(float v);
template <>
__device__ __forceinline__ float rounded<float>(float v) { return v; }
template <>
__device__ __forceinline__ float rounded<bf16_t>(float v) { return Num<bf16_t>::round(v); }

// MT: tiles of 16 rows of X a block; RT: tiles of 16 rows of W (SWIGLU: half of them gate rows, half their up rows); DEPTH:
// stages of a wavefront's ring.
template <int MT, int RT, int DEPTH, bool SWIGLU, typename OutT>
__global__ __launch_bounds__(kWaves * 64) void gemm_few_kernel(FewArgs p) {
  constexpr int PER = 2 * (MT + RT);               // loads of a stage, a kilobyte each
  constexpr int STAGE = (MT + RT) * kPiece;        // bytes of a wavefront's stage
  constexpr int CT = SWIGLU ? RT / 2 : RT;         // tiles of 16 columns of Y
  static_assert(kWaves * DEPTH * STAGE <= 160 * 1024 && MT * RT * 1024 <= DEPTH * STAGE, "shared memory");
  static_assert((DEPTH - 1) * PER < 64, "the counter of loads on their way has six bits");
  static_assert(!SWIGLU || RT % 2 == 0, "a gate tile for each tile of up");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int K = p.K, Nout = p.Nout;
  int e = blockIdx.z;
  if (p.slots) {
    // the blockIdx.z-th group that has rows: 64 groups a look, counted with a ballot
    int found = -1, seen = 0;
    for (int g0 = 0; g0 < p.groups && found < 0; g0 += 64) {
      const int gi = g0 + lane;
      const bool has = gi < p.groups && p.offsets[gi + 1] > p.offsets[gi];
      unsigned long long mask = __ballot(has);
      const int c = __popcll(mask);
      if ((int)blockIdx.z < seen + c) {
        for (int j = (int)blockIdx.z - seen; j > 0; --j) mask &= mask - 1;  // drop the lower set bits
        found = g0 + __ffsll((long long)mask) - 1;
      }
      seen += c;
    }
    if (found < 0) return;  // fewer groups have rows than there are slots
    e = __builtin_amdgcn_readfirstlane(found);
  }
  int row_lo = 0, row_hi = p.M;
  if (p.offsets != nullptr) {
    row_lo = p.offsets[e];
    row_hi = p.offsets[e + 1];
  }
  const int tok0 = row_lo + (int)blockIdx.y * (16 * MT);
  if (tok0 >= row_hi) return;  // the whole block
  const int live = min(16 * MT, row_hi - tok0);
  const bf16_t* We = p.W + (size_t)e * Nout * K;
  int tiled = p.tiled;
  if (p.W_last != nullptr && e == p.groups - 1) {  // the last group's matrix lies elsewhere (a shared expert)
    We = p.W_last;
    tiled = p.tiled_last;
  }
  const int half = Nout >> 1;
  const int n0 = (int)blockIdx.x * (16 * CT);  // first column of Y
  const uint32_t mine = (uint32_t)(uintptr_t)smem + (uint32_t)(wave * DEPTH * STAGE);
  const unsigned char* ring = smem + wave * DEPTH * STAGE;

  // where this lane's 16 bytes of each load come from: 8 rows' 128 bytes a load, a row's pieces in the order (piece ^ row),
  // so that reading 16 rows' pieces as an operand does not collide; a tiled matrix as it lies
  const uint32_t of_row = (uint32_t)(((lane & 7) ^ (lane >> 3)) * 16);
  uint32_t x_src[2 * MT], w_src[2 * RT];
#pragma unroll
  for (int i = 0; i < 2 * MT; ++i) {
    const int t = tok0 + min(8 * i + (lane >> 3), live - 1);
    x_src[i] = (uint32_t)(p.a_rows != nullptr ? p.a_rows[t] : t) * (uint32_t)(K * 2) + of_row;
  }
#pragma unroll
  for (int i = 0; i < 2 * RT; ++i) {
    const int ct = (i >> 1) % CT, up = (i >> 1) >= CT ? half : 0;  // (past the end: the last one, not stored)
    if (tiled) {
      const int tile = min((n0 >> 4) + ct, ((SWIGLU ? half : Nout) >> 4) - 1) + (up >> 4);
      w_src[i] = (uint32_t)tile * (uint32_t)(K * 32) + (uint32_t)((i & 1) * 1024 + lane * 16);
    } else {
      const int row = min(n0 + 16 * ct + 8 * (i & 1) + (lane >> 3), (SWIGLU ? half : Nout) - 1) + up;
      w_src[i] = (uint32_t)row * (uint32_t)(K * 2) + of_row;
    }
  }
  wait_loads<0>();  // the rows' numbers have come; from here on only the stages' loads count
  // This wavefront's lines: every fourth in the block's order, which starts at another line every 64 rows of W (blocks that
  // run together then read other channels of the memory) - by the place in W alone, so that a row's sums are formed in the
  // same order whatever the tiles.
  const int lines = K / kLine;
  const int stages = lines > wave ? (lines - wave - 1) / kWaves + 1 : 0;
  const int first = (int)(((unsigned)(n0 >> (SWIGLU ? 5 : 6)) * 17u) % (unsigned)lines);
  const int w_line = tiled ? 1024 : kLine;
  auto ask = [&](int s) __attribute__((always_inline)) {
    int line = wave + s * kWaves + first;
    if (line >= lines) line -= lines;
    const uint32_t to = mine + (uint32_t)((s % DEPTH) * STAGE);
#pragma unroll
    for (int i = 0; i < 2 * RT; ++i) load_to_lds16_once(We + (size_t)line * w_line, w_src[i], to + (uint32_t)(i * 1024));
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i)
      load_to_lds16(p.X + (size_t)line * kLine, x_src[i], to + (uint32_t)(RT * kPiece + i * 1024));
  };
  const int r = lane & 15, g = lane >> 4;
  const uint32_t rd = (uint32_t)(r * 128 + ((g ^ (r & 7)) * 16));  // (the line's second half: bit 6 the other way)
  const uint32_t w_rd[2] = {tiled ? (uint32_t)(lane * 16) : rd, tiled ? (uint32_t)(1024 + lane * 16) : rd ^ 64u};
  f32x4 acc[RT][MT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[i][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto work = [&](int s) __attribute__((always_inline)) {
    const unsigned char* at = ring + (s % DEPTH) * STAGE;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8 a[RT], b[MT];
#pragma unroll
      for (int i = 0; i < RT; ++i) a[i] = *reinterpret_cast<const bf16x8*>(at + i * kPiece + w_rd[ks]);
#pragma unroll
      for (int m = 0; m < MT; ++m) b[m] = *reinterpret_cast<const bf16x8*>(at + (RT + m) * kPiece + (rd ^ (ks * 64)));
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[i][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[m], acc[i][m], 0, 0, 0);
    }
  };
#pragma unroll
  for (int s = 0; s < DEPTH - 1; ++s)
    if (s < stages) ask(s);
  int s = 0;
  for (; s + DEPTH - 1 < stages; ++s) {
    // (the place that is filled now was read a stage ago: those reads have come)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    ask(s + DEPTH - 1);
    wait_loads<(DEPTH - 1) * PER>();
    work(s);
  }
  wait_loads<0>();
  for (; s < stages; ++s) work(s);

  // the wavefronts' sums, added up in their order
  __syncthreads();
  f32x4* red = reinterpret_cast<f32x4*>(smem);
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int m = 0; m < MT; ++m) red[(wave * RT * MT + i * MT + m) * 64 + lane] = acc[i][m];
  __syncthreads();
  auto total = [&](int at) __attribute__((always_inline)) {
    f32x4 v = red[at];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) v += red[w * RT * MT * 64 + at];
    return v;
  };
  // a lane finishes four neighbouring columns of a row of a tile: element j is weight row 4 g + j, row r of X
  const int width = SWIGLU ? half : Nout;
  for (int at = threadIdx.x; at < CT * MT * 64; at += kWaves * 64) {
    const int tile = at >> 6, i = tile / MT, m = tile - i * MT;
    const int row = m * 16 + r;
    if (row >= live) continue;
    const int t = tok0 + row;
    const float sc = p.scale != nullptr ? p.scale[t] : 1.f;
    f32x4 v = total(at) * sc;
    if (SWIGLU) {
      const f32x4 up = total(at + CT * MT * 64) * sc;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float x = v[j];
        v[j] = (p.act == 1 ? 0.5f * x * (1.0f + tanhf(0.7978845608028654f * (x + 0.044715f * x * x * x))) : x / (1.0f + expf(-x))) * up[j];
      }
    } else if (p.act == 1) {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = relu2(rounded<OutT>(v[j]));
    }
    const int c = n0 + i * 16 + 4 * g;
    OutT* y = (OutT*)p.Y + (size_t)t * width + c;
    if (width % 4 == 0) {
      if (c < width) store4<OutT>(y, v);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (c + j < width) Num<OutT>::store(y + j, v[j]);
    }
  }
}

// The tiles of a block.  What a compute unit reads of W and X together sets the time: rounds of blocks on the 256 compute
// units times the tiles that a block reads (2,048 x 2,048, 64 rows: 1 of W with 2 of X, 256 blocks, 6.0 us; 2 with 2 7.1,
// 1 with 4 7.7, 1 with 1 in two rounds 6.9; 8,192 x 2,048: 2 with 4 11.1, 4 with 2 11.2, 2 with 2 13.9, 1 with 2 17.2).
// Where there are many rounds anyway (an output head) and one tile of X, two of W, so that two blocks fit a compute unit and
// one's end hides behind the other: a tiled head of 50,000 x 3,072, 1 row 57 us with four, 52 with two (gemm_skinny 49), 8 rows
// 57 and 52 (55); 32,000 x 2,048, 1 row 25.2 and 23.2 (23.2).  Row-major matrices of up to two rounds are as fast with four.
// In groups likewise: two of W (8 groups of 4,096 x 2,048 with 128 rows: 2 with 2 24.5 us, 4 with 2 27.3, 2 with 1 30.5), and
// tiles of X that hold a group's rows, which scatter about their mean by its root or more (a second tile reads the weights
// again: gate and up of 8 of 14,336 x 4,096 with a dozen rows a group 160 us with one, 145 with two, 152 in gemm_skinny);
// four of W only beside four of X, where a block has the compute unit to itself either way (4 groups of 16,384 x 5,120, gate and
// up, with 128 rows 124 us, with two of W 153).  Up to a few rows a group one of W, three blocks a compute unit (us, one
// | two | gemm_skinny: a token's expert and the shared one of 5,120 x 8,192 32.6 | 36.1 | 33.6; 2 tokens, top 2, and the shared
// expert of 3,072 x 4,096 21.5 | 22.4 | 21.3, of 2,048 x 4,096 16.2 | 17.0 | 15.8); not where rows of W are short, whose blocks
// are over too soon (64 groups of 4,096 x 1,408, 16 choices 33.7 | 33.0), and not with more rows (16 groups of 7,168 x 2,048, 128
// choices 84.8 | 77.8).
struct Tiles {
  int mt, rt;
};

Tiles few_tiles(int M, int width, int K, bool swiglu, int G, bool grouped, bool tiled) {
  const int tiles = (width + 15) / 16 * (swiglu ? 2 : 1);  // of W's rows
  const int least = swiglu ? 2 : 1;
  if (grouped) {
    const int used = G < M ? G : M;
    const float mean = (float)M / (float)used;
    const int mt = mean < 12.f ? 1 : mean + sqrtf(mean) <= 32.f ? 2 : 4;
    const long long pairs = (long long)((tiles + 1) / 2) * used;
    if (mt == 1 && !swiglu && K >= 2048 && mean < 6.f) return {1, 1};
    return {mt, mt == 4 && pairs >= 512 ? 4 : pairs >= 256 ? 2 : least};
  }
  Tiles best = {0, 0};
  long long least_cost = 0;
  for (int mt = 1; mt <= 4; mt *= 2) {
    if (mt > 1 && M <= 8 * mt) break;
    for (int rt = least; rt <= 4; rt *= 2) {
      if (mt == 1 && rt == 4 && !swiglu && (tiled || tiles > 4 * 512)) break;
      const long long blocks = (long long)((tiles + rt - 1) / rt) * ((M + 16 * mt - 1) / (16 * mt));
      const long long cost = (blocks + 255) / 256 * (mt + rt);
      if (best.mt == 0 || cost < least_cost || (cost == least_cost && mt > best.mt)) {
        best = {mt, rt};
        least_cost = cost;
      }
    }
  }
  return best;
}

template <int MT, int RT, int DEPTH, bool SWIGLU, typename OutT>
int launch_few(const FewArgs& p, int max_rows, int zdim, hipStream_t s) {
  constexpr size_t lds = (size_t)kWaves * DEPTH * (MT + RT) * kPiece;
  constexpr int cols = 16 * (SWIGLU ? RT / 2 : RT);
  const dim3 grid(((SWIGLU ? p.Nout / 2 : p.Nout) + cols - 1) / cols, (max_rows + 16 * MT - 1) / (16 * MT), zdim);
  if (grid.y > 65535) return JLE_BAD_ARG;
  if (int rc = allow_lds(gemm_few_kernel<MT, RT, DEPTH, SWIGLU, OutT>, lds)) return rc;
  hipLaunchKernelGGL((gemm_few_kernel<MT, RT, DEPTH, SWIGLU, OutT>), grid, dim3(kWaves * 64), lds, s, p);
  JLE_LAUNCH_CHECK();
  return 0;
}

template <bool SWIGLU, typename OutT>
int pick_few(const FewArgs& p, Tiles t, int max_rows, int zdim, hipStream_t s) {
#define GO(MT, RT, DEPTH) \
  if (t.mt == MT && t.rt == RT) return launch_few<MT, RT, DEPTH, SWIGLU, OutT>(p, max_rows, zdim, s)
  if constexpr (!SWIGLU) {
    GO(1, 1, 3);
    GO(2, 1, 2);
    GO(4, 1, 2);
  }
  GO(1, 2, 3);
  GO(1, 4, 2);
  GO(2, 2, 2);
  GO(2, 4, 2);
  GO(4, 2, 2);
  GO(4, 4, 2);
#undef GO
  return JLE_BAD_ARG;
}

}  // namespace

// The tiles that jle_gemm_few takes by itself: row tiles of X * 10 + of W.
JLE_API int jle_gemm_few_tiles(int M, int Nout, int K, int G, int swiglu, int grouped, int tiled) {
  const Tiles t = few_tiles(M, swiglu ? Nout / 2 : Nout, K, swiglu != 0, G, grouped != 0, tiled != 0);
  return t.mt * 10 + t.rt;
}

// X [*, K] bf16, W [G, Nout, K] bf16 (row-major, or in the streaming layout: tiled), Y [M, Nout] (or [M, Nout / 2] with
// swiglu) bf16 or float32.  swiglu 0: plain, with act 1 max(., 0)^2; 1: silu(gate) * up; 2: gelu_tanh(gate) * up.
// max_rows: the most rows a group can have (M if unknown).  W_last, tiled_last: the last of the G groups' matrix, if it lies
// elsewhere (W then holds G - 1).  slots > 0: no more groups have rows than that.  tiles: 0, or row tiles of X * 10 + of W.
JLE_API int jle_gemm_few(const void* X, const void* W, void* Y, const int* offsets, const int* a_rows, const float* scale,
                         int swiglu, int act, int out_f32, int M, int Nout, int K, int G, int max_rows, int tiled,
                         const void* W_last, int tiled_last, int slots, int tiles, hipStream_t s) {
  if (M <= 0 || Nout <= 0) return 0;
  if (K < kLine || K % kLine || G < 1 || G > 65535 || (swiglu && Nout % 2)) return JLE_BAD_ARG;
  if ((((uintptr_t)X | (uintptr_t)W | (uintptr_t)W_last | (uintptr_t)Y) & 15) != 0) return JLE_BAD_ARG;
  if ((long long)Nout * K >= (1ll << 31)) return JLE_BAD_ARG;  // (a group's matrix is addressed with 32 bits)
  if (slots < 0 || (slots > 0 && (offsets == nullptr || slots > G))) return JLE_BAD_ARG;
  if (W_last != nullptr && (offsets == nullptr || G < 2)) return JLE_BAD_ARG;
  if ((tiled || (W_last != nullptr && tiled_last)) && (Nout % 16 || (swiglu && (Nout / 2) % 16))) return JLE_BAD_ARG;
  if (max_rows <= 0 || max_rows > M) max_rows = M;
  const FewArgs p = {(const bf16_t*)X, (const bf16_t*)W, Y, offsets, a_rows, scale, (const bf16_t*)W_last, M, Nout, K, G,
                     tiled, tiled_last, slots, swiglu ? swiglu - 1 : act};
  const Tiles t = tiles ? Tiles{tiles / 10, tiles % 10} : few_tiles(M, swiglu ? Nout / 2 : Nout, K, swiglu != 0, G, offsets != nullptr, tiled);
  const int zdim = slots > 0 ? slots : G;
  if (swiglu) return out_f32 ? pick_few<true, float>(p, t, max_rows, zdim, s) : pick_few<true, bf16_t>(p, t, max_rows, zdim, s);
  return out_f32 ? pick_few<false, float>(p, t, max_rows, zdim, s) : pick_few<false, bf16_t>(p, t, max_rows, zdim, s);
}
