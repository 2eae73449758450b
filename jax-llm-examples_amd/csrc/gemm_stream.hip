// Weight-streaming grouped matrix product for a moderate number of rows per group (prefill through
// experts: around a hundred tokens per expert): bfloat16 in, float32 accumulate on MFMA.
//
//   Y[t, n] = scale[t] * sum_k X[arow(t), k] * W[g(t)][n, k]          (plain; optionally max(., 0)^2 of the rounded sum)
//   Y[t, f] = silu(s * gate) * (s * up),  gate/up = rows f and F + f of W[g(t)]   (SWIGLU, s = scale[t])
//
// With so few rows the cost is reading W, and every element of W is needed by one wavefront only if
// that wavefront holds ALL rows of the group.  So a wavefront owns two 16-row tiles of W (SWIGLU: a
// gate tile and its up tile) and up to 192 rows of the group: the weights go from memory straight into
// the A operand (streaming layout: one contiguous kilobyte per load instruction, tiles along K contiguous)
// and are used once; the rows of X are what the wavefronts of a block share, through shared memory, 64 k
// at a time, laid out as the B operands are read (with the 16 rows of a piece swizzled so that neither
// writing nor reading collides).  A stage's weights are asked for four stages ahead (they come from memory,
// and every wavefront of the block waits for the slowest at every stage), its rows two stages ahead (they
// come from the cache after the first block that used them).  K must be a multiple of 256: whole rounds of
// four stages.  Groups with more than 192 rows are done in passes (each reads the weights again).
//
// Work items are (group, pass, block of WAVES * 32 weight rows), the last fastest, so the blocks of a group
// are dealt to all dies in turn and a group with many rows slows all of them alike; where a group's blocks are no multiple of
// the eight dies and there are up to two rounds of items, (pass, group, block) (locate).  How many there are is known on the
// device only (Items): every block counts the groups' passes itself, so that items are those with rows and nothing else.
// (The grid once had an item for every pass that any group could have: those without rows lay between those with, and where
// their number was even only some of the chiplets got work: 64 groups of 256 x 2,048 with 190 rows 328 us, counted 48; 32 of
// 1,536 x 2,048, gate and up, with 48 rows 78 -> 41; 12 of 2,560 x 6,144 with 250 237 -> 108.)
// A block has a compute unit to itself, and those left over behind the last full round keep a few of them busy for a round's
// time.  So some blocks of W, the last ones of every group, are cut along k into as many pieces as the round has places, whose
// float32 sums add_pieces_kernel adds up in their order and finishes (CUT).  Which blocks these are is known before the launch,
// from the numbers of groups and of their blocks: a row's sums have one order whatever rows lie beside it.
#include "common.h"
#include "dense_block.h"

using namespace jle;

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;

namespace {

constexpr int kRows = 192;       // rows of a pass
constexpr int BK = 64;           // k per stage (two MFMA steps)
constexpr int XAHEAD = 2;        // stages between asking for rows and using them (two register sets, two buffers)
constexpr int WAHEAD = 4;        // the same for weights (four register sets)

template <typename OutT>
__device__ __forceinline__ void store4(OutT* p, float a, float b, float c, float d);
template <>
__device__ __forceinline__ void store4<float>(float* p, float a, float b, float c, float d) {
  *reinterpret_cast<f32x4*>(p) = f32x4{a, b, c, d};
}
template <>
__device__ __forceinline__ void store4<bf16_t>(bf16_t* p, float a, float b, float c, float d) {
  *reinterpret_cast<uint2*>(p) = uint2{pack_bf16(a, b), pack_bf16(c, d)};
}

// The work items of a launch, found by every wavefront for itself: each group has its rows in tiles of at most `most`, times
// nblk blocks of its weights.  64 groups a look, the items before each by a sum over the lanes.
struct Items {
  const int* offsets;  // null: one group of M rows
  int M, G, nblk, most;

  __device__ __forceinline__ int rows_of(int g) const {
    return offsets == nullptr ? M : g < G ? offsets[g + 1] - offsets[g] : 0;
  }
  __device__ __forceinline__ int tiles_of_all() const {
    if (offsets == nullptr) return (M + most - 1) / most;
    const int lane = threadIdx.x & 63;
    int n = 0;
    for (int g0 = 0; g0 < G; g0 += 64) n += (rows_of(g0 + lane) + most - 1) / most;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
    return __builtin_amdgcn_readfirstlane(n);
  }
  // Item `left`'s group (-1: no such item), how many tiles the group has, and which of the group's items it is.
  __device__ __forceinline__ int find(int& left, int& tiles) const {
    if (offsets == nullptr) {
      tiles = (M + most - 1) / most;
      return left < tiles * nblk ? 0 : -1;
    }
    const int lane = threadIdx.x & 63;
    for (int g0 = 0; g0 < G; g0 += 64) {
      const int mine = (rows_of(g0 + lane) + most - 1) / most;
      int upto = mine * nblk;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(upto, o, 64);
        if (lane >= o) upto += v;
      }
      const unsigned long long mask = __ballot(left < upto);
      if (mask != 0) {
        const int at = __ffsll((long long)mask) - 1;
        tiles = __builtin_amdgcn_readfirstlane(__shfl(mine, at, 64));
        left = __builtin_amdgcn_readfirstlane(left - __shfl(upto, at, 64) + tiles * nblk);
        return __builtin_amdgcn_readfirstlane(g0 + at);
      }
      left -= __shfl(upto, 63, 64);
    }
    return -1;
  }
  // Up to 64 groups whose numbers of tiles differ from the first one's by one at most.
  __device__ __forceinline__ bool even() const {
    const int mine = (rows_of(threadIdx.x & 63) + most - 1) / most, of = __builtin_amdgcn_readfirstlane(mine);
    return G <= 64 && __ballot((int)(threadIdx.x & 63) < G && (mine > of + 1 || mine < of - 1)) == 0;
  }
  // find() of such groups with every group's first tile before all second ones (see locate).
  __device__ __forceinline__ int find_by_tile(int& left, int& tiles) const {
    const int mine = (rows_of(threadIdx.x & 63) + most - 1) / most;
    for (int t = 0;; ++t) {
      unsigned long long mask = __ballot(mine > t);
      const int n = __popcll(mask);
      if (n == 0) return -1;
      if (left < n * nblk) {
        for (int j = left / nblk; j > 0; --j) mask &= mask - 1;  // drop the lower set bits
        const int g = __ffsll((long long)mask) - 1;
        tiles = __builtin_amdgcn_readfirstlane(__shfl(mine, g, 64));
        left = __builtin_amdgcn_readfirstlane(left % nblk + t * nblk);
        return __builtin_amdgcn_readfirstlane(g);
      }
      left -= n * nblk;
    }
  }
};

// The stages that a piece of a cut item begins at: whole rounds of four.
__device__ __forceinline__ int piece_stage(int piece, int cuts, int nstage) { return nstage / WAHEAD * piece / cuts * WAHEAD; }

// Rows of a tile: a group's rows as even as multiples of 32 allow.
__device__ __forceinline__ int rows_a_tile(int rows, int tiles) { return ((rows + tiles - 1) / tiles + 31) / 32 * 32; }

// A lane's sums of a row, four neighbouring rows of two tiles of W, scaled and stored.
template <bool SWIGLU, typename OutT>
__device__ __forceinline__ void finish_pair(OutT* __restrict__ Y, int t, const float* __restrict__ scale, int act, f32x4 a0,
                                            f32x4 a1, int Nout, int t0, int t1, int g) {
  const float sc = scale != nullptr ? scale[t] : 1.f;
  a0 *= sc;
  a1 *= sc;
  if (SWIGLU) {
    float y[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = a0[i] / (1.0f + expf(-a0[i])) * a1[i];
    store4<OutT>(Y + (size_t)t * (Nout >> 1) + t0 * 16 + 4 * g, y[0], y[1], y[2], y[3]);
  } else {
    if (act) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a0[i] = relu2(Num<OutT>::round(a0[i]));
        a1[i] = relu2(Num<OutT>::round(a1[i]));
      }
    }
    store4<OutT>(Y + (size_t)t * Nout + t0 * 16 + 4 * g, a0[0], a0[1], a0[2], a0[3]);
    if (t1 != t0) store4<OutT>(Y + (size_t)t * Nout + t1 * 16 + 4 * g, a1[0], a1[1], a1[2], a1[3]);
  }
}

// The work of one block once it knows its rows and tiles; NTL = B tiles (of 16 rows) that hold live rows, even
// (the rows are brought in by whole rounds of the block's threads, 64 rows each: a round's rows past the live
// tiles land in tiles that nobody reads).  The main loop has no branch but its own: every load is asked for unconditionally (rows past
// the live ones read the pass's first row again, into their own places), so that the waits for the loads of
// two stages ago never include the loads asked for since.
template <bool SWIGLU, typename OutT, int WAVES, bool CUT, int NTL>
__device__ __forceinline__ void stream_block(const bf16_t* __restrict__ X, const bf16_t* __restrict__ w0,
                                             const bf16_t* __restrict__ w1, OutT* __restrict__ Y,
                                             const int* __restrict__ a_rows, const float* __restrict__ scale, int act,
                                             bf16_t (&sX)[2][kRows * BK], int tok0, int live, int K, int Nout, int t0,
                                             int t1, bool wave_ok, int first, int nstage, f32x4* __restrict__ piece) {
  constexpr int THREADS = WAVES * 64;
  constexpr int CHUNKS = NTL * 16 * (BK / 8);            // 16-byte pieces of X per stage
  constexpr int CPT = (CHUNKS + THREADS - 1) / THREADS;  // per thread
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  if constexpr (CUT) {  // (this block's stages: nstage of them, a multiple of 4)
    X += (size_t)first * BK;
    w0 += (size_t)first * 1024;
    w1 += (size_t)first * 1024;
  }

  // who brings which pieces of X: piece c is 8 k of row c / 8, 8 consecutive threads a row's 128 bytes
  uint32_t xsrc[CPT];  // elements from X (the host checks that X has fewer than 2^32)
  int xdst[CPT];
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int c = threadIdx.x + THREADS * i;
    const int row = (c >> 3) % kRows, kc = c & 7;  // (past the buffer only if CHUNKS is no multiple of THREADS)
    const int t = row < live ? tok0 + row : tok0;
    xsrc[i] = (uint32_t)(a_rows != nullptr ? a_rows[t] : t) * (uint32_t)K + kc * 8;
    // B operand order: [tile][k step][g][row], the row swizzled by (g, k step)
    const int nt = row >> 4, rr = row & 15, ks = kc >> 2, gg = kc & 3;
    xdst[i] = (((nt * 2 + ks) * 4 + gg) * 16 + (rr ^ (gg + 4 * ks))) * 8;
  }
  // what this lane reads as B operand: tile nt, k step ks at b_off[ks] + nt * 1024 elements
  int b_off[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) b_off[ks] = ((ks * 4 + g) * 16 + (r ^ (g + 4 * ks))) * 8;

  f32x4 acc0[NTL], acc1[NTL];
#pragma unroll
  for (int nt = 0; nt < NTL; ++nt) {
    acc0[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    acc1[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // registers on their way: the pieces of X of two stages (even and odd), the weights [k step][tile] of four
  u32x4 xa[CPT], xb[CPT], wa[2][2], wb[2][2], wc[2][2], wd[2][2];
  auto ask_rows = [&](u32x4 (&x)[CPT], int s) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) x[i] = *reinterpret_cast<const u32x4*>(X + xsrc[i] + (size_t)s * BK);
  };
  auto ask_weights = [&](u32x4 (&w)[2][2], int s) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      // (read by this wavefront alone, once: loads that the caches need not keep, which stream faster)
      w[ks][0] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(w0 + (size_t)(2 * s + ks) * 512));
      w[ks][1] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(w1 + (size_t)(2 * s + ks) * 512));
    }
  };
  auto put = [&](const u32x4 (&x)[CPT], bf16_t* buf) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) *reinterpret_cast<u32x4*>(buf + xdst[i]) = x[i];
  };
  auto work = [&](const u32x4 (&w)[2][2], const bf16_t* buf) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const bf16x8 a0 = __builtin_bit_cast(bf16x8, w[ks][0]);
      const bf16x8 a1 = __builtin_bit_cast(bf16x8, w[ks][1]);
#pragma unroll
      for (int nt = 0; nt < NTL; ++nt) {
        const u32x4 bv = *reinterpret_cast<const u32x4*>(buf + b_off[ks] + nt * 1024);
        const bf16x8 b = __builtin_bit_cast(bf16x8, bv);
        acc0[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b, acc0[nt], 0, 0, 0);
        acc1[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b, acc1[nt], 0, 0, 0);
      }
    }
  };
  // One stage: the rows that came two stages ago go to shared memory; then the registers they were in ask for
  // the rows of two stages on; the stage's weights, asked for four stages ago, are used and ask for those of
  // four stages on.
#define STAGE(x_, w_, buf_, s_, ASKX, ASKW)                  \
  do {                                                       \
    put(x_, sX[buf_]);                                       \
    __syncthreads();                                         \
    if (ASKX) ask_rows(x_, (s_) + XAHEAD);                   \
    __builtin_amdgcn_sched_barrier(0);                       \
    work(w_, sX[buf_]);                                      \
    if (ASKW) ask_weights(w_, (s_) + WAHEAD);                \
  } while (0)

  ask_weights(wa, 0);
  ask_rows(xa, 0);
  ask_weights(wb, 1);
  ask_rows(xb, 1);
  ask_weights(wc, 2);
  ask_weights(wd, 3);
  int s = 0;
  for (; s < nstage - WAHEAD; s += WAHEAD) {
    STAGE(xa, wa, 0, s, true, true);
    STAGE(xb, wb, 1, s + 1, true, true);
    STAGE(xa, wc, 0, s + 2, true, true);
    STAGE(xb, wd, 1, s + 3, true, true);
  }
  STAGE(xa, wa, 0, s, true, false);
  STAGE(xb, wb, 1, s + 1, true, false);
  STAGE(xa, wc, 0, s + 2, false, false);
  STAGE(xb, wd, 1, s + 3, false, false);
#undef STAGE
  if (!wave_ok) return;
  if constexpr (CUT) {
    if (piece != nullptr) {  // a piece of k: its sums as they are
#pragma unroll
      for (int nt = 0; nt < NTL; ++nt) {
        piece[(nt * WAVES * 2 + (threadIdx.x >> 6) * 2) * 64 + lane] = acc0[nt];
        piece[(nt * WAVES * 2 + (threadIdx.x >> 6) * 2 + 1) * 64 + lane] = acc1[nt];
      }
      return;
    }
  }

  // accumulators: element i of tile nt in lane (g, r) = weight row 4 g + i of the tile, row 16 nt + r of the pass
#pragma unroll
  for (int nt = 0; nt < NTL; ++nt) {
    const int row = nt * 16 + r;
    if (row >= live) continue;
    finish_pair<SWIGLU>(Y, tok0 + row, scale, act, acc0[nt], acc1[nt], Nout, t0, t1, g);
  }
}

struct StreamArgs {
  const bf16_t* X;
  const bf16_t* W;
  void* Y;
  const int* a_rows;
  const float* scale;
  Items items;
  f32x4* pieces;        // CUT: the sums of the last `cut` blocks of every group, each in `cuts` pieces of k
  int cut, cuts, room;  // room: tiles of 16 rows that a piece of one of the blocks has place for, of all passes
  int Nout, K, units, act;
};

// Item `left`'s group, how many passes the group has, and which of the group's items it is.
// The passes of a block of W are to run on one die, whose cache then has the weights for the second one.  Items are dealt to
// the eight dies in turn, so they do group after group if a group's blocks are a multiple of eight; else every group's first
// pass comes before all second ones.  Group after group | so, us: 16 groups of 1,024 x 4,096 (four blocks) with 250 rows
// 73 | 62, 400 99 | 85, 600 117 | 96; 32 of 1,024 x 2,048 with 300 86 | 60; 64 of 512 x 1,024 with 300 48 | 39; 12 of
// 2,560 x 6,144 (ten) with 250 155 | 116; but 8 of 4,096 x 2,048 (sixteen) with 450 85 | 91, 570 99 | 104, 700 107 | 121.  Where one
// group has most of the rows its last tiles would come last (16 of 5,120 x 8,192 with 128, 40 % in one, 287 | 352).
__device__ __forceinline__ int locate(const StreamArgs& p, int& left, int& passes) {
  const Items& it = p.items;
  if (it.offsets == nullptr || it.nblk % 8 == 0) return it.find(left, passes);
  const int items = it.tiles_of_all() * it.nblk;
  if (left >= items) return -1;
  return items <= 2 * p.units && it.even() ? it.find_by_tile(left, passes) : it.find(left, passes);
}

// The rows of item `left` of a group with `tiles` passes, the first of its block's pairs of tiles of W
struct Pass {
  int tok0, live, nb;

  __device__ __forceinline__ Pass(const Items& it, int e, int left, int tiles) {
    nb = left % it.nblk;
    const int lo = it.offsets == nullptr ? 0 : it.offsets[e], rows = it.rows_of(e), per = rows_a_tile(rows, tiles);
    tok0 = lo + left / it.nblk * per;
    live = min(per, rows - left / it.nblk * per);
  }
};

// The two tiles of W of wavefront `wave` of block nb; false: behind the last one.
template <bool SWIGLU, int WAVES>
__device__ __forceinline__ bool tiles_of(int nb, int wave, int Nout, int& t0, int& t1) {
  const int ntile = (SWIGLU ? Nout >> 1 : Nout) >> 4;
  const int ft = SWIGLU ? nb * WAVES + wave : (nb * WAVES + wave) * 2;
  t0 = ft < ntile ? ft : 0;
  t1 = SWIGLU ? ntile + t0 : min(t0 + 1, ntile - 1);
  return ft < ntile;
}

// A block of a CUT launch: the whole items come first, then the first pieces of all cut ones, their second pieces, and so on.
struct CutItem {
  Items items;         // of which it is one: the whole or the cut blocks of the groups
  int at, piece, nb0;  // which one, which piece (-1: whole), the first of the groups' blocks that are meant

  __device__ __forceinline__ CutItem(const StreamArgs& p, int block) : items(p.items), at(block), piece(-1), nb0(0) {
    const int passes = items.tiles_of_all(), whole = passes * (items.nblk - p.cut), a_piece = passes * p.cut;
    if (block < whole) {
      items.nblk -= p.cut;
      return;
    }
    nb0 = items.nblk - p.cut;
    items.nblk = p.cut;
    piece = a_piece > 0 ? (block - whole) / a_piece : p.cuts;
    at = block - whole - piece * a_piece;
  }
};

// Where the sums of a piece of cut item `at` begin, whose rows begin at tok0.  The tiles of rows of all passes lie behind each
// other; a pass of n rows has 2 * ceil(n / 32) of them, no more than floor(n / 16) + 2.
__device__ __forceinline__ f32x4* piece_sums(const StreamArgs& p, int piece, int at, int tok0) {
  return p.pieces + ((size_t)(piece * p.cut + at % p.cut) * p.room + (tok0 >> 4) + 2 * (at / p.cut)) * 1024;
}

template <bool SWIGLU, typename OutT, int WAVES, bool CUT>
__global__ __launch_bounds__(WAVES * 64, 2) void gemm_stream_kernel(StreamArgs p) {
  static_assert(WAVES == 8, "a tile of a piece's sums is 16 rows by 256 of W");
  __shared__ __attribute__((aligned(16))) bf16_t sX[2][kRows * BK];
  const int K = p.K, Nout = p.Nout;
  int e, left = blockIdx.x, passes, nb0 = 0, first = 0, stages = K / BK, at_piece = -1, item = 0;
  if constexpr (CUT) {
    const CutItem c(p, left);
    if (c.piece >= p.cuts) return;
    p.items = c.items;
    nb0 = c.nb0;
    at_piece = c.piece;
    left = item = c.at;
    e = p.items.find(left, passes);
    if (at_piece >= 0) {
      first = piece_stage(at_piece, p.cuts, K / BK);
      stages = piece_stage(at_piece + 1, p.cuts, K / BK) - first;
    }
  } else {
    e = locate(p, left, passes);
  }
  if (e < 0) return;  // (the grid is laid out for the most items that so many rows can make)
  const Pass at(p.items, e, left, passes);
  const int tok0 = at.tok0, live = at.live, nb = nb0 + at.nb;
  f32x4* piece = nullptr;
  if constexpr (CUT) {
    if (at_piece >= 0) piece = piece_sums(p, at_piece, item, tok0);
  }
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int nkb = K >> 5;
  const bf16_t* We = p.W + (size_t)e * Nout * K;
  int t0, t1;
  const bool wave_ok = tiles_of<SWIGLU, WAVES>(nb, wave, Nout, t0, t1);
  const bf16_t* w0 = We + (size_t)t0 * nkb * 512 + lane * 8;
  const bf16_t* w1 = We + (size_t)t1 * nkb * 512 + lane * 8;
#define GO(NTL_) \
  stream_block<SWIGLU, OutT, WAVES, CUT, NTL_>(p.X, w0, w1, (OutT*)p.Y, p.a_rows, p.scale, p.act, sX, tok0, live, K, Nout, t0, \
                                               t1, wave_ok, first, stages, piece)
  if (live <= 32) GO(2);
  else if (live <= 64) GO(4);
  else if (live <= 96) GO(6);
  else if (live <= 128) GO(8);
  else if (live <= 160) GO(10);
  else GO(12);
#undef GO
}

// The cut items' pieces, added up in their order and finished: blockIdx.x is the item, blockIdx.y which of its tiles of rows.
template <typename OutT, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void add_pieces_kernel(StreamArgs p) {
  const int nb0 = p.items.nblk - p.cut;
  p.items.nblk = p.cut;
  int left = blockIdx.x, passes;
  const int e = p.items.find(left, passes);
  if (e < 0) return;
  const Pass at(p.items, e, left, passes);
  const int lane = threadIdx.x & 63, r = lane & 15, wave = wave_index();
  int t0, t1;
  if (!tiles_of<false, WAVES>(nb0 + at.nb, wave, p.Nout, t0, t1)) return;
  for (int nt = blockIdx.y; nt * 16 < at.live; nt += gridDim.y) {
    const f32x4* from = piece_sums(p, 0, blockIdx.x, at.tok0) + (nt * WAVES * 2 + wave * 2) * 64 + lane;
    f32x4 a0 = from[0], a1 = from[64];
    for (int i = 1; i < p.cuts; ++i) {
      from += (size_t)p.cut * p.room * 1024;
      a0 += from[0];
      a1 += from[64];
    }
    if (nt * 16 + r < at.live)
      finish_pair<false>((OutT*)p.Y, at.tok0 + nt * 16 + r, p.scale, p.act, a0, a1, p.Nout, t0, t1, lane >> 4);
  }
}

// ------------------------------------------------------------------ groups of many rows
// A block of dense_block.h takes 32 * FN rows of W (SWIGLU: half of them gate rows, half their up rows) and up to 256 (FN = 4:
// 288) rows of a group.  A group's rows are cut into tiles as even as multiples of 32 allow, and a block multiplies no more than
// its tile has (full tiles and what is left instead: 8 groups of 14,336 x 4,096, gate and up, with 300 rows 298 -> 400 us).
// Work items: item = ((row block / 8) * tiles + tile) * 8 + row block % 8 within a group, so that the tiles that read the
// same weights run on one chiplet.  All blocks go through k from its beginning: begun elsewhere by row block, so that they read
// other channels of the memory, they no longer find each other's rows of X in the caches (with 410 rows 403 -> 490).
// In us, drawn groups, passes of 192 | tiles whose weights went straight into registers, X through a ring in shared memory | these:
// gate and up of 8 of 14,336 x 4,096 with 192 rows 258 | 234 | 221, 410 483 | 389 | 364 (1.06 PFLOP/s), 700 743 | 635 | 559; 16
// of 16,384 x 5,120 with 410 1,418 | 1,032 | 968; plain, 8 of 4,096 x 7,168 with 410 256 | 186 | 172, 16 of 5,120 x 8,192 762 |
// 572 | 552; FN = 4: 8 of 2,048 x 4,096 with 192 80 | 69 | 58, 410 82 | 72 | 62, 16 of 1,024 x 2,048 with 176 46 | 41 | 35.
// What bounds them is the last round of blocks and, below some 250 rows, the weights' bytes and the products that do not quite
// overlap: with all groups' weights in the caches 410 rows take 352 for 400, 128 rows 129 for 197 (full tiles and rest).
constexpr int wide_rows(int fn) { return fn == 8 ? 256 : 288; }  // of X, of a block

struct WideArgs {
  const bf16_t* X;
  const bf16_t* W;
  bf16_t* Y;
  const int* offsets;
  const int* a_rows;
  const float* scale;
  int act, Nout, K, G, nblk8;
};

template <int FN, bool SWIGLU>
__global__ __launch_bounds__(256, 1) void wide_kernel(WideArgs p) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  constexpr int BN = SWIGLU ? FN * 16 : FN * 32;
  const Items items = {p.offsets, 0, p.G, p.nblk8, wide_rows(FN)};
  int left = blockIdx.x, tiles;
  const int e = items.find(left, tiles);
  if (e < 0) return;  // (the grid is laid out for the most tiles that so many rows can make)
  const int nb = left / (8 * tiles) * 8 + (left & 7), tile = (left >> 3) % tiles, N = SWIGLU ? p.Nout >> 1 : p.Nout;
  if (nb * BN >= N) return;
  const int rows = p.offsets[e + 1] - p.offsets[e], per = rows_a_tile(rows, tiles), lo = p.offsets[e] + tile * per, live = min(per, rows - tile * per);
  if (live <= 0) return;
  const dense::DenseBlock b = {p.X, p.W + (size_t)e * p.Nout * p.K, p.Y, nullptr, p.a_rows, p.scale, p.act, lo, live, nb * BN, N, p.K};
#define GO(FM, RX, RW) dense::dense_block<FM, FN, RX, RW, SWIGLU, true>(b, smem)
  if constexpr (FN == 8) {
    if (live <= 64) GO(2, 6, 6);
    else if (live <= 96) GO(3, 6, 6);
    else if (live <= 128) GO(4, 6, 6);
    else if (live <= 160) GO(5, 6, 6);
    else if (live <= 192) GO(6, 5, 6);
    else if (live <= 224) GO(7, 4, 6);
    else GO(8, 4, 6);
  } else {
    if (live <= 64) GO(2, 6, 6);
    else if (live <= 96) GO(3, 6, 6);
    else if (live <= 128) GO(4, 6, 6);
    else if (live <= 160) GO(5, 6, 6);
    else if (live <= 192) GO(6, 6, 6);
    else if (live <= 224) GO(7, 6, 6);
    else if (live <= 256) GO(8, 6, 6);
    else GO(9, 6, 6);
  }
#undef GO
}

template <int FN, bool SW>
int launch_wide(WideArgs p, int M, hipStream_t s) {
  constexpr uint32_t lds = 160 * 1024;  // (a compute unit's: the largest tile's rings take it all or most of it)
  static_assert(dense::dense_bytes<8, FN, 4, 6, SW>() <= lds && dense::dense_bytes<9, 4, 6, 6, SW>() <= lds, "");
  if (const int rc = allow_lds(wide_kernel<FN, SW>, lds)) return rc;
  constexpr int of8 = 8 * (SW ? FN * 16 : FN * 32);  // columns of Y of eight blocks
  p.nblk8 = ((SW ? p.Nout / 2 : p.Nout) + of8 - 1) / of8 * 8;
  const long long items = ((long long)M / wide_rows(FN) + p.G) * p.nblk8;
  if (items > (1ll << 30)) return JLE_BAD_ARG;
  hipLaunchKernelGGL((wide_kernel<FN, SW>), dim3((unsigned)items), dim3(256), lds, s, p);
  JLE_LAUNCH_CHECK();
  return 0;
}

// passes: the most that so many rows can make
template <bool SW, typename OT, int WV>
int launch_stream(const StreamArgs& p, long long passes, hipStream_t s) {
  hipLaunchKernelGGL((gemm_stream_kernel<SW, OT, WV, false>), dim3((unsigned)(passes * p.items.nblk)), dim3(WV * 64), 0, s, p);
  JLE_LAUNCH_CHECK();
  return 0;
}

template <typename OT, int WV>
int launch_cut(const StreamArgs& p, long long passes, hipStream_t s) {
  const long long blocks = passes * (p.items.nblk - p.cut + p.cut * p.cuts);
  if (blocks > (1ll << 30)) return JLE_BAD_ARG;
  hipLaunchKernelGGL((gemm_stream_kernel<false, OT, WV, true>), dim3((unsigned)blocks), dim3(WV * 64), 0, s, p);
  JLE_LAUNCH_CHECK();
  hipLaunchKernelGGL((add_pieces_kernel<OT, WV>), dim3((unsigned)(passes * p.cut), 4), dim3(WV * 64), 0, s, p);
  JLE_LAUNCH_CHECK();
  return 0;
}

}  // namespace

// Whether jle_gemm_stream takes these sizes (W must be in the streaming layout).
JLE_API int jle_gemm_stream_supported(int Nout, int K, int swiglu) {
  if (K <= 0 || K % (BK * WAHEAD)) return 0;
  if (swiglu) return Nout > 0 && Nout % 32 == 0;
  return Nout > 0 && Nout % 16 == 0;
}

// Tiles of rows that the pieces of a cut block of all groups have place for; 16 KB a tile and piece.
JLE_API int jle_gemm_stream_room(int M, int G) { return (M >> 4) + 2 * (M / kRows + G); }

// X [*, K] bf16, W [G, Nout, K] bf16 in the streaming layout, Y [M, Nout] (or [M, Nout / 2] with swiglu) bf16 or
// float32; X must have fewer than 2^32 elements (wide: 2^32 bytes).  wide: wide_kernel (groups, bfloat16 out, K below 2^23; with
// swiglu half of a group's W, and 128 rows more, have fewer than 2^32 bytes), 2 (plain): with FN = 4.
// act 1 (plain): max(., 0)^2 of the rounded sums.  cuts > 1 (plain, not wide): the last `cut` of a group's blocks of 256 rows of
// W are cut into `cuts` pieces along k; pieces: place for jle_gemm_stream_room(M, G) * cut * cuts tiles of 16 KB.
// Blocks are 8 wavefronts (two per SIMD, one block per compute unit): measured against 4, 5 and 6 on expert
// shapes with even and with skewed numbers of rows per expert.
JLE_API int jle_gemm_stream(const void* X, const void* W, void* Y, const int* offsets, const int* a_rows,
                            const float* scale, int swiglu, int act, int out_f32, int M, int Nout, int K, int G,
                            int wide, void* pieces, int cut, int cuts, int units, hipStream_t s) {
  if (M <= 0 || Nout <= 0) return 0;
  if (wide) {
    if (offsets == nullptr || out_f32 || G < 1 || G > 65535 || !jle_gemm_stream_supported(Nout, K, swiglu) ||
        K >= 1 << 23 || (swiglu && ((long long)Nout / 2 + 128) * K >= (1ll << 31)) || ((uintptr_t)X | (uintptr_t)W | (uintptr_t)Y) % 16)
      return JLE_BAD_ARG;
    const WideArgs p = {(const bf16_t*)X, (const bf16_t*)W, (bf16_t*)Y, offsets, a_rows, scale, act, Nout, K, G, 0};
    if (swiglu) return launch_wide<8, true>(p, M, s);
    return wide == 2 ? launch_wide<4, false>(p, M, s) : launch_wide<8, false>(p, M, s);
  }
  if (G < 1 || G > 65535 || (offsets == nullptr && G != 1) || !jle_gemm_stream_supported(Nout, K, swiglu)) return JLE_BAD_ARG;
  constexpr int kWaves = 8;
  const int pairs = swiglu ? Nout / 32 : (Nout / 16 + 1) / 2;  // pairs of weight tiles = wavefronts needed per group
  const int nblk = (pairs + kWaves - 1) / kWaves;
  const long long passes = offsets == nullptr ? ((long long)M + kRows - 1) / kRows : (long long)M / kRows + G;
  if (passes * nblk > (1ll << 30)) return JLE_BAD_ARG;
  const StreamArgs p = {(const bf16_t*)X, (const bf16_t*)W, Y, a_rows, scale, {offsets, M, G, nblk, kRows}, (f32x4*)pieces,
                        cut, cuts, jle_gemm_stream_room(M, G), Nout, K, units, act};
  if (cuts > 1) {
    if (swiglu || cut < 1 || cut > nblk || cuts > K / (BK * WAHEAD) || pieces == nullptr || (uintptr_t)pieces % 16)
      return JLE_BAD_ARG;
    return out_f32 ? launch_cut<float, kWaves>(p, passes, s) : launch_cut<bf16_t, kWaves>(p, passes, s);
  }
  if (swiglu) return out_f32 ? launch_stream<true, float, kWaves>(p, passes, s) : launch_stream<true, bf16_t, kWaves>(p, passes, s);
  return out_f32 ? launch_stream<false, float, kWaves>(p, passes, s) : launch_stream<false, bf16_t, kWaves>(p, passes, s);
}
