// Dense float32 products: of many rows on the bfloat16 matrix instructions, every operand as the sum of three bfloat16
// numbers, and of up to eight rows (further down).
//
//   Y[t, n] = sum_k X[t, k] * W[n, k]                                              (plain)
//   Y[t, f] = act(gate) * up, gate / up = rows f and F + f of W                    (ACT: silu or the tanh form of gelu)
//
// The float32 matrix instruction does 256 operations a cycle of a compute unit, the bfloat16 one 4,096.  A float32
// number is the sum of three bfloat16 numbers, x = h + m + l, without any loss: h is x rounded to the nearest, m what is
// left rounded to the nearest, l the rest; both differences are exact.  Of the nine products the six largest are formed
// (smallest first: h l, l h, m m, h m, m h, then h h); the three others are at most 2^-24 of a product, of either sign,
// and 2^-27 of it in the mean square.  (Cut off instead of rounded, the parts carry the number's sign: up to 2^-21 left out,
// always towards zero.)  The bfloat16 instruction's sums are not rounded to the nearest: what it drops is below the last
// place of its largest addend, always downwards.  So h h, whose products are exact, has a sum of its own beside the five
// small ones', and both are added to the whole on the vector units, once a stage: 1 rounding of the whole for 32 k, where
// the float32 instruction has one for every 4.  Against 64 bits, of the result's norm, here | the library's float32 product:
// sums of like terms 1.5e-7 | 4.1e-7 (K = 2048), 2.3e-7 | 6.4e-7 (5120), 2.9e-7 | 8.1e-7 (8192); a single term 2.6e-8 |
// 2.5e-8, at most 1.6 * 2^-24 of it | 2^-24.  (All six in one sum: a single term 3.4e-8 and a shift of 2^-26 downwards, 4 %
// faster; the parts cut off: 6.6e-8, at most 8.2 * 2^-24.)
//
// Six instructions of 16 times the rate: at best 2.7 times the float32 peak of 157 TFLOP/s.  Reached: 137 to 182 where the
// library reaches 107 to 150.  What bounds it: the matrix cores are busy about half the time; splitting (22 operations for
// 4 numbers) and the way through shared memory run beside them only as far as the other block's phases fall in between.
//
// What the parts cannot hold - infinities, NaN, numbers and partial products below 2^-126 - shows as a sum that is not
// finite, or as one too small for what may have been lost: the wavefront then forms its tile again with float32
// instructions straight from memory, and the result is what float32 arithmetic gives.
//
// A block is 128 rows of W by 128 of X, four wavefronts of 64 x 64 (a wavefront reads 24 KB of shared memory for 96
// instructions of 16 cycles: half of what shared memory gives).  32 k at a time: every thread has its 32 numbers of the next
// stage on their way in registers while the instructions of this one run, splits them (5.5 operations a number) and
// leaves them in shared memory in the order in which the operands are read: tiles of 16 rows of 1 KB a part, 16
// bytes (8 k) a lane; the 16 rows of a k-lane stand rotated by it (4 g), so that writing 8 bytes at a time (8 lanes
// a row's line of 128 bytes) spreads over the banks too.  Shared memory holds one stage (48 KB) and two blocks share
// a compute unit: one splits while the other multiplies.
#include <type_traits>

#include "common.h"
#include "gate_act.h"

using namespace jle;

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;

namespace {

constexpr int kTile = 128;              // rows of W and of X a block
constexpr int kStage = 32;              // k a stage
constexpr int kPart = kTile * kStage;   // bfloat16 numbers of a part of an operand
constexpr int kPanel = 8;               // tiles of W whose blocks run together

// four float32 numbers as three times four bfloat16 numbers, each what is left rounded to the nearest
__device__ __forceinline__ void split4(f32x4 x, u32x2 (&p)[3]) {
#pragma unroll
  for (int i = 0; i < 3; ++i) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      p[i][j] = pack_bf16(x[2 * j], x[2 * j + 1]);
      if (i < 2) {
        x[2 * j] -= __uint_as_float(p[i][j] << 16);
        x[2 * j + 1] -= __uint_as_float(p[i][j] & 0xffff0000u);
      }
    }
  }
}

// ACT: -1 plain, 0 silu, 1 gelu (tanh form): tiles 0 and 1 of a wavefront's four are gate rows, 2 and 3 their up rows
template <int ACT>
__global__ __launch_bounds__(256, 2) void gemm_f32_split_kernel(const float* __restrict__ X, const float* __restrict__ W,
                                                                float* __restrict__ Y, int M, int Nout, int ld, int nb,
                                                                int mb, int ranges, int per) {
  __shared__ __attribute__((aligned(16))) uint16_t parts[2][3][kPart];  // [W, X][part]
  __shared__ __attribute__((aligned(16))) float largest[2][kTile];      // of the rows, without their signs
  constexpr bool GATED = ACT >= 0;
  // A die's blocks are neighbours: panels of kPanel tiles of W, in a panel all tiles of X one after the other.  The
  // 64 blocks that a die runs at a time read 16 tiles instead of 128.
  const int total = nb * mb * ranges, die = blockIdx.x & 7, share = total >> 3, rem = total & 7;
  const int item = die * share + min(die, rem) + (blockIdx.x >> 3);
  const int range = item / (nb * mb), o = item - range * nb * mb;
  const int first = range * per, K = min(per, ld - first);  // the numbers of k that this block adds up
  const int panel = o / (kPanel * mb), in = o - panel * kPanel * mb;
  const int wide = min(kPanel, nb - panel * kPanel);
  const int n_tile = panel * kPanel + in % wide, m_tile = in / wide;
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int half = Nout >> 1, cols = GATED ? half : Nout;
  const int col0 = n_tile * (GATED ? kTile / 2 : kTile), row0 = m_tile * kTile;
  // row of W that is row l of the block's 128 (past the end: the last one, computed and not stored)
  auto w_row = [&](int l) {
    if (!GATED) return min(col0 + l, cols - 1);
    const int f = min(col0 + (l >> 6) * 32 + (l & 31), cols - 1);
    return f + ((l >> 5) & 1) * half;
  };
  // what this thread brings: piece lc (4 k) of rows 32 wave + 8 i + lr of W and of X
  const int lr = lane >> 3, lc = lane & 7;
  const float* src[8];
  uint32_t dst[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int l = 32 * wave + 8 * i + lr;
    src[i] = W + (size_t)w_row(l) * ld + first + 4 * lc;
    src[4 + i] = X + (size_t)min(row0 + l, M - 1) * ld + first + 4 * lc;
    dst[i] = (l >> 4) * 512 + (lc >> 1) * 128 + (((l & 15) ^ ((lc >> 1) * 4)) * 8) + (lc & 1) * 4;
  }
  const int r = lane & 15, g = lane >> 4;
  const int wm = wave & 1, wn = wave >> 1;
  const uint32_t at = g * 128 + ((r ^ (4 * g)) * 8);
  const uint16_t* a_at = &parts[0][0][wm * 4 * 512 + at];
  const uint16_t* b_at = &parts[1][0][wn * 4 * 512 + at];
  f32x4 acc[4][4];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int n = 0; n < 4; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 x[8];  // on their way: the numbers of the next stage
  float most[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};  // the largest number in this thread's pieces of the rows
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = *reinterpret_cast<const f32x4*>(src[i]);
  for (int k = 0; k < K; k += kStage) {
    __syncthreads();  // nobody reads the stage before any more
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      u32x2 p[3];
#pragma unroll
      for (int j = 0; j < 4; ++j) most[i] = fmaxf(most[i], fabsf(x[i][j]));
      split4(x[i], p);
#pragma unroll
      for (int j = 0; j < 3; ++j) *reinterpret_cast<u32x2*>(&parts[i >> 2][j][dst[i & 3]]) = p[j];
    }
    const int next = min(k + kStage, K - kStage);  // (past the end: the last stage once more, not used)
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = *reinterpret_cast<const f32x4*>(src[i] + next);
    __syncthreads();
    bf16x8 b[4][3];
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int j = 0; j < 3; ++j) b[n][j] = *reinterpret_cast<const bf16x8*>(b_at + j * kPart + n * 512);
    f32x4 sum[2][4], top[2][4];  // of the stage alone, the largest products apart from the others: added to the whole once,
                                 // not six times, while the next tile's products run
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      bf16x8 a[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) a[j] = *reinterpret_cast<const bf16x8*>(a_at + j * kPart + m * 512);
      constexpr int kOfA[5] = {0, 2, 1, 0, 1}, kOfB[5] = {2, 0, 1, 1, 0};  // smallest first
#pragma unroll
      for (int n = 0; n < 4; ++n) sum[m & 1][n] = top[m & 1][n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < 5; ++q)
#pragma unroll
        for (int n = 0; n < 4; ++n)
          sum[m & 1][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[kOfA[q]], b[n][kOfB[q]], sum[m & 1][n], 0, 0, 0);
#pragma unroll
      for (int n = 0; n < 4; ++n)
        top[m & 1][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[n][0], top[m & 1][n], 0, 0, 0);
      if (m > 0)
#pragma unroll
        for (int n = 0; n < 4; ++n) acc[m - 1][n] += top[(m - 1) & 1][n] + sum[(m - 1) & 1][n];
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int n = 0; n < 4; ++n) acc[3][n] += top[1][n] + sum[1][n];
  }
  // element i of acc[m][n] in lane (g, r): row 4 g + i of W's tile m, row r of X's tile n
  auto store = [&](int m, int row, f32x4 y) {
    const int c = col0 + (GATED ? wm * 32 : wm * 64) + m * 16 + 4 * g;
    if (row < M && c < cols) *reinterpret_cast<f32x4*>(Y + ((size_t)range * M + row) * cols + c) = y;
  };
  auto gated = [&](f32x4 gate, f32x4 up) {
    f32x4 y;
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = gate_act<GATED ? ACT : 0>(gate[i]) * up[i];
    return y;
  };
  // What float32 holds and the parts do not: parts and products of parts below 2^-126 are lost, in all no more than
  // K 2^-122 times the largest number of the two rows (or 1).  A sum that is 2^24 times as large has lost nothing; one that
  // is not, and is no sum of zeros because one of the rows is all zeros, is formed again, like one that is not finite.
#pragma unroll
  for (int i = 0; i < 8; ++i) {
#pragma unroll
    for (int step = 1; step < 8; step <<= 1) most[i] = fmaxf(most[i], __shfl_xor(most[i], step));
    if (lc == 0) largest[i >> 2][32 * wave + 8 * (i & 3) + lr] = most[i];
  }
  __syncthreads();
  const float lost = (float)K * 0x1p-98f;
  bool odd = false;
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const float of_x = largest[1][wn * 64 + n * 16 + r];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const f32x4 of_w = *reinterpret_cast<const f32x4*>(&largest[0][wm * 64 + m * 16 + 4 * g]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float y = fabsf(acc[m][n][i]);
        const bool small = y < lost * fmaxf(fmaxf(of_x, of_w[i]), 1.f) && of_x != 0.f && of_w[i] != 0.f;
        odd |= small || !(y <= 3.402823466e38f);
      }
    }
  }
  if (__any(odd)) {
    for (int n = 0; n < 4; ++n) {
      const int row = row0 + wn * 64 + n * 16 + r;
      const float* xr = X + (size_t)min(row, M - 1) * ld + first + 4 * g;
      for (int m = 0; m < (GATED ? 2 : 4); ++m) {
        f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
        const float* w0 = W + (size_t)w_row(wm * 64 + m * 16 + r) * ld + first + 4 * g;
        const float* w1 = W + (size_t)w_row(wm * 64 + (GATED ? m + 2 : m) * 16 + r) * ld + first + 4 * g;
        for (int k = 0; k < K; k += 16) {
          const f32x4 xv = *reinterpret_cast<const f32x4*>(xr + k), v0 = *reinterpret_cast<const f32x4*>(w0 + k);
          const f32x4 v1 = *reinterpret_cast<const f32x4*>(w1 + k);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(v0[i], xv[i], s0, 0, 0, 0);
            if (GATED) s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(v1[i], xv[i], s1, 0, 0, 0);
          }
        }
        store(m, row, GATED ? gated(s0, s1) : s0);
      }
    }
    return;
  }
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const int row = row0 + wn * 64 + n * 16 + r;
#pragma unroll
    for (int m = 0; m < (GATED ? 2 : 4); ++m) store(m, row, GATED ? gated(acc[m][n], acc[(m + 2) & 3][n]) : acc[m][n]);
  }
}

// y = the ranges' sums, added in the order of k
__global__ __launch_bounds__(256) void add_ranges_kernel(const f32x4* __restrict__ parts, f32x4* __restrict__ y, size_t n,
                                                         int ranges) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  f32x4 sum = parts[i];
  for (int j = 1; j < ranges; ++j) sum += parts[j * n + i];
  y[i] = sum;
}

// ------------------------------------------------------------------------------------------ up to eight rows
// Reading W once is the cost, and multiplications on the vector units are free beside it (M a number of W), so nothing
// has to be in an operand's order: a wavefront reads 1 KB of a row of W at a time, R rows together (gated: R gate
// and R up rows), and the same piece of the rows of X, which the caches hold.  The block's four wavefronts share k by chunks
// of 256, a thread adds up its own numbers in ascending order, and the threads' sums are added in a fixed order: the
// order depends on K only, not on the number of rows.
template <int M, int R, int ACT>
__global__ __launch_bounds__(256) void gemm_f32_rows_kernel(const float* __restrict__ X, const float* __restrict__ W,
                                                            float* __restrict__ Y, int Nout, int K) {
  constexpr bool GATED = ACT >= 0;
  constexpr int RT = GATED ? 2 * R : R, WAVES = 4, CHUNK = 256;
  __shared__ __attribute__((aligned(16))) float part[RT * M][WAVES * 64];
  __shared__ float sums[RT * M];
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int half = Nout >> 1, cols = GATED ? half : Nout;
  const int n0 = blockIdx.x * R;
  const float* w[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) w[i] = W + ((size_t)min(n0 + i % R, cols - 1) + (i / R) * half) * K + 4 * lane;
  const float* x = X + 4 * lane;
  float acc[RT][M];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int m = 0; m < M; ++m) acc[i][m] = 0.f;
  auto chunks = [&](auto count, int c, bool ok) {  // chunks c, c + 4, ..; ok: this lane's piece lies inside the rows
    constexpr int U = decltype(count)::value;
    f32x4 wv[U][RT], xv[U][M];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = ok ? (c + WAVES * u) * CHUNK : -4 * lane;
#pragma unroll
      for (int i = 0; i < RT; ++i) wv[u][i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(w[i] + k));
#pragma unroll
      for (int m = 0; m < M; ++m) xv[u][m] = *reinterpret_cast<const f32x4*>(x + (size_t)m * K + k);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int m = 0; m < M; ++m)
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[i][m] = ok ? __builtin_fmaf(wv[u][i][j], xv[u][m][j], acc[i][m]) : acc[i][m];
  };
  const int full = K / CHUNK;
  int c = wave;
  for (; c + WAVES < full; c += 2 * WAVES) chunks(std::integral_constant<int, 2>(), c, true);
  if (c < full) chunks(std::integral_constant<int, 1>(), c, true);
  if (K % CHUNK != 0 && wave == full % WAVES) chunks(std::integral_constant<int, 1>(), full, full * CHUNK + 4 * lane < K);
  // the threads' sums through shared memory, eight threads a value (a sum over the wavefront's lanes by exchanges took
  // six trips through shared memory a value: 50 us against 27 with 8 rows of 16384 x 2048)
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int m = 0; m < M; ++m) part[i * M + m][threadIdx.x] = acc[i][m];
  __syncthreads();
  for (int j = threadIdx.x >> 3; j < RT * M; j += 32) {
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < 8; ++q) s += *reinterpret_cast<const f32x4*>(&part[j][32 * q + 4 * (threadIdx.x & 7)]);
    float v = (s[0] + s[1]) + (s[2] + s[3]);
#pragma unroll
    for (int step = 1; step < 8; step <<= 1) v += __shfl_xor(v, step);
    if ((threadIdx.x & 7) == 0) sums[j] = v;
  }
  __syncthreads();
  const int i = threadIdx.x % R, m = threadIdx.x / R;
  if (m >= M || n0 + i >= cols) return;
  const float v = sums[i * M + m];
  Y[(size_t)m * cols + n0 + i] = GATED ? gate_act<GATED ? ACT : 0>(v) * sums[(GATED ? R + i : i) * M + m] : v;
}

template <int M, int ACT>
void launch_rows(const float* X, const float* W, float* Y, int Nout, int K, hipStream_t s) {
  constexpr int R = ACT >= 0 ? 2 : 4;
  const int cols = ACT >= 0 ? Nout / 2 : Nout;
  hipLaunchKernelGGL((gemm_f32_rows_kernel<M, R, ACT>), dim3((cols + R - 1) / R), dim3(256), 0, s, X, W, Y, Nout, K);
}

template <int M>
bool rows_of(int rows, const float* X, const float* W, float* Y, int act, int Nout, int K, hipStream_t s) {
  if (rows != M) {
    if constexpr (M < 8) return rows_of<M + 1>(rows, X, W, Y, act, Nout, K, s);
    return false;
  }
  if (act == 0) launch_rows<M, 0>(X, W, Y, Nout, K, s);
  else if (act == 1) launch_rows<M, 1>(X, W, Y, Nout, K, s);
  else launch_rows<M, -1>(X, W, Y, Nout, K, s);
  return true;
}

}  // namespace

// X [M, K], W [Nout, K], Y [M, Nout] (act >= 0: [M, Nout / 2]), float32, contiguous, 16-byte aligned; K a multiple of
// 32, the columns of Y one of 4.  act: -1 plain, 0 silu, 1 gelu (tanh form).  ranges > 1 (plain only): so many ranges
// of k are added up by blocks of their own into `parts` [ranges, M, Nout] and then together.
JLE_API int jle_gemm_f32_split(const float* X, const float* W, float* Y, float* parts, int act, int M, int Nout, int K,
                               int ranges, hipStream_t s) {
  if (M <= 0 || Nout <= 0) return 0;
  if (act < -1 || act > 1 || K <= 0 || K % kStage || Nout % (act >= 0 ? 8 : 4)) return JLE_BAD_ARG;
  if (ranges < 1 || ranges > K / kStage || (ranges > 1 && (act >= 0 || parts == nullptr))) return JLE_BAD_ARG;
  if ((((uintptr_t)X | (uintptr_t)W | (uintptr_t)Y | (uintptr_t)parts) & 15) != 0) return JLE_BAD_ARG;
  const int cols = act >= 0 ? Nout / 2 : Nout, tile = act >= 0 ? kTile / 2 : kTile;
  const int nb = (cols + tile - 1) / tile, mb = (M + kTile - 1) / kTile;
  const int per = (K / kStage + ranges - 1) / ranges * kStage;
  ranges = (K + per - 1) / per;  // (none is empty)
  if ((long long)nb * mb * ranges > (1ll << 24)) return JLE_BAD_ARG;
  const dim3 grid(nb * mb * ranges), block(256);
  float* out = ranges > 1 ? parts : Y;
#define GO(ACT_) \
  hipLaunchKernelGGL(gemm_f32_split_kernel<ACT_>, grid, block, 0, s, X, W, out, M, Nout, K, nb, mb, ranges, per)
  if (act == 0) GO(0);
  else if (act == 1) GO(1);
  else GO(-1);
#undef GO
  if (ranges > 1) {
    const size_t n = (size_t)M * Nout / 4;
    hipLaunchKernelGGL(add_ranges_kernel, dim3((unsigned)((n + 255) / 256)), block, 0, s, (const f32x4*)parts, (f32x4*)Y,
                       n, ranges);
  }
  JLE_LAUNCH_CHECK();
  return 0;
}

// The same product of up to eight rows: X, W 16-byte aligned, K a multiple of 4, an even Nout with act >= 0.
JLE_API int jle_gemm_f32_rows(const float* X, const float* W, float* Y, int act, int M, int Nout, int K, hipStream_t s) {
  if (M <= 0 || Nout <= 0) return 0;
  if (act < -1 || act > 1 || K <= 0 || K % 4 || (act >= 0 && Nout % 2)) return JLE_BAD_ARG;
  if ((((uintptr_t)X | (uintptr_t)W) & 15) != 0) return JLE_BAD_ARG;
  if (!rows_of<1>(M, X, W, Y, act, Nout, K, s)) return JLE_BAD_ARG;
  JLE_LAUNCH_CHECK();
  return 0;
}
