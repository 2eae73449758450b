// Dense matrix product of many rows: bfloat16 in and out, float32 accumulate on MFMA.
//
//   Y[t, n] = sum_k X[t, k] * W[n, k]  (+ bias[n])
//
// Tiles of 128 x 128 to 256 x 256, each a block's work (dense_block.h).
#include "dense_block.h"

using namespace jle;
using namespace jle::dense;

namespace {

struct DenseArgs {
  const bf16_t* X;
  const bf16_t* W;
  bf16_t* Y;
  const bf16_t* bias;
  int M, N, K;            // N: columns of Y
  int mt, nt, band;       // tiles of rows, of columns; rows of tiles that are gone through together
};

// The block's tile.  Blocks are dealt to the eight chiplets in turn; a chiplet takes a run of tiles, `band` rows of tiles high,
// so that those that it has at one time share rows of X and of W in its cache.
__device__ __forceinline__ void tile_of(const DenseArgs& p, int& tm, int& tn) {
  const int total = p.mt * p.nt, die = blockIdx.x & 7;
  const int t = die * (total >> 3) + min(die, total & 7) + (int)(blockIdx.x >> 3);
  const int g = t / (p.band * p.nt), in = t - g * p.band * p.nt;
  const int rows = min(p.band, p.mt - g * p.band);
  tm = g * p.band + in % rows;
  tn = in / rows;
}

template <int FM, int FN, int RX, int RW, int BLOCKS>
__global__ __launch_bounds__(256, BLOCKS) void dense_kernel(DenseArgs p) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  int tm, tn;
  tile_of(p, tm, tn);
  const int m0 = tm * FM * 32;
  const DenseBlock b = {p.X, p.W, p.Y, p.bias, nullptr, nullptr, 0, m0, p.M - m0, tn * FN * 32, p.N, p.K};
  dense_block<FM, FN, RX, RW, false, false>(b, smem);
}

template <int FM, int FN, int RX, int RW, int BLOCKS>
int launch(DenseArgs p, int units, hipStream_t s) {
  constexpr int BM = FM * 32, BN = FN * 32;
  constexpr uint32_t lds = dense_bytes<FM, FN, RX, RW, false>();
  static_assert(lds * BLOCKS <= 160 * 1024, "");
  const auto k = dense_kernel<FM, FN, RX, RW, BLOCKS>;
  if (const int rc = allow_lds(k, lds)) return rc;
  p.mt = (p.M + BM - 1) / BM;
  p.nt = (p.N + BN - 1) / BN;
  if ((long long)p.mt * p.nt > (1ll << 30)) return JLE_BAD_ARG;
  // rows of tiles that are gone through together: those with which the tiles that a chiplet has at one time need the fewest rows
  const int at_once = max(1, min((p.mt * p.nt + 7) / 8, units * BLOCKS / 8));
  int best = 0;
  for (int band = 1; band <= p.mt; band *= 2) {
    const int need = min(band, at_once) * FM + (at_once + band - 1) / band * FN;
    if (best == 0 || need < best) {
      best = need;
      p.band = band;
    }
  }
  hipLaunchKernelGGL(k, dim3((unsigned)(p.mt * p.nt)), dim3(256), lds, s, p);
  JLE_LAUNCH_CHECK();
  return 0;
}

}  // namespace

// X [M, K], W [N, K], Y [M, N], bias [N] or null: bfloat16, 16-byte aligned rows.  K a multiple of 64, N of 8; a tile's rows have
// fewer than 2^32 bytes.  tile: FM * 16 + FN; units: compute units.
JLE_API int jle_gemm_dense(const void* X, const void* W, void* Y, const void* bias, int M, int N, int K, int tile, int units, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (K < BK || K % BK || N % 8 || units < 8 || ((uintptr_t)X | (uintptr_t)W | (uintptr_t)Y) % 16 || (uintptr_t)bias % 8 ||
      (long long)K * 512 >= (1ll << 32))
    return JLE_BAD_ARG;
  const DenseArgs p = {(const bf16_t*)X, (const bf16_t*)W, (bf16_t*)Y, (const bf16_t*)bias, M, N, K, 0, 0, 1};
#define GO(FM, FN, RX, RW, BLOCKS) \
  case FM * 16 + FN: return launch<FM, FN, RX, RW, BLOCKS>(p, units, s)
  switch (tile) {
    GO(8, 8, 5, 5, 1);
    GO(8, 7, 5, 4, 1);
    GO(8, 6, 5, 6, 1);
    GO(6, 8, 6, 5, 1);
    GO(8, 5, 6, 6, 1);
    GO(8, 4, 6, 6, 1);
    GO(6, 4, 6, 6, 1);
    GO(4, 5, 6, 6, 1);
    GO(4, 4, 5, 5, 2);
  }
#undef GO
  return JLE_BAD_ARG;
}
