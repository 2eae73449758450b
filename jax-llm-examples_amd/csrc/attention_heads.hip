// Between an attention mixer's projected (and convolved) rows and the attention kernels, for mixers whose heads do
// not fit the fused preparation kernels: queries and keys of dk elements a head, values of dv, pages with heads of
// D >= max(dk, dv) elements (zeros behind the real ones), more key heads than value heads (a value head is written
// once for each of the `share` key heads that use it: two score maps over the same values), an RMS norm of q and k
// with or without weights before or behind the rotation, the rotation over adjacent or half-split pairs of the
// leading elements with a magnitude on sines and cosines.
//     rows [N, Hq dk + Hk dk + Hv dv] (or the leading part of wider rows)  ->  q_out [N, Hq, D],  pages [.., 2, Hk, ps, D] (values [D][ps])
// and the combination of two score maps' outputs into one head's:
//     d = a1 - lam a2;  d / sqrt(mean(d^2) + eps) * scale * sigmoid(gate)
// One wavefront per (token, head); a lane holds elements lane, lane + 64, ... (PER of them, so that a step of few tokens runs
// through no more code than its heads need).  Everything in float32; the order of every sum depends on the sizes only.
// Values lie transposed in their pages: a token's are single elements a row of the page apart, so many tokens' are brought
// sixteen at a time through shared memory and written in runs of a page's row.
// 16 query and 8 key heads of 128 on 8 value heads of 128, us: 2,048 tokens 31 -> 22.6 (34 MB: what is left is a wavefront's work
// for every head; with eight heads a wavefront, which share sines and cosines, the same), 300 6.9 -> 5.3, 255 7.0 -> 6.5, 8 3.6 ->
// 3.3; on 4 of 256, 2,048 36 -> 26.1; queries alone, 2,048 19 -> 11.5.
#include "common.h"

using namespace jle;

namespace {

constexpr int kMaxPerLane = 8;  // heads of up to 512 elements
constexpr int per_lane(int D) { return D <= 128 ? 2 : D <= 256 ? 4 : kMaxPerLane; }

template <typename T>
struct HeadsArgs {
  const T* rows;
  const int* positions;
  const int* slot_mapping;
  const float* inv_freq;  // [rotary_dim / 2] or null
  const float* wq;        // [dk], or [Hq][dk] (wq_stride = dk), or null
  const float* wk;
  T* q_out;
  T* kv_cache;  // or null
  float magnitude, norm_eps;  // norm_eps < 0: no norm
  int rotary_dim, half_pairs, norm_first, Hq, Hk, Hv, dk, dv, D, ps;
  int ld;         // from one row to the next (at least their width)
  int wq_stride;  // from one query head's norm weights to the next's (0: one for all)
};

// A block's sixteen tokens and 128 elements of a value head into their pages.
constexpr int kTileTokens = 16, kTileWidth = 128, kTilePitch = kTileWidth + 8;  // (256 threads: two rows at a time)
template <typename T>
__device__ __forceinline__ void write_values(const HeadsArgs<T>& a, T* tile, int N, int block) {
  const int columns = (a.D + kTileWidth - 1) / kTileWidth, d0 = block % columns * kTileWidth;
  const int vh = block / columns % a.Hv, t0 = block / columns / a.Hv * kTileTokens;
  const int share = a.Hk / a.Hv, j = threadIdx.x & 15;
  const size_t plane = (size_t)a.Hk * a.ps * a.D;
  const int slot = t0 + j < N ? a.slot_mapping[t0 + j] : -1;
  const T* src = a.rows + (size_t)t0 * a.ld + (a.Hq + a.Hk) * a.dk + vh * a.dv;
#pragma unroll
  for (int i = 0; i < kTileTokens * kTileWidth / 256; ++i) {  // (zeros behind the real elements)
    const int t = 2 * i + (threadIdx.x >> 7), e = threadIdx.x & (kTileWidth - 1);
    tile[t * kTilePitch + e] = t0 + t < N && d0 + e < a.dv ? src[(size_t)t * a.ld + d0 + e] : T(0);
  }
  __syncthreads();
  if (slot < 0) return;
  const int width = min(kTileWidth, a.D - d0);
  for (int s = 0; s < share; ++s) {
    T* dst = a.kv_cache + (size_t)(slot / a.ps) * 2 * plane + plane + ((size_t)(vh * share + s) * a.D + d0) * a.ps + slot % a.ps;
    for (int d = threadIdx.x >> 4; d < width; d += 16) dst[(size_t)d * a.ps] = tile[j * kTilePitch + d];
  }
}

// TILES: the first value_blocks blocks write the values sixteen tokens at a time, four wavefronts of the others a token's head each.
// Else a block is a wavefront of token blockIdx.x and head blockIdx.y, the values' heads behind the keys'.
template <typename T, int PER, bool TILES>
__global__ __launch_bounds__(TILES ? 256 : 64) void heads_prepare_kernel(HeadsArgs<T> a, int N, int value_blocks) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];  // a value tile, or PER * 64 floats a wavefront
  if (TILES && (int)blockIdx.x < value_blocks) {
    write_values(a, reinterpret_cast<T*>(smem), N, blockIdx.x);
    return;
  }
  const int lane = threadIdx.x & 63, wave = TILES ? wave_index() : 0;
  float* sh = reinterpret_cast<float*>(smem) + wave * PER * 64;
  int n = blockIdx.x, h = blockIdx.y;
  if (TILES) {
    const int heads = a.Hq + a.Hk, item = (int)(blockIdx.x - value_blocks) * 4 + wave;
    n = item / heads;
    h = item - n * heads;
    if (n >= N) return;
  }
  const bool is_q = h < a.Hq, is_v = h >= a.Hq + a.Hk;
  const int dim = is_v ? a.dv : a.dk;
  const int c0 = is_v ? (a.Hq + a.Hk) * a.dk + (h - a.Hq - a.Hk) * a.dv : h * a.dk;
  const T* src = a.rows + (size_t)n * a.ld + c0;
  float x[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = lane + 64 * i;
    x[i] = e < dim ? Num<T>::load(src + e) : 0.f;
  }
  if (!is_v) {
    const float* w = is_q ? (a.wq == nullptr ? nullptr : a.wq + (size_t)h * a.wq_stride) : a.wk;
    if (a.norm_eps >= 0.f && a.norm_first) {
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < PER; ++i) ss = __builtin_fmaf(x[i], x[i], ss);
      const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)dim + a.norm_eps);
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int e = lane + 64 * i;
        if (e < dim) x[i] = w != nullptr ? x[i] * inv * w[e] : x[i] * inv;
      }
    }
    if (a.inv_freq != nullptr && a.rotary_dim > 0) {
      const int rd = a.rotary_dim, hr = rd / 2;
      const float pos = (float)a.positions[n];
#pragma unroll
      for (int i = 0; i < PER; ++i) sh[lane + 64 * i] = x[i];
      asm volatile("" ::: "memory");  // (the wavefront's own place: its writes come before its reads)
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int e = lane + 64 * i;
        if (e < rd) {
          const bool first = a.half_pairs ? e < hr : (e & 1) == 0;
          const int j = a.half_pairs ? (first ? e : e - hr) : e >> 1;
          const int partner = a.half_pairs ? (first ? e + hr : e - hr) : e ^ 1;
          float sn, cs;
          sincosf(pos * a.inv_freq[j], &sn, &cs);
          sn *= a.magnitude;
          cs *= a.magnitude;
          const float other = sh[partner];
          x[i] = first ? x[i] * cs - other * sn : x[i] * cs + other * sn;
        }
      }
    }
    if (a.norm_eps >= 0.f && !a.norm_first) {
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < PER; ++i) ss = __builtin_fmaf(x[i], x[i], ss);
      const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)dim + a.norm_eps);
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int e = lane + 64 * i;
        if (e < dim) x[i] = w != nullptr ? x[i] * inv * w[e] : x[i] * inv;
      }
    }
  }
  if (is_q) {
    T* dst = a.q_out + ((size_t)n * a.Hq + h) * a.D;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = lane + 64 * i;
      if (e < a.D) Num<T>::store(dst + e, x[i]);  // (zeros behind the real elements)
    }
    return;
  }
  const int slot = a.slot_mapping[n];
  const size_t page = (size_t)(slot / a.ps);
  const int off = slot % a.ps;
  const size_t plane = (size_t)a.Hk * a.ps * a.D;
  if (!is_v) {
    T* dst = a.kv_cache + page * 2 * plane + ((size_t)(h - a.Hq) * a.ps + off) * a.D;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = lane + 64 * i;
      if (e < a.D) Num<T>::store(dst + e, x[i]);
    }
    return;
  }
  const int share = a.Hk / a.Hv, vh = h - a.Hq - a.Hk;
  for (int s = 0; s < share; ++s) {
    T* dst = a.kv_cache + page * 2 * plane + plane + (size_t)(vh * share + s) * a.ps * a.D + off;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = lane + 64 * i;
      if (e < a.D) Num<T>::store(dst + (size_t)e * a.ps, x[i]);
    }
  }
}

template <typename T>
__global__ __launch_bounds__(64) void diff_combine_kernel(const T* __restrict__ o, const T* __restrict__ gate,
                                                          T* __restrict__ out, float lam, float out_scale, float eps,
                                                          int H, int G, int D, int dv) {
  const int n = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int r = H / G, g = h / r, j = h - g * r;
  const T* a1 = o + ((size_t)n * 2 * H + (size_t)(g * 2 + 0) * r + j) * D;
  const T* a2 = o + ((size_t)n * 2 * H + (size_t)(g * 2 + 1) * r + j) * D;
  float d[kMaxPerLane];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < kMaxPerLane; ++i) {
    const int e = lane + 64 * i;
    d[i] = e < dv ? Num<T>::load(a1 + e) - lam * Num<T>::load(a2 + e) : 0.f;
    ss = __builtin_fmaf(d[i], d[i], ss);
  }
  const float inv = out_scale / sqrtf(wave_sum(ss) / (float)dv + eps);
#pragma unroll
  for (int i = 0; i < kMaxPerLane; ++i) {
    const int e = lane + 64 * i;
    if (e < dv) {
      float v = d[i] * inv;
      const size_t at = ((size_t)n * H + h) * dv + e;
      if (gate != nullptr) v *= 1.0f / (1.0f + expf(-Num<T>::load(gate + at)));
      Num<T>::store(out + at, v);
    }
  }
}

// How N tokens are prepared.  Values through shared memory from 256 tokens on (fewer are mostly single tokens of several requests,
// each in a page of its own).  A block has the shared memory of what it does and no more, and blocks of one wavefront are dealt
// out head by head: with room for four wavefronts and a tile in every block, token by token, us: 255 tokens of 16, 8 and 8 heads of 64
// in bfloat16 6.9, now 5.4; queries alone, float32, 16 heads of 256, 2,048 tokens 29.6, now 16.2.  Wide heads' values are
// written by a block for every 128 elements: 256 tokens of 2 value heads of 512 10.0, now 5.4.
struct HeadsPlan {
  bool tiles;
  int columns;  // parts of 128 elements of a value head
  uint32_t lds;
  int step;  // tokens a launch: its threads are fewer than 2^32
};
HeadsPlan heads_plan(int N, int heads, int D, bool paged, bool rotary, int size) {
  HeadsPlan p;
  p.tiles = paged && N >= 256;
  p.columns = (D + kTileWidth - 1) / kTileWidth;
  const uint32_t rows = rotary ? (p.tiles ? 4 : 1) * per_lane(D) * 256 : 0, tile = p.tiles ? kTileTokens * kTilePitch * size : 0;
  p.lds = rows > tile ? rows : tile;
  p.step = max(kTileTokens, (1 << 25) / heads / kTileTokens * kTileTokens);
  return p;
}

template <typename T, int PER>
int launch_heads(HeadsArgs<T> a, int N, hipStream_t s) {
  const HeadsPlan plan = heads_plan(N, a.Hq + a.Hk + a.Hv, a.D, a.kv_cache != nullptr, a.rotary_dim > 0, sizeof(T));
  for (int left = N; left > 0; left -= plan.step) {
    const int n = min(left, plan.step);
    if (plan.tiles) {
      const int value_blocks = (n + kTileTokens - 1) / kTileTokens * a.Hv * plan.columns;
      const int blocks = value_blocks + (n * (a.Hq + a.Hk) + 3) / 4;
      hipLaunchKernelGGL((heads_prepare_kernel<T, PER, true>), dim3((unsigned)blocks), dim3(256), plan.lds, s, a, n, value_blocks);
    } else {
      const int heads = a.kv_cache == nullptr ? a.Hq : a.Hq + a.Hk + a.Hv;
      hipLaunchKernelGGL((heads_prepare_kernel<T, PER, false>), dim3(n, heads), dim3(64), plan.lds, s, a, n, 0);
    }
    JLE_LAUNCH_CHECK();
    a.rows += (size_t)n * a.ld;
    a.q_out += (size_t)n * a.Hq * a.D;
    if (a.positions != nullptr) a.positions += n;
    if (a.slot_mapping != nullptr) a.slot_mapping += n;
  }
  return 0;
}

}  // namespace

// Bytes of shared memory of a block that prepares some of N tokens.
JLE_API int jle_heads_prepare_shared(int N, int D, int paged, int rotary, int is_bf16) {
  return (int)heads_plan(N, 1, D, paged != 0, rotary != 0, is_bf16 ? 2 : 4).lds;
}

JLE_API int jle_heads_prepare(const void* rows, int ld, const int* positions, const int* slot_mapping, const float* inv_freq,
                              int rotary_dim, int half_pairs, float magnitude, float norm_eps, int norm_first,
                              const float* wq, int wq_stride, const float* wk, void* q_out, void* kv_cache, int is_bf16, int N, int Hq,
                              int Hk, int Hv, int dk, int dv, int D, int ps, hipStream_t s) {
  if (N <= 0) return 0;
  if (rows == nullptr || q_out == nullptr || Hq <= 0 || Hk <= 0 || Hv <= 0 || Hk % Hv || dk <= 0 || dv <= 0 ||
      D < dk || D < dv || D > 64 * kMaxPerLane || Hq + Hk + Hv > 65535 || ps <= 0)
    return JLE_BAD_ARG;
  if (rotary_dim < 0 || rotary_dim % 2 || rotary_dim > dk || (rotary_dim > 0 && (inv_freq == nullptr || positions == nullptr)))
    return JLE_BAD_ARG;
  if (kv_cache != nullptr && slot_mapping == nullptr) return JLE_BAD_ARG;
  if (wq_stride != 0 && wq_stride != dk) return JLE_BAD_ARG;
  if (ld < (Hq + Hk) * dk + Hv * dv) return JLE_BAD_ARG;
  const HeadsArgs<bf16_t> a = {(const bf16_t*)rows, positions, slot_mapping, inv_freq, wq, wk, (bf16_t*)q_out, (bf16_t*)kv_cache, magnitude,
                               norm_eps, rotary_dim, half_pairs, norm_first, Hq, Hk, Hv, dk, dv, D, ps, ld, wq_stride};
  const HeadsArgs<float> f = {(const float*)rows, positions, slot_mapping, inv_freq, wq, wk, (float*)q_out, (float*)kv_cache, magnitude,
                              norm_eps, rotary_dim, half_pairs, norm_first, Hq, Hk, Hv, dk, dv, D, ps, ld, wq_stride};
  if (per_lane(D) == 2) return is_bf16 ? launch_heads<bf16_t, 2>(a, N, s) : launch_heads<float, 2>(f, N, s);
  if (per_lane(D) == 4) return is_bf16 ? launch_heads<bf16_t, 4>(a, N, s) : launch_heads<float, 4>(f, N, s);
  return is_bf16 ? launch_heads<bf16_t, kMaxPerLane>(a, N, s) : launch_heads<float, kMaxPerLane>(f, N, s);
}

// o [N, 2 H, D] in the order [kv head][map][query head of the group]; gate [N, H dv] or null; out [N, H dv].
JLE_API int jle_diff_combine(const void* o, const void* gate, void* out, float lam, float out_scale, float eps,
                             int is_bf16, int N, int H, int G, int D, int dv, hipStream_t s) {
  if (N <= 0) return 0;
  if (o == nullptr || out == nullptr || H <= 0 || G <= 0 || H % G || dv <= 0 || D < dv || dv > 64 * kMaxPerLane ||
      H > 65535)
    return JLE_BAD_ARG;
  if (is_bf16)
    hipLaunchKernelGGL(diff_combine_kernel<bf16_t>, dim3(N, H), dim3(64), 0, s, (const bf16_t*)o, (const bf16_t*)gate,
                       (bf16_t*)out, lam, out_scale, eps, H, G, D, dv);
  else
    hipLaunchKernelGGL(diff_combine_kernel<float>, dim3(N, H), dim3(64), 0, s, (const float*)o, (const float*)gate,
                       (float*)out, lam, out_scale, eps, H, G, D, dv);
  JLE_LAUNCH_CHECK();
  return 0;
}
