// Router: float32 logits, the k largest per token (lowest index first among equals),
// gate = sigmoid(logit); and the stable grouping of (token, choice) pairs by expert.
#include <limits.h>

#include "common.h"
#include "route.h"
#include "rows.h"

using namespace jle;

constexpr int kMaxTopK = 8;

// Router logits: logits[n, e] = sum_d h[n, d] * W[e, d], float32.  One wavefront per EPW experts and
// TPB tokens; a lane adds the terms of its float4 chunks (chunk = lane, lane + 64, ...) in
// order (each term one fused multiply-add, written out so that the compiler has no choice in it), then the
// lanes' sums are added by a butterfly: the order, and so the result, is the same for any TPB and EPW (a
// token's expert choice must not depend on what else is in the step).
template <int TPB, int EPW, bool VEC>
__global__ __launch_bounds__(256) void moe_logits_kernel(const float* __restrict__ h, const float* __restrict__ w,
                                                         float* __restrict__ logits, int N, int D, int E) {
  const int lane = threadIdx.x & 63;
  const int e0 = (blockIdx.y * 4 + wave_index()) * EPW;
  const int n0 = blockIdx.x * TPB;
  if (e0 >= E) return;
  const float* we[EPW];
#pragma unroll
  for (int j = 0; j < EPW; ++j) we[j] = w + (size_t)min(e0 + j, E - 1) * D;  // past the last: computed, not stored
  float acc[TPB][EPW];
#pragma unroll
  for (int t = 0; t < TPB; ++t)
#pragma unroll
    for (int j = 0; j < EPW; ++j) acc[t][j] = 0.f;
  if (VEC) {  // D is a multiple of 4: rows are 16-byte aligned
    const int D4 = D >> 2;
    // U chunks are loaded before any is used (a lone wavefront would otherwise wait for memory once per chunk);
    // chunks past the row's end are loaded from its last chunk and count as zeros
    constexpr int U = TPB * EPW == 1 ? 8 : TPB * EPW >= 64 ? 1 : 2;
    for (int c0 = lane; c0 < D4; c0 += 64 * U) {
      float4 wv[U][EPW], xv[U][TPB];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = min(c0 + 64 * u, D4 - 1);
#pragma unroll
        for (int j = 0; j < EPW; ++j) wv[u][j] = *reinterpret_cast<const float4*>(we[j] + 4 * c);
#pragma unroll
        for (int t = 0; t < TPB; ++t)
          xv[u][t] = *reinterpret_cast<const float4*>(h + (size_t)min(n0 + t, N - 1) * D + 4 * c);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (c0 + 64 * u < D4) {
#pragma unroll
          for (int t = 0; t < TPB; ++t)
#pragma unroll
            for (int j = 0; j < EPW; ++j) {
              acc[t][j] = __builtin_fmaf(xv[u][t].x, wv[u][j].x, acc[t][j]);
              acc[t][j] = __builtin_fmaf(xv[u][t].y, wv[u][j].y, acc[t][j]);
              acc[t][j] = __builtin_fmaf(xv[u][t].z, wv[u][j].z, acc[t][j]);
              acc[t][j] = __builtin_fmaf(xv[u][t].w, wv[u][j].w, acc[t][j]);
            }
        }
      }
    }
  } else {
    for (int d = lane; d < D; d += 64) {
#pragma unroll
      for (int t = 0; t < TPB; ++t)
        if (n0 + t < N) {
          const float xv = h[(size_t)(n0 + t) * D + d];
#pragma unroll
          for (int j = 0; j < EPW; ++j) acc[t][j] += xv * we[j][d];
        }
    }
  }
#pragma unroll
  for (int t = 0; t < TPB; ++t)
#pragma unroll
    for (int j = 0; j < EPW; ++j) {
      const float v = wave_sum(acc[t][j]);
      if (lane == 0 && n0 + t < N && e0 + j < E) logits[(size_t)(n0 + t) * E + e0 + j] = v;
    }
}

// The k largest logits of token n (lowest index first among equals) and their sigmoids.
// ACROSS: the logits were written by other blocks of this same launch (see put_shared).
template <bool ACROSS = false>
__device__ __forceinline__ void topk_of_token(const float* __restrict__ logits, size_t n, int E, int k,
                                              int (&best_i)[kMaxTopK], float (&gate)[kMaxTopK]) {
  float best_v[kMaxTopK];
#pragma unroll
  for (int j = 0; j < kMaxTopK; ++j) {
    best_v[j] = -INFINITY;
    best_i[j] = -1;
  }
  for (int e = 0; e < E; ++e) {
    float v = ACROSS ? get_shared(logits + n * E + e) : logits[n * E + e];
    // insert into the sorted list; strict '>' keeps the lower index ahead among equals,
    // and everything behind the insertion point moves down by one
    int ci = e;
    bool carrying = false;
#pragma unroll
    for (int j = 0; j < kMaxTopK; ++j) {
      if (j < k && (carrying || v > best_v[j] || best_i[j] < 0)) {
        const float tv = best_v[j];
        const int ti = best_i[j];
        best_v[j] = v;
        best_i[j] = ci;
        v = tv;
        ci = ti;
        carrying = true;
      }
    }
  }
#pragma unroll
  for (int j = 0; j < kMaxTopK; ++j) gate[j] = 1.0f / (1.0f + expf(-best_v[j]));
}

// The same choice made by a whole wavefront for one token, for 64 to 64 * kWaveTopKPerLane experts: every lane
// fetches its experts' logits at once (expert = lane, lane + 64, ...), then k times the lanes agree on the largest
// logit not yet taken (the lowest index among equals) with a butterfly of compares.  All lanes return the result.
constexpr int kWaveTopKPerLane = 4;
template <bool ACROSS = false>
__device__ __forceinline__ void topk_of_token_by_wave(const float* __restrict__ logits, size_t n, int E, int k,
                                                      int (&best_i)[kMaxTopK], float (&gate)[kMaxTopK]) {
  const int lane = threadIdx.x & 63;
  float v[kWaveTopKPerLane];
  bool open[kWaveTopKPerLane];  // an expert of this lane that is not taken yet
#pragma unroll
  for (int j = 0; j < kWaveTopKPerLane; ++j) {
    const int e = lane + 64 * j;
    open[j] = e < E;
    v[j] = 0.f;
    if (open[j]) v[j] = ACROSS ? get_shared(logits + n * E + e) : logits[n * E + e];
  }
#pragma unroll
  for (int r = 0; r < kMaxTopK; ++r) {
    best_i[r] = -1;
    gate[r] = 0.f;
    if (r < k) {
      float bv = 0.f;
      int be = INT_MAX;  // (none)
#pragma unroll
      for (int j = 0; j < kWaveTopKPerLane; ++j)
        if (open[j] && (be == INT_MAX || v[j] > bv)) {  // strict '>' keeps the lower index ahead among equals
          bv = v[j];
          be = lane + 64 * j;
        }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const float ov = __shfl_xor(bv, o, 64);
        const int oe = __shfl_xor(be, o, 64);
        if (oe != INT_MAX && (be == INT_MAX || ov > bv || (ov == bv && oe < be))) {
          bv = ov;
          be = oe;
        }
      }
      best_i[r] = be;
      gate[r] = 1.0f / (1.0f + expf(-bv));
#pragma unroll
      for (int j = 0; j < kWaveTopKPerLane; ++j)
        if (be == lane + 64 * j) open[j] = false;
    }
  }
}

__global__ void moe_topk_kernel(const float* __restrict__ logits, int* __restrict__ ids, float* __restrict__ gates,
                                int N, int E, int k) {
  const size_t n = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= (size_t)N) return;
  int best_i[kMaxTopK];
  float gate[kMaxTopK];
  topk_of_token(logits, n, E, k, best_i, gate);
#pragma unroll
  for (int j = 0; j < kMaxTopK; ++j) {
    if (j < k) {
      ids[n * k + j] = best_i[j];
      gates[n * k + j] = gate[j];
    }
  }
}

// The same grouping for any number of pairs that lie in memory.  Every wavefront has a run of the pairs: it counts them by
// expert; from all wavefronts' counts follows where each one's pairs of an expert begin; then it goes through its run once
// more, 64 pairs at a time, and a pair's row is its expert's next one plus how many of the lanes before it have the same expert,
// which a ballot for each bit of the experts' numbers tells.  Counting and placing are shared by all wavefronts whatever the
// number of experts.  (With a wavefront for every expert that looks through all pairs, 64 at a time and each look behind
// the last, us: 1,024 pairs of 8 experts 5.4 -> 4.4, 2,048 8.0 -> 5.4, 4,096 14.0 -> 7.2, 16,384 51 -> 20; 2,048 of 128 39 -> 6.0.)
// What is left is one block's trips to memory and shared memory, one behind the other.  The order of the rows is the pairs'.
constexpr int kAlignWaves = 16, kAlignAhead = 4;  // (pairs a lane asks for at once)
__global__ __launch_bounds__(kAlignWaves * 64) void moe_align_kernel(const int* __restrict__ ids, const float* __restrict__ gates,
                                                                     int* __restrict__ offsets, int* __restrict__ sorted_token,
                                                                     float* __restrict__ sorted_gate, int* __restrict__ inv,
                                                                     int M, int E, int k, int extra, int inv_ld) {
  extern __shared__ int smem[];  // counts[waves][E], starts[E + 1]
  const int lane = threadIdx.x & 63, wave = wave_index(), waves = blockDim.x >> 6;
  int* mine = smem + wave * E;
  int* starts = smem + waves * E;
  const int per = ((M + 63) / 64 + waves - 1) / waves * 64, lo = wave * per, hi = min(M, lo + per);
  int e[kAlignAhead];
  auto ask = [&](int base) __attribute__((always_inline)) {  // (E: no pair, or one without a row)
#pragma unroll
    for (int j = 0; j < kAlignAhead; ++j) {
      const int r = base + 64 * j + lane;
      e[j] = r < hi ? min(ids[r], E) : E;
    }
  };
  ask(lo);
  for (int i = threadIdx.x; i < waves * E; i += blockDim.x) smem[i] = 0;
  __syncthreads();
  for (int base = lo; base < hi; base += 64 * kAlignAhead) {
    if (base != lo) ask(base);
#pragma unroll
    for (int j = 0; j < kAlignAhead; ++j)
      if (e[j] < E) atomicAdd(&mine[e[j]], 1);
  }
  __syncthreads();
  for (int x = threadIdx.x; x < E; x += blockDim.x) {
    int c[kAlignWaves], run = 0;
#pragma unroll
    for (int w = 0; w < kAlignWaves; ++w) c[w] = w < waves ? smem[w * E + x] : 0;
#pragma unroll
    for (int w = 0; w < kAlignWaves; ++w) {
      if (w < waves) smem[w * E + x] = run;
      run += c[w];
    }
    starts[x] = run;
  }
  __syncthreads();
  if (wave == 0) {
    int before = 0;
    for (int x0 = 0; x0 < E; x0 += 64) {
      const int own = x0 + lane < E ? starts[x0 + lane] : 0;
      int upto = own;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(upto, o, 64);
        if (lane >= o) upto += v;
      }
      if (x0 + lane < E) starts[x0 + lane] = before + upto - own;
      before += __shfl(upto, 63, 64);
    }
    if (lane == 0) starts[E] = before;
  }
  __syncthreads();
  extra_group(starts[E], offsets, sorted_token, sorted_gate, inv, E, k, extra, inv_ld);
  for (int x = threadIdx.x; x <= E; x += blockDim.x) offsets[x] = starts[x];
  const int bits = 32 - __clz(E);
  for (int base = lo; base < hi; base += 64 * kAlignAhead) {
    float gate[kAlignAhead];
    if (hi - lo > 64 * kAlignAhead) ask(base);  // (else they are still here)
#pragma unroll
    for (int j = 0; j < kAlignAhead; ++j) gate[j] = e[j] < E ? gates[base + 64 * j + lane] : 0.f;
#pragma unroll
    for (int j = 0; j < kAlignAhead; ++j) {
      const int r = base + 64 * j + lane;
      if (base + 64 * j >= hi) break;
      unsigned long long same = ~0ull;
      for (int b = 0; b < bits; ++b) {
        const bool one = e[j] >> b & 1;
        const unsigned long long with = __ballot(one);
        same &= one ? with : ~with;
      }
      const int rank = __popcll(same & ((1ull << lane) - 1ull));
      int first = 0;
      if (rank == 0 && e[j] < E) first = starts[e[j]] + atomicAdd(&mine[e[j]], __popcll(same));
      first = __shfl(first, __ffsll((long long)same) - 1, 64);
      if (r >= hi) continue;
      const int pos = e[j] < E ? first + rank : -1, t = r / k;
      inv[t * inv_ld + r - t * k] = pos;
      if (pos >= 0) {
        sorted_token[pos] = t;
        sorted_gate[pos] = gate[j];
      }
    }
  }
}

// Both in one block, for steps of few tokens (N <= 1024): thread n chooses for token n and leaves its pairs in
// shared memory, from where the block groups them.
__global__ __launch_bounds__(1024) void moe_topk_align_kernel(const float* __restrict__ logits, int* __restrict__ ids,
                                                              float* __restrict__ gates, int* __restrict__ offsets,
                                                              int* __restrict__ sorted_token,
                                                              float* __restrict__ sorted_gate, int* __restrict__ inv,
                                                              int N, int E, int k, int extra) {
  extern __shared__ int smem[];  // counts[E], starts[E + 1], ids[N * k], gates[N * k]
  const int M = N * k;
  int* ids_s = smem + 2 * E + 1;
  float* gates_s = reinterpret_cast<float*>(ids_s + M);
  const int n = threadIdx.x;
  if (n < N) {
    int best_i[kMaxTopK];
    float gate[kMaxTopK];
    topk_of_token(logits, (size_t)n, E, k, best_i, gate);
#pragma unroll
    for (int j = 0; j < kMaxTopK; ++j) {
      if (j < k) {
        ids[n * k + j] = best_i[j];
        gates[n * k + j] = gate[j];
        ids_s[n * k + j] = best_i[j];
        gates_s[n * k + j] = gate[j];
      }
    }
  }
  __syncthreads();
  align_by_block(ids_s, gates_s, smem, smem + E, offsets, sorted_token, sorted_gate, inv, M, E, k, extra, k);
}

constexpr int kTokenExperts = 16;  // of the kernels whose block takes a token with all its experts

// The grouping of up to 64 R pairs by up to 63 experts by one wavefront: lane l has the experts and gates of the pairs l, l + 64,
// ...  What align_by_block writes, without its barriers and trips through shared memory.
template <int R>
__device__ __forceinline__ void align_by_wave(const int (&id)[R], const float (&gate)[R], int M, int E, int k, int extra,
                                              int inv_ld, int* __restrict__ offsets, int* __restrict__ sorted_token,
                                              float* __restrict__ sorted_gate, int* __restrict__ inv) {
  const int lane = threadIdx.x & 63;
  int pos[R], off = 0, run = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) pos[r] = -1;  // (an identity expert's pair has no row)
  for (int e = 0; e < E; ++e) {
    if (lane == e) off = run;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const bool match = id[r] == e && lane + 64 * r < M;
      const unsigned long long bal = __ballot(match);
      if (match) pos[r] = run + __popcll(bal & ((1ull << lane) - 1ull));
      run += __popcll(bal);
    }
  }
  if (lane < E) offsets[lane] = off;
  if (lane == 0) offsets[E] = run;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int pair = lane + 64 * r;
    if (pair >= M) continue;
    inv[pair / k * inv_ld + pair % k] = pos[r];
    if (pos[r] < 0) continue;
    sorted_token[pos[r]] = pair / k;
    sorted_gate[pos[r]] = gate[r];
  }
  if (extra > 0) {
    if (lane == 0) offsets[E + 1] = run + extra;
    for (int t = lane; t < extra; t += 64) {
      sorted_token[run + t] = t;
      sorted_gate[run + t] = 1.0f;
      if (inv_ld > k) inv[t * inv_ld + k] = run + t;
    }
  }
}

// The same as a launch of its own, for few pairs of few experts that lie in memory (see launch_align).
template <int R>
__global__ __launch_bounds__(64) void moe_align_wave_kernel(const int* __restrict__ ids, const float* __restrict__ gates,
                                                            int* __restrict__ offsets, int* __restrict__ sorted_token,
                                                            float* __restrict__ sorted_gate, int* __restrict__ inv, int M,
                                                            int E, int k, int extra, int inv_ld) {
  int id[R];
  float gate[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int pair = min((int)threadIdx.x + 64 * r, M - 1);
    id[r] = ids[pair];
    gate[r] = gates[pair];
  }
  align_by_wave(id, gate, M, E, k, extra, inv_ld, offsets, sorted_token, sorted_gate, inv);
}

// The router and the choice by scores of up to 16 experts, a block a token, a wavefront an expert (its sum in the order of
// moe_logits_kernel: the same bits).  Launches of their own, 4.6 and 4.8 us for 64 tokens, are mostly their start and end.  With
// the grouping behind it, before | so, us: 8 experts of 2,048, two a token: 17 tokens 9.0 | 7.0, 64 9.2 | 7.3, 256 10.9 | 9.2; 10 of
// 4,096: 64 10.4 | 8.7, 256 12.7 | 10.9.
template <int WAVES>
__global__ __launch_bounds__(WAVES * 64) void moe_logits_choose_kernel(const float* __restrict__ h,
                                                                       const float* __restrict__ router, int* __restrict__ ids,
                                                                       float* __restrict__ weights, int D, Choice choice) {
  constexpr int U = 8;  // pieces of a row a lane asks for at once
  __shared__ float z[kTokenExperts], scores[kTokenExperts], choices[kTokenExperts];
  const size_t n = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int D4 = D >> 2;
  if (wave < choice.E) {
    const float4* x = reinterpret_cast<const float4*>(h + n * D);
    const float4* w = reinterpret_cast<const float4*>(router + (size_t)wave * D);
    float acc = 0.f;
    for (int c0 = lane; c0 - lane < D4; c0 += 64 * U) {
      float4 xv[U], wv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = min(c0 + 64 * u, D4 - 1);
        xv[u] = x[c];
        wv[u] = w[c];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (c0 + 64 * u >= D4) continue;
        acc = __builtin_fmaf(xv[u].x, wv[u].x, acc);
        acc = __builtin_fmaf(xv[u].y, wv[u].y, acc);
        acc = __builtin_fmaf(xv[u].z, wv[u].z, acc);
        acc = __builtin_fmaf(xv[u].w, wv[u].w, acc);
      }
    }
    acc = wave_sum(acc);
    if (lane == 0) z[wave] = acc;
  }
  __syncthreads();
  if (wave != 0) return;
  int id;
  float weight;
  choose_by_wave<false>(z, choice, scores, choices, id, weight);
  if (lane < choice.top_k) {
    ids[n * choice.top_k + lane] = id;
    weights[n * choice.top_k + lane] = weight;
  }
}

// The residual row n and what is added to it, normed: into shared memory (all threads of the block), and by the writer stored.
template <typename DT, typename OT, int CPT>
__device__ __forceinline__ void normed_row(const float* __restrict__ x, const Delta<DT>& delta, const float* __restrict__ w,
                                           float eps, float* __restrict__ x_out, OT* __restrict__ h_out, size_t n, int D,
                                           bool writer, float* row, float* red) {
  constexpr int THREADS = 256;
  f32x4_t wv[CPT];
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int d = (threadIdx.x + THREADS * i) * 4;
    wv[i] = (w != nullptr && d < D) ? load4<float>(w + d) : f32x4_t{1.f, 1.f, 1.f, 1.f};
  }
  f32x4_t v[CPT];
  float ss = 0.f;
  const bool add = delta.any();
  const DeltaRow<DT> drow = delta_row(delta, n, D);
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int d = (threadIdx.x + THREADS * i) * 4;
    v[i] = d < D ? load4<float>(x + d) : f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  // (every load before the first store: see add_rmsnorm_vec_kernel)
  if (add) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int d = (threadIdx.x + THREADS * i) * 4;
      v[i] += d < D ? delta_row_at4<false, DT>(delta, drow, n, d, D) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
  }
  if (writer) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int d = (threadIdx.x + THREADS * i) * 4;
      if (d < D) store4<float>(x_out + d, v[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < CPT; ++i) ss = add_squares4(ss, v[i]);
  const float tot = block_sum<THREADS>(ss, red);
  const float rs = 1.0f / sqrtf(tot / (float)D + eps);
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int d = (threadIdx.x + THREADS * i) * 4;
    if (d < D) {
      f32x4_t h = v[i] * rs;
      if (w != nullptr) h *= wv[i];
      *reinterpret_cast<f32x4_t*>(row + d) = h;
      if (writer && h_out != nullptr) store4<OT>(h_out + d, h);
    }
  }
}

// Steps of few tokens: the addition of the pending branch output to the residual, the norm of the sum, the
// router's logits, the choice of experts and the grouping of the choices, in one launch.  A block is (token,
// four experts): it forms the token's normed row (every block of a token the same row, with the arithmetic of
// add_rmsnorm_vec_kernel: the same bits), keeps it in shared memory, and each of its wavefronts adds up one
// expert's logit (the arithmetic of moe_logits_kernel<1, 1, true>).  The block of a token's first four experts
// also writes the new residual and the normed row.  The block that finishes last (a ticket counter, zero between
// launches) chooses and groups for all tokens.  N <= 256, D a multiple of 8 in (1024, 8192], CPT: pieces of four a thread
// (as many as the width needs: 16 tokens of 2,048 19.4 us with the eight of the widest row, 17.9 with two).
// SCORED: the choice is made by scores (see Choice, route.h); `experts` of the router's E rows have matrices and are
// grouped, a token's row in the extra group is noted behind its choices' (inv_ld = k + 1 then).
template <typename DT, typename OT, bool SCORED, int CPT>
__global__ __launch_bounds__(256) void norm_route_kernel(const float* __restrict__ x, Delta<DT> delta,
                                                         const float* __restrict__ w, float eps,
                                                         float* __restrict__ x_out, OT* __restrict__ h_out,
                                                         const float* __restrict__ router,
                                                         float* __restrict__ logits, int* __restrict__ ids,
                                                         float* __restrict__ gates, int* __restrict__ offsets,
                                                         int* __restrict__ sorted_token,
                                                         float* __restrict__ sorted_gate, int* __restrict__ inv,
                                                         int* __restrict__ ticket, int N, int D, int E, int k,
                                                         int extra, Choice choice, int experts) {
  constexpr int THREADS = 256;
  extern __shared__ int smem[];  // the normed row [D] (floats); afterwards the grouping's counters and pairs
  float* row = reinterpret_cast<float*>(smem);
  __shared__ float red[THREADS / 64];
  __shared__ int last_flag;
  const size_t n = blockIdx.x;
  const size_t base = n * D;
  const bool writer = blockIdx.y == 0;
  normed_row<DT, OT, CPT>(x + base, delta, w, eps, x_out + base, h_out != nullptr ? h_out + base : nullptr, n, D, writer, row, red);
  __syncthreads();
  // one expert's logit per wavefront
  const int lane = threadIdx.x & 63;
  const int e = blockIdx.y * 4 + wave_index();
  if (e < E) {
    const float* we = router + (size_t)e * D;
    const int D4 = D >> 2;
    constexpr int U = 8;
    float acc = 0.f;
    for (int c0 = lane; c0 < D4; c0 += 64 * U) {
      float4 rv[U], xv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = min(c0 + 64 * u, D4 - 1);
        rv[u] = *reinterpret_cast<const float4*>(we + 4 * c);
        xv[u] = *reinterpret_cast<const float4*>(row + 4 * c);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (c0 + 64 * u < D4) {
          acc = __builtin_fmaf(xv[u].x, rv[u].x, acc);
          acc = __builtin_fmaf(xv[u].y, rv[u].y, acc);
          acc = __builtin_fmaf(xv[u].z, rv[u].z, acc);
          acc = __builtin_fmaf(xv[u].w, rv[u].w, acc);
        }
      }
    }
    const float val = wave_sum(acc);
    if (lane == 0) put_shared(logits + n * E + e, val);
  }
  // the last block to get here chooses and groups.  The logits were written through to where every compute unit
  // reads them (put_shared: a store acknowledged only when it has got there); every wavefront waits for the
  // acknowledgement of its outstanding stores (vmcnt(0): neither the workgroup-scope fence nor the barrier
  // does), the barrier for all the block's wavefronts, and only then the block takes its ticket (an atomic at
  // agent scope).  The block with the last ticket reads the logits past its own die's caches (get_shared),
  // after the ticket's value has come back.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __syncthreads();
  if (threadIdx.x == 0) {
    const int total = (int)(gridDim.x * gridDim.y);
    const int t = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last_flag = t == total - 1;
    if (last_flag) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!last_flag) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  int* ismem = smem;  // counts[E], starts[E + 1], ids[N * k], gates[N * k]
  const int M = N * k;
  int* ids_s = ismem + 2 * E + 1;
  float* gates_s = reinterpret_cast<float*>(ids_s + M);
  if (SCORED) {
    float* scores = gates_s + M + (size_t)wave_index() * 2 * E;
    for (int t = wave_index(); t < N; t += THREADS / 64) {
      int id;
      float weight;
      choose_by_wave<true>(logits + (size_t)t * E, choice, scores, scores + E, id, weight);
      if (lane < k) {
        ids[t * k + lane] = id;
        gates[t * k + lane] = weight;
        ids_s[t * k + lane] = id;
        gates_s[t * k + lane] = weight;
      }
    }
    __syncthreads();
    align_by_block(ids_s, gates_s, ismem, ismem + E, offsets, sorted_token, sorted_gate, inv, M, experts, k, extra,
                   extra > 0 ? k + 1 : k);
    return;
  }
  if (E >= 64 && E <= 64 * kWaveTopKPerLane) {
    // many experts: a wavefront per token, the token's logits fetched in one trip
    for (int t = wave_index(); t < N; t += THREADS / 64) {
      int best_i[kMaxTopK];
      float gate[kMaxTopK];
      topk_of_token_by_wave<true>(logits, (size_t)t, E, k, best_i, gate);
      if (lane == 0) {
#pragma unroll
        for (int j = 0; j < kMaxTopK; ++j) {
          if (j < k) {
            ids[t * k + j] = best_i[j];
            gates[t * k + j] = gate[j];
            ids_s[t * k + j] = best_i[j];
            gates_s[t * k + j] = gate[j];
          }
        }
      }
    }
  } else {
    const int t = threadIdx.x;
    if (t < N) {
      int best_i[kMaxTopK];
      float gate[kMaxTopK];
      topk_of_token<true>(logits, (size_t)t, E, k, best_i, gate);
#pragma unroll
      for (int j = 0; j < kMaxTopK; ++j) {
        if (j < k) {
          ids[t * k + j] = best_i[j];
          gates[t * k + j] = gate[j];
          ids_s[t * k + j] = best_i[j];
          gates_s[t * k + j] = gate[j];
        }
      }
    }
  }
  __syncthreads();
  align_by_block(ids_s, gates_s, ismem, ismem + E, offsets, sorted_token, sorted_gate, inv, M, E, k, extra, k);
}

// norm_route_kernel for choices by scores of up to 16 experts, up to 64 pairs of more than a few tokens: a block takes a token
// with all its experts, EPW a wavefront, chooses from its own shared memory, and only the choices are handed to the block that
// groups.  Where norm_route_kernel's time goes (16 tokens of 2,048, 10 experts, two by scores): row and addition 2.6 us, sum of
// squares and row 0.9, logits 1.4, handed over 0.8, choice 10.3 (the last block alone, four tokens a wavefront one after the
// other), grouping 1.8.  Here all tokens are chosen for at once, the router's first rows come while the token's row is added and
// normed, and one wavefront groups in registers.  norm_route_kernel | this, us, 10 experts: 16 tokens of 2,048 19.0 | 13.5, 32
// 30.0 | 15.0; 16 of 4,096 21.6 | 16.3; 8 of 3,072, 16 experts 17.2 | 14.4; 16 of 6,144, 8 experts 22.8 | 16.8; but a lone token,
// whose experts are shared out over compute units there, 9.7 | 10.3, and 4 of 4,096, 16 experts 13.5 | 13.8; nor up to 8 whose rows
// with more than 8 experts are long: 5 of 8,192, 10 experts 16.1 | 17.5, 8 16.7 | 17.6, 16 19.6 | 17.6.
template <typename DT, typename OT, int CPT, int EPW>
__global__ __launch_bounds__(256) void norm_route_token_kernel(const float* __restrict__ x, Delta<DT> delta,
                                                               const float* __restrict__ w, float eps,
                                                               float* __restrict__ x_out, OT* __restrict__ h_out,
                                                               const float* __restrict__ router,
                                                               float* __restrict__ logits, int* __restrict__ ids,
                                                               float* __restrict__ gates, int* __restrict__ offsets,
                                                               int* __restrict__ sorted_token,
                                                               float* __restrict__ sorted_gate, int* __restrict__ inv,
                                                               int* __restrict__ ticket, int N, int D, int E, int k,
                                                               int extra, Choice choice, int experts) {
  constexpr int U = 4;  // pieces of a router row a lane asks for at once
  extern __shared__ int smem[];  // the normed row [D] (floats)
  float* row = reinterpret_cast<float*>(smem);
  __shared__ float red[4];
  __shared__ float z[kTokenExperts], scores[kTokenExperts], choices[kTokenExperts];
  const size_t n = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int D4 = D >> 2;
  const float4* we[EPW];
#pragma unroll
  for (int j = 0; j < EPW; ++j) we[j] = reinterpret_cast<const float4*>(router + (size_t)min(wave + 4 * j, E - 1) * D);
  float4 rv[U][EPW];
  auto ask = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < EPW; ++j) rv[u][j] = we[j][min(c0 + 64 * u, D4 - 1)];
  };
  ask(lane);
  normed_row<DT, OT, CPT>(x + n * D, delta, w, eps, x_out + n * D, h_out != nullptr ? h_out + n * D : nullptr, n, D, true, row, red);
  __syncthreads();
  float acc[EPW];
#pragma unroll
  for (int j = 0; j < EPW; ++j) acc[j] = 0.f;
  for (int c0 = lane; c0 - lane < D4; c0 += 64 * U) {  // (a lane's terms in the order of moe_logits_kernel)
    float4 cur[U][EPW];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < EPW; ++j) cur[u][j] = rv[u][j];
    if (c0 - lane + 64 * U < D4) ask(c0 + 64 * U);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = c0 + 64 * u;
      if (c >= D4) continue;
      const float4 h = *reinterpret_cast<const float4*>(row + 4 * c);
#pragma unroll
      for (int j = 0; j < EPW; ++j) {
        acc[j] = __builtin_fmaf(h.x, cur[u][j].x, acc[j]);
        acc[j] = __builtin_fmaf(h.y, cur[u][j].y, acc[j]);
        acc[j] = __builtin_fmaf(h.z, cur[u][j].z, acc[j]);
        acc[j] = __builtin_fmaf(h.w, cur[u][j].w, acc[j]);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < EPW; ++j) {
    const int e = wave + 4 * j;
    const float v = wave_sum(acc[j]);
    if (lane == 0 && e < E) {
      z[e] = v;
      logits[n * E + e] = v;
    }
  }
  __syncthreads();
  if (wave != 0) return;
  int id[1];  // lane r < k: the token's r-th choice
  float gate[1];
  choose_by_wave<false>(z, choice, scores, choices, id[0], gate[0]);
  const int M = N * k;
  // handed over as norm_route_kernel hands over its logits
  if (lane < k) {
    __hip_atomic_store(ids + n * k + lane, id[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    put_shared(gates + n * k + lane, gate[0]);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  int t = 0;
  if (lane == 0) t = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (__builtin_amdgcn_readfirstlane(t) != N - 1) return;
  if (lane == 0) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (lane < M) {
    id[0] = __hip_atomic_load(ids + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    gate[0] = get_shared(gates + lane);
  }
  align_by_wave(id, gate, M, experts, k, extra, extra > 0 ? k + 1 : k, offsets, sorted_token, sorted_gate, inv);
}

static int launch_logits(const float* h, const float* w, float* logits, int N, int D, int E, hipStream_t s) {
  const bool vec = D % 4 == 0 && (((uintptr_t)h | (uintptr_t)w) & 15) == 0;
  // few rows: a wavefront per (token, expert) keeps more of them in flight; many: a wavefront takes several
  // tokens and experts, so that the rows of h and w are read that much less often (measured with 128 experts:
  // 400 rows 118 -> 73 us, 128 rows 60 -> 48)
  const bool many = (long long)N * E >= 8192;  // (512 rows x 16 experts; with 128 experts from 64 rows on)
  dim3 b(256);
  const auto blocks = [&](int tokens, int experts) {
    return (long long)((N + tokens - 1) / tokens) * ((E + 4 * experts - 1) / (4 * experts));
  };
#define LOGITS(T_, E_)                                                                                    \
  hipLaunchKernelGGL((moe_logits_kernel<T_, E_, true>), dim3((N + T_ - 1) / T_, (E + 4 * E_ - 1) / (4 * E_)), b, 0, s, \
                     h, w, logits, N, D, E)
  // many rows: the larger the piece of a wavefront (tokens x experts), the fewer loads per multiply-add (the
  // first-level cache's bandwidth is the limit), as long as the pieces still fill the compute units several
  // times over.  Measured at 5,120 wide: 2,048 rows x 128 experts 212 -> 134 us, 8,192 x 16 141 -> 96.
  if (many && vec && E >= 32 && blocks(8, 8) >= 1024) {
    LOGITS(8, 8);
  } else if (many && vec && blocks(8, 4) >= 1024) {
    LOGITS(8, 4);
  } else if (many && vec && blocks(4, 4) >= 512) {
    LOGITS(4, 4);
  } else if (many) {
    dim3 g((N + 1) / 2, (E + 15) / 16);
    if (vec) hipLaunchKernelGGL((moe_logits_kernel<2, 4, true>), g, b, 0, s, h, w, logits, N, D, E);
    else hipLaunchKernelGGL((moe_logits_kernel<2, 4, false>), g, b, 0, s, h, w, logits, N, D, E);
  } else {
    dim3 g(N, (E + 3) / 4);
    if (vec) hipLaunchKernelGGL((moe_logits_kernel<1, 1, true>), g, b, 0, s, h, w, logits, N, D, E);
    else hipLaunchKernelGGL((moe_logits_kernel<1, 1, false>), g, b, 0, s, h, w, logits, N, D, E);
  }
#undef LOGITS
  JLE_LAUNCH_CHECK();
  return 0;
}

static int launch_align(const int* ids, const float* gates, int* offsets, int* sorted_token, float* sorted_gate,
                        int* inv, int M, int E, int k, int extra, int inv_ld, hipStream_t s) {
  // A wavefront looks at all its pairs for every expert; moe_align_kernel's meet at four barriers, 3.6 to 3.7 us up to 256 pairs
  // whatever the experts.  One wavefront, us: 64 pairs of 8 experts 2.3, of 32 3.6, of 48 5.4; 128 of 8 2.6, of 16 3.2; 256 of 8
  // 3.1, of 16 4.1, of 32 6.1.  Above 256 pairs, one | all: 320 of 2 experts 2.7 | 3.7, of 4 3.0 | 3.7, of 6 3.4 | 3.7, of 8 3.7 | 3.7.
  if (M <= (E <= 6 ? 384 : 256) && (M + 63) / 64 * E <= 40) {
#define WAVE(R_) \
  hipLaunchKernelGGL(moe_align_wave_kernel<R_>, dim3(1), dim3(64), 0, s, ids, gates, offsets, sorted_token, sorted_gate, inv, M, E, \
                     k, extra, inv_ld)
    if (M <= 64) WAVE(1);
    else if (M <= 128) WAVE(2);
    else if (M <= 256) WAVE(4);
    else WAVE(6);
#undef WAVE
    JLE_LAUNCH_CHECK();
    return 0;
  }
  // (64 KB of counts: fewer wavefronts with thousands of experts)
  const int waves = min(min(kAlignWaves, (M + 63) / 64), (16384 - (E + 1)) / E);
  if (waves < 1) return JLE_BAD_ARG;
  hipLaunchKernelGGL(moe_align_kernel, dim3(1), dim3(64 * waves), ((waves + 1) * E + 1) * sizeof(int), s, ids, gates, offsets,
                     sorted_token, sorted_gate, inv, M, E, k, extra, inv_ld);
  JLE_LAUNCH_CHECK();
  return 0;
}

// logits: [N, E] float32 workspace (also the caller's copy of the router logits)
JLE_API int jle_moe_route(const float* h, const float* w, int* ids, float* gates, float* logits, int N, int D, int E,
                          int k, hipStream_t s) {
  if (N <= 0) return 0;
  if (k < 1 || k > kMaxTopK || k > E || E > 4096 || logits == nullptr) return JLE_BAD_ARG;
  if (int rc = launch_logits(h, w, logits, N, D, E, s)) return rc;
  hipLaunchKernelGGL(moe_topk_kernel, dim3((N + 127) / 128), dim3(128), 0, s, logits, ids, gates, N, E, k);
  JLE_LAUNCH_CHECK();
  return 0;
}

// The logits alone (for a choice that another kernel makes).
JLE_API int jle_moe_logits(const float* h, const float* w, float* logits, int N, int D, int E, hipStream_t s) {
  if (N <= 0) return 0;
  if (E < 1 || E > 4096 || logits == nullptr) return JLE_BAD_ARG;
  return launch_logits(h, w, logits, N, D, E, s);
}

// The router of up to 16 experts and the choice by scores (the same results as jle_moe_logits, then jle_moe_choose).
JLE_API int jle_moe_logits_choose(const float* h, const float* w, const float* correction, int* ids, float* weights, int N, int D,
                                  int E, int top_k, int groups, int keep, int terms, int softmax, float floor_, float scale,
                                  hipStream_t s) {
  if (N <= 0) return 0;
  const Choice a = {correction, E, top_k, groups, keep, terms, softmax, floor_, scale};
  if (!choice_ok(a) || E > kTokenExperts || D <= 0 || D % 4 || (((uintptr_t)h | (uintptr_t)w) & 15) != 0) return JLE_BAD_ARG;
  if (E <= 4) hipLaunchKernelGGL(moe_logits_choose_kernel<4>, dim3(N), dim3(256), 0, s, h, w, ids, weights, D, a);
  else if (E <= 8) hipLaunchKernelGGL(moe_logits_choose_kernel<8>, dim3(N), dim3(512), 0, s, h, w, ids, weights, D, a);
  else hipLaunchKernelGGL(moe_logits_choose_kernel<16>, dim3(N), dim3(1024), 0, s, h, w, ids, weights, D, a);
  JLE_LAUNCH_CHECK();
  return 0;
}

// The router and the grouping of its choices in one call (the same results as jle_moe_route, then jle_moe_align).
// extra_group: offsets has E + 2 entries, sorted_token and sorted_gate N * k + N (see align_by_block).
JLE_API int jle_moe_route_align(const float* h, const float* w, int* ids, float* gates, float* logits, int* offsets,
                                int* sorted_token, float* sorted_gate, int* inv, int N, int D, int E, int k,
                                int extra_group, hipStream_t s) {
  if (N <= 0) return 0;
  if (k < 1 || k > kMaxTopK || k > E || E > 4096 || logits == nullptr) return JLE_BAD_ARG;
  if (int rc = launch_logits(h, w, logits, N, D, E, s)) return rc;
  const size_t words = (size_t)2 * E + 1 + (size_t)2 * N * k;
  if (N <= 1024 && words <= 12000) {
    hipLaunchKernelGGL(moe_topk_align_kernel, dim3(1), dim3(1024), words * sizeof(int), s, logits, ids, gates,
                       offsets, sorted_token, sorted_gate, inv, N, E, k, extra_group ? N : 0);
    JLE_LAUNCH_CHECK();
    return 0;
  }
  hipLaunchKernelGGL(moe_topk_kernel, dim3((N + 127) / 128), dim3(128), 0, s, logits, ids, gates, N, E, k);
  JLE_LAUNCH_CHECK();
  return launch_align(ids, gates, offsets, sorted_token, sorted_gate, inv, N * k, E, k, extra_group ? N : 0, k, s);
}

// inv_ld: k, or k + 1 to note a token's row in the extra group behind its choices' rows; choices of E and beyond get
// no row (see route.h).
JLE_API int jle_moe_align(const int* ids, const float* gates, int* offsets, int* sorted_token, float* sorted_gate,
                          int* inv, int M, int E, int k, int extra_group, int inv_ld, hipStream_t s) {
  if (M <= 0) return 0;
  if (E < 1 || E > 4096 || k < 1 || M % k || inv_ld < k || inv_ld > k + 1) return JLE_BAD_ARG;
  return launch_align(ids, gates, offsets, sorted_token, sorted_gate, inv, M, E, k, extra_group ? M / k : 0, inv_ld, s);
}

// add + norm + router + choice + grouping in one launch, for steps of at most 256 tokens (see norm_route_kernel).
// delta_kind: 0 none, 1 plain (delta), 2 expert sum (routed, inv_in, k_in, shared, self, self_w, self_k), as for
// jle_add_rmsnorm.  experts > 0: the choice is made by scores (correction .. scale: see Choice, route.h), E counts the
// router's rows, the first `experts` of them have matrices; with the extra group inv has k + 1 entries a token.
// x_out: the residual after the addition (another array than x: the blocks of a token read x while one writes).
// ticket: one counter, zero before the first launch and after every launch.
// Returns JLE_BAD_ARG for sizes the fused kernel does not take (the caller then uses the separate kernels).
JLE_API int jle_norm_route(const float* x, int delta_kind, const void* delta, const void* routed, const int* inv_in,
                           int k_in, const void* shared, int delta_is_bf16, const float* w, float eps, float* x_out,
                           void* h_out, int out_is_bf16, const float* router, float* logits, int* ids, float* gates,
                           int* offsets, int* sorted_token, float* sorted_gate, int* inv, int* ticket, int N, int D,
                           int E, int k, int extra_group, const void* self, const float* self_w, int self_k,
                           int experts, const float* correction, int groups, int keep, int terms, int softmax,
                           float floor_, float scale, hipStream_t s) {
  if (N <= 0) return 0;
  const bool scored = experts > 0;
  const Choice choice = {correction, E, k, groups, keep, terms, softmax, floor_, scale};
  if (N > 256 || D % 8 || D <= 1024 || D > 8192 || k < 1 || k > E || E > 4096) return JLE_BAD_ARG;
  if (scored ? (!choice_ok(choice) || experts > E) : k > kMaxTopK) return JLE_BAD_ARG;
  const uintptr_t all = (uintptr_t)x | (uintptr_t)delta | (uintptr_t)routed | (uintptr_t)shared | (uintptr_t)w | (uintptr_t)self |
                        (uintptr_t)x_out | (uintptr_t)h_out | (uintptr_t)router;
  if ((all & 15) != 0 || ticket == nullptr || logits == nullptr || x_out == x) return JLE_BAD_ARG;
  const size_t words = (size_t)2 * E + 1 + (size_t)2 * N * k + (scored ? (size_t)8 * E : 0);
  const size_t lds = (words > (size_t)D ? words : (size_t)D) * sizeof(float);
  if (lds > 48 * 1024) return JLE_BAD_ARG;
  dim3 g(N, (E + 3) / 4), b(256);
#define LAUNCH(DT, OT, SCORED, CPT)                                                                              \
  hipLaunchKernelGGL((norm_route_kernel<DT, OT, SCORED, CPT>), g, b, lds, s, x, dl, w, eps, x_out, (OT*)h_out,   \
                     router, logits, ids, gates, offsets, sorted_token, sorted_gate, inv, ticket, N, D, E, k,    \
                     extra_group ? N : 0, choice, experts)
  // (the same bits: which of the two is a question of time alone)
  const bool by_token = scored && E <= kTokenExperts && N > (E > 8 && D > 4096 ? 8 : 4) && N * k <= 64;
#define LAUNCH_T(DT, OT, CPT, EPW)                                                                               \
  hipLaunchKernelGGL((norm_route_token_kernel<DT, OT, CPT, EPW>), dim3(N), b, D * sizeof(float), s, x, dl, w, eps, x_out, \
                     (OT*)h_out, router, logits, ids, gates, offsets, sorted_token, sorted_gate, inv, ticket, N, D, E, k, \
                     extra_group ? N : 0, choice, experts)
#define TOKEN_BY_WIDTH(DT, OT, EPW)                                                                              \
  do {                                                                                                           \
    if (D <= 2048) LAUNCH_T(DT, OT, 2, EPW);                                                                     \
    else if (D <= 4096) LAUNCH_T(DT, OT, 4, EPW);                                                                \
    else LAUNCH_T(DT, OT, 8, EPW);                                                                               \
  } while (0)
#define BY_WIDTH(DT, OT, SCORED)                                                                                 \
  do {                                                                                                           \
    if (D <= 2048) LAUNCH(DT, OT, SCORED, 2);                                                                    \
    else if (D <= 4096) LAUNCH(DT, OT, SCORED, 4);                                                               \
    else if (D <= 6144) LAUNCH(DT, OT, SCORED, 6);                                                               \
    else LAUNCH(DT, OT, SCORED, 8);                                                                              \
  } while (0)
#define GO(DT, OT)                                                                                               \
  do {                                                                                                           \
    Delta<DT> dl = {delta_kind == 1 ? (const DT*)delta : nullptr,                                                \
                    delta_kind == 2 ? (const DT*)routed : nullptr, inv_in, (const DT*)shared, k_in,              \
                    (const DT*)self, self_w, self_k};                                                            \
    if (by_token && E <= 8) TOKEN_BY_WIDTH(DT, OT, 2);                                                           \
    else if (by_token) TOKEN_BY_WIDTH(DT, OT, 4);                                                                \
    else if (scored) BY_WIDTH(DT, OT, true);                                                                     \
    else BY_WIDTH(DT, OT, false);                                                                                \
  } while (0)
  if (delta_is_bf16) {
    if (out_is_bf16) GO(bf16_t, bf16_t); else GO(bf16_t, float);
  } else {
    if (out_is_bf16) GO(float, bf16_t); else GO(float, float);
  }
#undef GO
#undef BY_WIDTH
#undef TOKEN_BY_WIDTH
#undef LAUNCH_T
#undef LAUNCH
  JLE_LAUNCH_CHECK();
  return 0;
}
