// The gated delta rule: a matrix memory S (dk x dv, float32) per head and request, written and read token by token,
//     S <- g S;   u = beta (v - S^T k);   S <- S + k u^T;   o = S^T q
// with q, k unit vectors per kv head (x / sqrt(sum(x^2) + floor), q times dk^(-1/2)), beta = sigmoid(b),
// g = exp(-exp(A) softplus(a + dt)).  Kernels:
//   gdr_prepare_kernel   the unit vectors (float32), beta and the decay of every token of the step
//   gdr_scan_kernel      the recurrence: a column of S depends on nothing but itself, k, q, v of its own place, beta
//                        and g, so a wavefront takes 64 / KS columns of one head, KS neighbouring lanes share a
//                        column (each holds R consecutive rows of it in registers), and the two dot products are
//                        finished with log2(KS) lane swaps; the next tokens' rows are asked for before these are used
//   gdr_chunk_kernel, gdr_carry_kernel   the same recurrence 64 tokens at a time on the float32 matrix instructions, for
//                        segments of many tokens (below)
//   gdr_single_kernel    all of it in one launch, for steps of single tokens
//   gdr_out_kernel       o / sqrt(mean(o^2) + eps) * w * silu(gate), rounded to the run dtype
// The memory lies [slot][half][H][dv][dk] (a column's rows together); a step reads the half `phase` and writes the other.
// What a token's result depends on beside its own sequence is rounding: the scan goes token after token, its sums over a
// column in an order that follows from how many lanes share the column, which follows from the sizes and the number of
// segments in the step; single tokens have a third order; and whether a segment goes by chunks, which begin at the step's
// first token of it, is a question of its length and of the work of all such segments together.
#include "common.h"

using namespace jle;

namespace {

template <typename T>
__global__ __launch_bounds__(64) void gdr_prepare_kernel(const T* __restrict__ rows, const float* __restrict__ gates,
                                                         const float* __restrict__ a_log,
                                                         const float* __restrict__ dt_bias, float* __restrict__ qn,
                                                         float* __restrict__ kn, float* __restrict__ beta,
                                                         float* __restrict__ decay, float* __restrict__ kq,
                                                         float floor, int H, int G, int dk, int dv, int dkp) {
  const int n = blockIdx.x, g = blockIdx.y, lane = threadIdx.x;
  const int C = 2 * G * dk + H * dv;
  if (g == G) {  // the write strengths and decays of the token's heads
    for (int h = lane; h < H; h += 64) {
      const float b = gates[(size_t)n * 2 * H + h], a = gates[(size_t)n * 2 * H + H + h] + dt_bias[h];
      beta[(size_t)n * H + h] = 1.0f / (1.0f + expf(-b));
      const float sp = a > 20.f ? a : log1pf(expf(a));
      decay[(size_t)n * H + h] = expf(-expf(a_log[h]) * sp);
    }
    return;
  }
  for (int which = 0; which < 2; ++which) {
    const T* src = rows + (size_t)n * C + (size_t)(which * G + g) * dk;
    float* dst = (which == 0 ? qn : kn) + ((size_t)n * G + g) * dkp;  // (rows of dkp >= dk floats, zeros behind)
    float ss = 0.f;
    for (int e = lane; e < dk; e += 64) {
      const float x = Num<T>::load(src + e);
      ss = __builtin_fmaf(x, x, ss);
    }
    float inv = 1.0f / sqrtf(wave_sum(ss) + floor);
    if (which == 0) inv *= 1.0f / sqrtf((float)dk);
    for (int e = lane; e < dkp; e += 64) dst[e] = e < dk ? Num<T>::load(src + e) * inv : 0.f;
  }
  // the product of the token's own two unit vectors (what its write adds to its own read-out)
  const float* qd = qn + ((size_t)n * G + g) * dkp;
  const float* kd = kn + ((size_t)n * G + g) * dkp;
  float d = 0.f;
  for (int e = lane; e < dk; e += 64) d = __builtin_fmaf(qd[e], kd[e], d);  // (this lane's own stores)
  d = wave_sum(d);
  if (lane == 0) kq[(size_t)n * G + g] = d;
}

// KS lanes share a column, each with R consecutive rows of it (KS * R = dkp >= dk, the unit vectors' rows padded with
// zeros to that).  The wavefront brings the unit vectors, write strengths and decays of TB tokens into shared memory
// at a time (asked for while the TB tokens before are worked on), and a lane its own values into registers.
// the sum over the KS neighbouring lanes that share a column (every one of them gets it, the same bits in all):
// within a row of 16 lanes by the lane-permuting operand modes, beyond by the cross-lane read
template <int CTRL>
__device__ __forceinline__ float lanes_permuted(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
template <int KS>
__device__ __forceinline__ float column_lanes_sum(float v) {
  if (KS >= 2) v += lanes_permuted<0xB1>(v);    // lanes 1 0 3 2 of every four
  if (KS >= 4) v += lanes_permuted<0x4E>(v);    // lanes 2 3 0 1 of every four
  if (KS >= 8) v += lanes_permuted<0x141>(v);   // every eight mirrored
  if (KS >= 16) v += lanes_permuted<0x140>(v);  // every sixteen mirrored
  if (KS >= 32) v += __shfl_xor(v, 16, 64);
  if (KS >= 64) v += __shfl_xor(v, 32, 64);
  return v;
}

typedef float f32x4 __attribute__((ext_vector_type(4)));  // (a plain vector type: arrays of it stay in registers)

template <int KS, int R>
struct ScanShape {
  static constexpr int kDkp = KS * R;
  static constexpr int kTB = kDkp <= 256 ? 16 : kDkp <= 512 ? 8 : kDkp <= 1024 ? 4 : 2;
  static constexpr int kVecs = (kTB * kDkp / 4 + 63) / 64;  // 16-byte pieces a lane brings in per array
};

template <typename T, int KS, int R>
__global__ __launch_bounds__(64) void gdr_scan_kernel(const T* __restrict__ rows, const float* __restrict__ qn,
                                                      const float* __restrict__ kn, const float* __restrict__ beta,
                                                      const float* __restrict__ decay, const float* __restrict__ kq,
                                                      float* __restrict__ state,
                                                      const int* __restrict__ cu_seqlens,
                                                      const int* __restrict__ state_slots,
                                                      const int* __restrict__ state_phase, float* __restrict__ o_raw,
                                                      int H, int G, int dk, int dv,
                                                      int chunked_from /* longer segments go by chunks */) {
  using Shape = ScanShape<KS, R>;
  constexpr int TB = Shape::kTB, DKP = Shape::kDkp, NV = Shape::kVecs, cols = 64 / KS;
  __shared__ f32x4 sk[TB * DKP / 4], sq[TB * DKP / 4];
  __shared__ f32x4 ssc[TB];  // a token's decay, write strength and k . q together: one trip to shared memory
  const int seg = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int ks = lane % KS, c = blockIdx.z * cols + lane / KS;  // (a column's lanes are neighbours)
  const bool live = c < dv;
  const int g = h / (H / G);
  const int C = 2 * G * dk + H * dv;
  const int t0 = cu_seqlens[seg], t1 = cu_seqlens[seg + 1];
  if (t0 >= t1 || t1 - t0 >= chunked_from) return;
  const size_t slot = (size_t)state_slots[seg];
  const int phase = state_phase[seg];
  const float* s_old = state + ((slot * 2 + phase) * H + h) * (size_t)dk * dv;
  float* s_new = state + ((slot * 2 + (1 - phase)) * H + h) * (size_t)dk * dv;
  const int k0 = ks * R;
  float S[R];
#pragma unroll
  for (int i = 0; i < R; ++i) S[i] = 0.f;
  // (a column's dk rows lie together: its KS lanes read neighbouring pieces of R floats)
  if (live) {
    if (dk % 4 == 0) {
#pragma unroll
      for (int i = 0; i < R; i += 4) {
        if (k0 + i < dk) {
          const float4 v = *reinterpret_cast<const float4*>(s_old + (size_t)c * dk + k0 + i);
          S[i] = v.x; S[i + 1] = v.y; S[i + 2] = v.z; S[i + 3] = v.w;
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < R; ++i)
        if (k0 + i < dk) S[i] = s_old[(size_t)c * dk + k0 + i];
    }
  }

  f32x4 stk[NV], stq[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) stk[j] = stq[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float vnext[TB], vcur[TB], bnext = 0.f, gnext = 1.f, kqnext = 0.f;
  auto ask = [&](int tb) __attribute__((always_inline)) {  // the TB tokens from tb on (those beyond the segment's end: its last token again, unused)
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int f = lane + 64 * j;
      if (f < TB * DKP / 4) {
        const int tt = f / (DKP / 4), off = f - tt * (DKP / 4);
        const size_t row = ((size_t)min(tb + tt, t1 - 1) * G + g) * DKP;
        stk[j] = reinterpret_cast<const f32x4*>(kn + row)[off];
        stq[j] = reinterpret_cast<const f32x4*>(qn + row)[off];
      }
    }
#pragma unroll
    for (int tt = 0; tt < TB; ++tt)
      vnext[tt] = live ? Num<T>::load(rows + (size_t)min(tb + tt, t1 - 1) * C + 2 * G * dk + (size_t)h * dv + c) : 0.f;
    if (lane < TB) {  // (places behind the segment's end: a step that changes nothing, no write and no decay)
      const size_t at = (size_t)min(tb + lane, t1 - 1) * H + h;
      bnext = tb + lane < t1 ? beta[at] : 0.f;
      gnext = tb + lane < t1 ? decay[at] : 1.f;
      kqnext = kq[(size_t)min(tb + lane, t1 - 1) * G + g];
    }
  };
  auto put = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int f = lane + 64 * j;
      if (f < TB * DKP / 4) {
        sk[f] = stk[j];
        sq[f] = stq[j];
      }
    }
    if (lane < TB) {
      ssc[lane] = f32x4{gnext, bnext, kqnext, 0.f};
    }
#pragma unroll
    for (int tt = 0; tt < TB; ++tt) vcur[tt] = vnext[tt];
  };
  ask(t0);
  put();
  __syncthreads();
  for (int tb = t0; tb < t1; tb += TB) {
    const bool more = tb + TB < t1;
    if (more) ask(tb + TB);
    float outs[TB];  // (the block's read-outs: stored together behind its last token)
    auto token = [&](int tt) __attribute__((always_inline)) {
      float kc[R], qc[R];
#pragma unroll
      for (int i = 0; i < R; i += 4) {
        const f32x4 a = sk[(tt * DKP + k0 + i) / 4], b = sq[(tt * DKP + k0 + i) / 4];
        kc[i] = a.x; kc[i + 1] = a.y; kc[i + 2] = a.z; kc[i + 3] = a.w;
        qc[i] = b.x; qc[i + 1] = b.y; qc[i + 2] = b.z; qc[i + 3] = b.w;
      }
      // With S the memory before the token: the write is u = beta (v - g S^T k), the read-out S'^T q of the memory
      // after it, S' = g S + k u^T, is g S^T q + (k . q) u: both products with S stand side by side, and from one
      // token to the next leads one multiply-add of the memory.
      const f32x4 sc = ssc[tt];
      const float gc = sc.x, bc = sc.y, kqc = sc.z;
      float d4[4] = {0.f, 0.f, 0.f, 0.f}, o4[4] = {0.f, 0.f, 0.f, 0.f};  // (four sums side by side, not a chain of R)
#pragma unroll
      for (int i = 0; i < R; ++i) {
        d4[i & 3] = __builtin_fmaf(S[i], kc[i], d4[i & 3]);
        o4[i & 3] = __builtin_fmaf(S[i], qc[i], o4[i & 3]);
      }
      const float dot = column_lanes_sum<KS>((d4[0] + d4[1]) + (d4[2] + d4[3]));
      const float oq = column_lanes_sum<KS>((o4[0] + o4[1]) + (o4[2] + o4[3]));
      const float u = bc * (vcur[tt] - gc * dot);
      const float out = __builtin_fmaf(kqc, u, gc * oq);
#pragma unroll
      for (int i = 0; i < R; ++i) S[i] = __builtin_fmaf(kc[i], u, gc * S[i]);
      outs[tt] = out;
    };
    if (tb + TB <= t1) {  // a whole block: no branch around a token, one stretch of code that the compiler may interleave
#pragma unroll
      for (int tt = 0; tt < TB; ++tt) token(tt);
    } else {  // (the segment's last tokens, or all of a short one: no work for places behind its end)
#pragma unroll
      for (int tt = 0; tt < TB; ++tt)
        if (tb + tt < t1) token(tt);
    }
    if (live && ks == 0) {
      float* op = o_raw + ((size_t)tb * H + h) * dv + c;
#pragma unroll
      for (int tt = 0; tt < TB; ++tt)
        if (tb + tt < t1) op[(size_t)tt * H * dv] = outs[tt];
    }
    __syncthreads();
    if (more) put();
    __syncthreads();
  }
  if (live) {
    if (dk % 4 == 0) {
#pragma unroll
      for (int i = 0; i < R; i += 4)
        if (k0 + i < dk)
          *reinterpret_cast<float4*>(s_new + (size_t)c * dk + k0 + i) = float4{S[i], S[i + 1], S[i + 2], S[i + 3]};
    } else {
#pragma unroll
      for (int i = 0; i < R; ++i)
        if (k0 + i < dk) s_new[(size_t)c * dk + k0 + i] = S[i];
    }
  }
}

// ------------------------------------------------------------------ many tokens: 64 at a time
// Within a chunk that starts with the memory S, let d(t, j) be the product of the decays behind token j up to token t, and
// c(t) of those from the chunk's start up to t.  The writes follow from the memory before the chunk and from each other,
//     u_t = beta_t (v_t - c(t) S^T k_t) - sum_{j < t} L_tj u_j,      L_tj = beta_t d(t, j) (k_t . k_j),
// a unit lower triangular system.  With T = (I + L)^-1, per chunk and independent of S (gdr_chunk_kernel):
//     U0 = T (beta V),   W = T (beta c K),   P_tj = d(t, j) (q_t . k_j) for j <= t;
// then from chunk to chunk (gdr_carry_kernel):
//     U = U0 - W S,   O = c Q S + P U,   S <- c(end) S + K^T (d(end, .) U).
// Everything is float32 on the float32 matrix instructions, the decays' products formed by multiplying, as the scan does
// (differences of summed logarithms would lose what a strong decay leaves of a later weak one).  One prompt of 2,048
// tokens, 16 heads of 128 x 128 on 8 kv heads: 31 + 93 us instead of the scan's 726; a step's 25 prompts of 80 tokens
// 51 + 88 instead of 165.
// v_mfma_f32_16x16x4: lane (m = lane % 16, g = lane / 16) holds A[m][k] and B[k][m] of one k, and of the result the rows
// 4 g .. 4 g + 3 of column m.  Taking k = 16 r + 4 g + i for the i-th product of tile r, A and B are 16-byte pieces of
// rows, and a result's registers are the next product's B operand as they are.
constexpr int kChunk = 64;

__device__ __forceinline__ f32x4 mfma4(const f32x4& a, const f32x4& b, f32x4 c) {  // 16 of k: four products
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], c, 0, 0, 0);
  return c;
}

// What goes from one kernel to the other lies as the operands that the second reads: a tile of 16 x 16 numbers is a
// kilobyte, a lane's 16 bytes in the lanes' order.  (As plain matrices, 16 rows a load instruction, every lane's piece was
// a request of its own to the first-level cache: 142 us instead of 93 for the second kernel, 2,048 tokens, 16 heads.)
__device__ __forceinline__ int operand_at(int row, int col) {  // of an A operand's tile (rows its lanes, columns its k)
  return (((col & 15) >> 2) * 16 + (row & 15)) * 4 + (col & 3);
}

// One block per (chunk, head).  ws: per (chunk, head) W (negated) [4][DK / 16] tiles, U0 [dv / 16][4] tiles as results, P
// [4][4] tiles, and c(t), d(end, t) [2][64]; per (chunk, kv head) K^T [DK / 16][4] and Q [4][DK / 16] tiles.
template <typename T, int DK>
__global__ __launch_bounds__(256, 2) void gdr_chunk_kernel(const T* __restrict__ rows, const float* __restrict__ qn,
                                                           const float* __restrict__ kn, const float* __restrict__ beta,
                                                           const float* __restrict__ decay, const int* __restrict__ chunks,
                                                           float* __restrict__ ws_w, float* __restrict__ ws_u,
                                                           float* __restrict__ ws_p, float* __restrict__ ws_kt,
                                                           float* __restrict__ ws_q, float* __restrict__ ws_s, int H, int G,
                                                           int dv) {
  constexpr int NT = DK / 16, KP = DK + 4, LP = kChunk + 4;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  float* sk = smem;               // [64][KP]: the chunk's keys
  float* sd = sk + kChunk * KP;   // [64][LP]: d(t, j), then T
  float* sl = sd + kChunk * LP;   // [64][LP]: L
  float* sb = sl + kChunk * LP;   // beta, decay, c(t)
  float *sg = sb + kChunk, *sc = sg + kChunk;
  const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, g = lane >> 4;
  const int w = wave_index();
  const int c = blockIdx.x, h = blockIdx.y, kv = h / (H / G);
  const int tok0 = chunks[3 * c + 1], nt = chunks[3 * c + 2];
  const size_t at = (size_t)c * H + h;
  // (places behind the segment's end: keys of zeros, no write, no decay)
  for (int idx = tid; idx < kChunk * DK / 4; idx += 256) {
    const int t = idx / (DK / 4), e = idx - t * (DK / 4);
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (t < nt) v = reinterpret_cast<const f32x4*>(kn + ((size_t)(tok0 + t) * G + kv) * DK)[e];
    *reinterpret_cast<f32x4*>(sk + t * KP + 4 * e) = v;
  }
  if (tid < kChunk) {
    sb[tid] = tid < nt ? beta[(size_t)(tok0 + tid) * H + h] : 0.f;
    sg[tid] = tid < nt ? decay[(size_t)(tok0 + tid) * H + h] : 1.f;
  }
  __syncthreads();
  if (w == 3) {  // a column of d a lane
    float d = 0.f, p = 1.f, mine = 1.f;
    for (int t = 0; t < kChunk; ++t) {
      const float gt = sg[t];
      d = t == lane ? 1.f : d * gt;
      p *= gt;
      mine = t == lane ? p : mine;
      sd[t * LP + lane] = d;
    }
    sc[lane] = mine;
  }
  // the lower tiles (i, j) of K K^T and Q K^T, ten pairs for four wavefronts (the third and fourth: two each)
  f32x4 kk[3], qk[3];
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    const int pair = w + 4 * s;
    if (pair >= 10) break;
    const int i = pair >= 6 ? 3 : pair >= 3 ? 2 : pair >= 1 ? 1 : 0, j = pair - i * (i + 1) / 2;
    const int t = min(16 * i + c16, nt - 1);
    const float* qrow = qn + ((size_t)(tok0 + t) * G + kv) * DK + 4 * g;
    const float* krow = sk + (16 * i + c16) * KP + 4 * g;
    const float* brow = sk + (16 * j + c16) * KP + 4 * g;
    f32x4 qa[NT];
#pragma unroll
    for (int r = 0; r < NT; ++r) qa[r] = *reinterpret_cast<const f32x4*>(qrow + 16 * r);
    kk[s] = qk[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < NT; ++r) {
      const f32x4 b = *reinterpret_cast<const f32x4*>(brow + 16 * r), a = *reinterpret_cast<const f32x4*>(krow + 16 * r);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        kk[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[x], b[x], kk[s], 0, 0, 0);
        qk[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[r][x], b[x], qk[s], 0, 0, 0);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    const int pair = w + 4 * s;
    if (pair >= 10) break;
    const int i = pair >= 6 ? 3 : pair >= 3 ? 2 : pair >= 1 ? 1 : 0, j = pair - i * (i + 1) / 2;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int t = 16 * i + 4 * g + x, u = 16 * j + c16;
      const float d = sd[t * LP + u];
      sl[t * LP + u] = u < t ? sb[t] * (d * kk[s][x]) : 0.f;
      ws_p[(at * 16 + 4 * i + j) * 256 + operand_at(t, u)] = u <= t ? d * qk[s][x] : 0.f;
    }
  }
  for (int idx = tid; idx < 6 * 256; idx += 256) {  // (the tiles above the diagonal)
    const int pair = idx >> 8, j = pair >= 3 ? 3 : pair >= 1 ? 2 : 1, i = pair - j * (j - 1) / 2;
    ws_p[(at * 16 + 4 * i + j) * 256 + tid] = 0.f;
  }
  if (tid < kChunk) {
    ws_s[at * 2 * kChunk + tid] = sc[tid];
    ws_s[at * 2 * kChunk + kChunk + tid] = sd[(kChunk - 1) * LP + tid];
  }
  if (h % (H / G) == 0) {  // (the head's keys are its group's)
    f32x4* kt = reinterpret_cast<f32x4*>(ws_kt + ((size_t)c * G + kv) * DK * kChunk);
    f32x4* qt = reinterpret_cast<f32x4*>(ws_q + ((size_t)c * G + kv) * DK * kChunk);
    for (int idx = tid; idx < DK * kChunk / 4; idx += 256) {
      const int tile = idx >> 6;  // (lane: idx % 64, as tid)
      const float* src = sk + (16 * (tile & 3) + 4 * g) * KP + 16 * (tile >> 2) + c16;
      kt[idx] = f32x4{src[0], src[KP], src[2 * KP], src[3 * KP]};
      const int t = min(16 * (tile / NT) + c16, nt - 1);
      qt[idx] = *reinterpret_cast<const f32x4*>(qn + ((size_t)(tok0 + t) * G + kv) * DK + 16 * (tile % NT) + 4 * g);
    }
  }
  __syncthreads();
  // T: the inverses of the four diagonal tiles, a column a lane, by forward substitution
  if (lane < 16) {
    const float* lt = sl + 16 * w * LP + 16 * w;
    float x[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      float v = t == lane ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < t; ++j) v = __builtin_fmaf(-lt[t * LP + j], x[j], v);
      x[t] = v;
    }
#pragma unroll
    for (int t = 0; t < 16; ++t) sd[(16 * w + t) * LP + 16 * w + lane] = x[t];
  }
  __syncthreads();
  // the tiles below them, a column of tiles a wavefront: T_ij = -T_ii sum_{j <= k < i} L_ik T_kj
  if (w < 3) {
    f32x4 col[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) col[0][x] = sd[(16 * w + 4 * g + x) * LP + 16 * w + c16];
#pragma unroll
    for (int n = 1; n < 4; ++n) {
      const int i = w + n;
      if (i > 3) break;
      f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < n; ++k)
        sum = mfma4(*reinterpret_cast<const f32x4*>(sl + (16 * i + c16) * LP + 16 * (w + k) + 4 * g), col[k], sum);
      const f32x4 t = mfma4(*reinterpret_cast<const f32x4*>(sd + (16 * i + c16) * LP + 16 * i + 4 * g), sum, f32x4{0.f, 0.f, 0.f, 0.f});
      col[n] = -t;
#pragma unroll
      for (int x = 0; x < 4; ++x) sd[(16 * i + 4 * g + x) * LP + 16 * w + c16] = col[n][x];
    }
  }
  __syncthreads();
  // W and U0, a tile of 16 columns a wavefront and turn
  const int C = 2 * G * DK + H * dv;
  for (int ct = w; ct < NT + dv / 16; ct += 4) {
    f32x4 b[4];
    if (ct < NT) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const int t = 16 * r + 4 * g + x;
          b[r][x] = -(sb[t] * sc[t]) * sk[t * KP + 16 * ct + c16];
        }
    } else {
      const T* v = rows + 2 * G * DK + (size_t)h * dv + 16 * (ct - NT) + c16;
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const int t = 16 * r + 4 * g + x;
          b[r][x] = sb[t] * Num<T>::load(v + (size_t)(tok0 + min(t, nt - 1)) * C);
        }
    }
    f32x4 acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int i = r; i < 4; ++i)
        acc[i] = mfma4(*reinterpret_cast<const f32x4*>(sd + (16 * i + c16) * LP + 16 * r + 4 * g), b[r], acc[i]);
    if (ct < NT) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int x = 0; x < 4; ++x) ws_w[((at * 4 + i) * NT + ct) * 256 + operand_at(4 * g + x, c16)] = acc[i][x];
    } else {
      f32x4* dst = reinterpret_cast<f32x4*>(ws_u + at * kChunk * dv) + (size_t)(ct - NT) * 256 + lane;
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[64 * i] = acc[i];
    }
  }
}

// One block per (segment, head, 16 columns of the memory): four wavefronts, each with 16 of a chunk's tokens and a quarter
// of the memory's rows; the writes and the memory go round through shared memory (two barriers a chunk), every operand
// comes straight from the scratch arrays into registers and is asked for as soon as the chunk before has used its
// registers.  A chunk is 112 matrix instructions a wavefront (DK = 128), 1.5 us of the 2.9 it takes at 2,048 tokens and 16
// heads (128 blocks); without its loads it takes 2.3, so what the rest is made of is barriers and trips through shared
// memory first, the 110 KB of operands second.
// In a chunk the zeros above the diagonals of T and P meet what later tokens write, and zero times an infinity or NaN is
// NaN: one in a token's value, key or gates would reach the tokens before it.  It stays in the memory's column, so a column
// that is not finite at the segment's end is worked out again token by token, in the order of gdr_scan_kernel with 16 lanes
// a column, from the memory before the segment (which this step leaves as it is).
template <typename T, int DK>
__global__ __launch_bounds__(256, 2) void gdr_carry_kernel(const float* __restrict__ ws_q, const int* __restrict__ segs,
                                                           const int* __restrict__ cu_seqlens,
                                                           const int* __restrict__ state_slots,
                                                           const int* __restrict__ state_phase, float* __restrict__ state,
                                                           const float* __restrict__ ws_w, const float* __restrict__ ws_u,
                                                           const float* __restrict__ ws_p, const float* __restrict__ ws_kt,
                                                           const float* __restrict__ ws_s, float* __restrict__ o_raw, int N,
                                                           int H, int G, int dv, const T* __restrict__ rows,
                                                           const float* __restrict__ qn, const float* __restrict__ kn,
                                                           const float* __restrict__ beta, const float* __restrict__ decay,
                                                           const float* __restrict__ kq) {
  constexpr int NT = DK / 16, OWN = NT / 4;
  __shared__ f32x4 s_mem[NT][64], s_u[4][64], s_du[4][64];
  __shared__ int s_bad[4];
  const int lane = threadIdx.x & 63, c16 = lane & 15, g = lane >> 4;
  const int w = wave_index();
  const int h = blockIdx.x % H, kv = h / (H / G);
  const int cb = blockIdx.x / H % (dv / 16), col = 16 * cb + c16;
  const int* sgm = segs + 3 * (blockIdx.x / H / (dv / 16));
  const int seg = sgm[0], c0 = sgm[1], c1 = c0 + sgm[2];
  const size_t slot = (size_t)state_slots[seg];
  const int phase = state_phase[seg];
  const size_t own = (((slot * 2 + phase) * H + h) * (size_t)dv + col) * DK;
  const size_t own_new = (((slot * 2 + (1 - phase)) * H + h) * (size_t)dv + col) * DK;
  f32x4 S[NT];
#pragma unroll
  for (int r = 0; r < NT; ++r) S[r] = *reinterpret_cast<const f32x4*>(state + own + 16 * r + 4 * g);
  f32x4 W[NT], Q[NT], P[4], KT[OWN][4], U0, cs, ds;
  float cend;
  const int tok0 = cu_seqlens[seg], len = cu_seqlens[seg + 1] - tok0;
  int zero;  // (not known to be the same in all lanes: a load by it goes the vectors' way, in order with the others)
  asm("v_mov_b32 %0, 0" : "=v"(zero));
  auto ask_front = [&](int c) __attribute__((always_inline)) {
    const f32x4* wr = reinterpret_cast<const f32x4*>(ws_w + (((size_t)c * H + h) * 4 + w) * DK * 16) + lane;
    const f32x4* qr = reinterpret_cast<const f32x4*>(ws_q + (((size_t)c * G + kv) * 4 + w) * DK * 16) + lane;
#pragma unroll
    for (int r = 0; r < NT; ++r) {
      W[r] = wr[64 * r];
      Q[r] = qr[64 * r];
    }
    U0 = reinterpret_cast<const f32x4*>(ws_u + ((size_t)c * H + h) * kChunk * dv)[(4 * cb + w) * 64 + lane];
  };
  auto ask_back = [&](int c) __attribute__((always_inline)) {
    const float* sr = ws_s + ((size_t)c * H + h) * 2 * kChunk;
    cs = *reinterpret_cast<const f32x4*>(sr + 16 * w + 4 * g);
    ds = *reinterpret_cast<const f32x4*>(sr + kChunk + 16 * w + 4 * g);
    cend = sr[kChunk - 1 + zero];
    const f32x4* pr = reinterpret_cast<const f32x4*>(ws_p + (((size_t)c * H + h) * 4 + w) * 1024) + lane;
#pragma unroll
    for (int r = 0; r < 4; ++r) P[r] = pr[64 * r];
    const f32x4* kr = reinterpret_cast<const f32x4*>(ws_kt + ((size_t)c * G + kv) * DK * kChunk) + (size_t)OWN * w * 256 + lane;
#pragma unroll
    for (int q = 0; q < OWN; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) KT[q][r] = kr[64 * (4 * q + r)];
  };
  const size_t behind = (size_t)N * H * dv;  // (64 places that nobody reads)
  ask_front(c0);
  __builtin_amdgcn_sched_barrier(0);
  ask_back(c0);
  __builtin_amdgcn_sched_barrier(0);
  f32x4 mine[OWN];
  for (int c = c0; c < c1; ++c) {
    // (loads and stores without branches around them: the compiler then knows how many are on their way and waits for those
    // it needs; with the last chunk's loads and the rows behind the segment's end under conditions it waited for all of
    // them, the stores too, at every chunk's start)
    const int next = min(c + 1, c1 - 1);
    f32x4 u = U0, o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < NT; ++r)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        u = __builtin_amdgcn_mfma_f32_16x16x4f32(W[r][x], S[r][x], u, 0, 0, 0);
        o = __builtin_amdgcn_mfma_f32_16x16x4f32(Q[r][x], S[r][x], o, 0, 0, 0);
      }
    s_u[w][lane] = u;
    s_du[w][lane] = u * ds;
    o *= cs;
    ask_front(next);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) o = mfma4(P[r], s_u[r][lane], o);
#pragma unroll
    for (int q = 0; q < OWN; ++q) {
      // (the memory's tiles are all in registers; which of them are this wavefront's is known at run time only)
      mine[q] = S[q];
#pragma unroll
      for (int n = 1; n < 4; ++n) mine[q] = w == n ? S[OWN * n + q] : mine[q];
      mine[q] *= cend;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const f32x4 du = s_du[r][lane];
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int q = 0; q < OWN; ++q) mine[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(KT[q][r][x], du[x], mine[q], 0, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < OWN; ++q) s_mem[OWN * w + q][lane] = mine[q];
    ask_back(next);
    __builtin_amdgcn_sched_barrier(0);
    const int t = kChunk * (c - c0) + 16 * w + 4 * g;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const size_t dst = ((size_t)(tok0 + t + x) * H + h) * dv + col;
      o_raw[t + x < len ? dst : behind + lane] = o[x];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < NT; ++r) S[r] = s_mem[r][lane];
  }
  bool bad = false;
#pragma unroll
  for (int q = 0; q < OWN; ++q)
#pragma unroll
    for (int x = 0; x < 4; ++x) bad |= !(fabsf(mine[q][x]) <= 3.402823466e38f);
  unsigned long long mask = __ballot(bad);
  mask |= mask >> 32;
  mask |= mask >> 16;
  if (lane == 0) s_bad[w] = (int)(mask & 0xffff);
  __syncthreads();
  const int bad_cols = s_bad[0] | s_bad[1] | s_bad[2] | s_bad[3];
  if (!(bad_cols >> c16 & 1)) {
#pragma unroll
    for (int q = 0; q < OWN; ++q) *reinterpret_cast<f32x4*>(state + own_new + 16 * (OWN * w + q) + 4 * g) = mine[q];
  }
  if (bad_cols == 0) return;
  constexpr int R = DK / 16;  // rows of a column in each of its 16 lanes
  const int mc = threadIdx.x >> 4, ks = threadIdx.x & 15;
  const bool redo = bad_cols >> mc & 1;
  if (!__any(redo)) return;
  const size_t at = (size_t)(16 * cb + mc) * DK + R * ks;
  const float* s_old = state + ((slot * 2 + phase) * H + h) * (size_t)dv * DK + at;
  float* s_new = state + ((slot * 2 + (1 - phase)) * H + h) * (size_t)dv * DK + at;
  float M[R];
#pragma unroll
  for (int i = 0; i < R; ++i) M[i] = s_old[i];
  const int C = 2 * G * DK + H * dv;
  for (int t = tok0; t < tok0 + len; ++t) {
    const float* kr = kn + ((size_t)t * G + kv) * DK + R * ks;
    const float* qr = qn + ((size_t)t * G + kv) * DK + R * ks;
    const float v = Num<T>::load(rows + (size_t)t * C + 2 * G * DK + (size_t)h * dv + 16 * cb + mc);
    const float gc = decay[(size_t)t * H + h], bc = beta[(size_t)t * H + h], kqc = kq[(size_t)t * G + kv];
    float d4[4] = {0.f, 0.f, 0.f, 0.f}, o4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < R; ++i) {
      d4[i & 3] = __builtin_fmaf(M[i], kr[i], d4[i & 3]);
      o4[i & 3] = __builtin_fmaf(M[i], qr[i], o4[i & 3]);
    }
    const float dot = column_lanes_sum<16>((d4[0] + d4[1]) + (d4[2] + d4[3]));
    const float oq = column_lanes_sum<16>((o4[0] + o4[1]) + (o4[2] + o4[3]));
    const float u = bc * (v - gc * dot);
#pragma unroll
    for (int i = 0; i < R; ++i) M[i] = __builtin_fmaf(kr[i], u, gc * M[i]);
    if (redo && ks == 0) o_raw[((size_t)t * H + h) * dv + 16 * cb + mc] = __builtin_fmaf(kqc, u, gc * oq);
  }
  if (redo) {
#pragma unroll
    for (int i = 0; i < R; ++i) s_new[i] = M[i];
  }
}

// What the chunked form needs of a step: its chunks (segment, first token, tokens), the segments that go by chunks
// (segment, first chunk, chunks) - those of `from` tokens and more -, whether others are left, and scratch.
struct ByChunks {
  const int *chunks, *segs;
  int num_chunks, num_segs, from, others;
  float* ws;
};

inline size_t chunk_floats(int H, int G, int dk, int dv) {  // scratch of one chunk
  return (size_t)H * (kChunk * (dk + dv) + kChunk * kChunk + 2 * kChunk) + (size_t)2 * G * dk * kChunk;
}

template <typename T, int DK>
int launch_chunks(const ByChunks& b, const T* rows, const float* qn, const float* kn, const float* beta, const float* decay,
                  const float* kq, float* state, const int* cu_seqlens, const int* state_slots, const int* state_phase, float* o_raw, int N,
                  int H, int G, int dv, hipStream_t s) {
  const size_t n = (size_t)b.num_chunks * H;
  float* ws_w = b.ws;
  float* ws_u = ws_w + n * kChunk * DK;
  float* ws_p = ws_u + n * kChunk * dv;
  float* ws_s = ws_p + n * kChunk * kChunk;
  float* ws_kt = ws_s + n * 2 * kChunk;
  float* ws_q = ws_kt + (size_t)b.num_chunks * G * DK * kChunk;
  constexpr int smem = (kChunk * (DK + 4) + 2 * kChunk * (kChunk + 4) + 3 * kChunk) * (int)sizeof(float);
  if (const int rc = allow_lds(gdr_chunk_kernel<T, DK>, smem)) return rc;
  hipLaunchKernelGGL((gdr_chunk_kernel<T, DK>), dim3(b.num_chunks, H), dim3(256), smem, s, rows, qn, kn, beta, decay,
                     b.chunks, ws_w, ws_u, ws_p, ws_kt, ws_q, ws_s, H, G, dv);
  JLE_LAUNCH_CHECK();
  hipLaunchKernelGGL((gdr_carry_kernel<T, DK>), dim3((unsigned)(b.num_segs * H * (dv / 16))), dim3(256), 0, s, ws_q, b.segs,
                     cu_seqlens, state_slots, state_phase, state, ws_w, ws_u, ws_p, ws_kt, ws_s, o_raw, N, H, G, dv, rows, qn,
                     kn, beta, decay, kq);
  JLE_LAUNCH_CHECK();
  return 0;
}

template <typename T>
__global__ __launch_bounds__(64) void gdr_out_kernel(const float* __restrict__ o_raw, const T* __restrict__ gate,
                                                     const float* __restrict__ w, T* __restrict__ out, float eps, int H,
                                                     int dv) {
  const int n = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const size_t base = ((size_t)n * H + h) * dv;
  float ss = 0.f;
  for (int e = lane; e < dv; e += 64) {
    const float x = o_raw[base + e];
    ss = __builtin_fmaf(x, x, ss);
  }
  const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)dv + eps);
  for (int e = lane; e < dv; e += 64) {
    const float z = Num<T>::load(gate + base + e);
    Num<T>::store(out + base + e, o_raw[base + e] * inv * w[e] * (z / (1.0f + expf(-z))));
  }
}

// ------------------------------------------------------------------ a step of single tokens
// One block per (request, head) does all of a token: unit vectors, write strength and decay (as gdr_prepare_kernel forms
// them), the memory's step, norm and gate (as gdr_out_kernel).  Eight lanes share a column of the memory and read its rows
// 128 bytes at a time, 64 columns a turn of the block's eight wavefronts; a lane has asked for all its pieces of CP turns
// before the first barrier, so the memory is on its way while the vectors are normed.  Bound by the memory's bytes, read
// once and written once: 64 requests with 16 heads of 128 x 128 23 us (134 MB, 5.8 TB/s), 8 requests 5.5, where the three
// launches, whose scan lays out 16 tokens' vectors for one, took 67 and 18.
template <typename T, int DK, int CP>
__global__ __launch_bounds__(512) void gdr_single_kernel(const T* __restrict__ rows, const float* __restrict__ gates,
                                                         const float* __restrict__ a_log, const float* __restrict__ dt_bias,
                                                         const float* __restrict__ norm_w, const T* __restrict__ gate,
                                                         float* __restrict__ state, const int* __restrict__ state_slots,
                                                         const int* __restrict__ state_phase, T* __restrict__ out, float eps,
                                                         float floor, int H, int G, int dv) {
  constexpr int PC = DK / 32;  // 16-byte pieces of a column in a lane
  __shared__ f32x4 sk[DK / 4], sq[DK / 4];
  __shared__ float so[64 * CP], s_beta, s_decay, s_kq;
  const int n = blockIdx.x, h = blockIdx.y, kv = h / (H / G);
  const int tid = threadIdx.x, lane = tid & 63, ks = tid & 7, c0 = tid >> 3;
  const int w = wave_index();
  const int C = 2 * G * DK + H * dv;
  const size_t slot = (size_t)state_slots[n];
  const int phase = state_phase[n];
  const float* s_old = state + ((slot * 2 + phase) * H + h) * (size_t)dv * DK + 4 * ks;
  float* s_new = state + ((slot * 2 + (1 - phase)) * H + h) * (size_t)dv * DK + 4 * ks;
  f32x4 S[CP][PC];
  float v[CP];
#pragma unroll
  for (int p = 0; p < CP; ++p) {
    const int c = min(c0 + 64 * p, dv - 1);
#pragma unroll
    for (int j = 0; j < PC; ++j)
      S[p][j] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(s_old + (size_t)c * DK + 32 * j));
    v[p] = Num<T>::load(rows + (size_t)n * C + 2 * G * DK + (size_t)h * dv + c);
  }
  if (w == 0) {
    float* dst[2] = {reinterpret_cast<float*>(sq), reinterpret_cast<float*>(sk)};
    float x[2][DK / 64];
#pragma unroll
    for (int which = 0; which < 2; ++which) {
      const T* src = rows + (size_t)n * C + (size_t)(which * G + kv) * DK;
      float ss = 0.f;
#pragma unroll
      for (int e = 0; e < DK / 64; ++e) {
        x[which][e] = Num<T>::load(src + lane + 64 * e);
        ss = __builtin_fmaf(x[which][e], x[which][e], ss);
      }
      float inv = 1.0f / sqrtf(wave_sum(ss) + floor);
      if (which == 0) inv *= 1.0f / sqrtf((float)DK);
#pragma unroll
      for (int e = 0; e < DK / 64; ++e) {
        x[which][e] *= inv;
        dst[which][lane + 64 * e] = x[which][e];
      }
    }
    float d = 0.f;
#pragma unroll
    for (int e = 0; e < DK / 64; ++e) d = __builtin_fmaf(x[0][e], x[1][e], d);
    d = wave_sum(d);
    if (lane == 0) s_kq = d;
  }
  if (tid == 64) {
    const float b = gates[(size_t)n * 2 * H + h], a = gates[(size_t)n * 2 * H + H + h] + dt_bias[h];
    s_beta = 1.0f / (1.0f + expf(-b));
    const float sp = a > 20.f ? a : log1pf(expf(a));
    s_decay = expf(-expf(a_log[h]) * sp);
  }
  __syncthreads();
  const float gc = s_decay, bc = s_beta, kqc = s_kq;
  f32x4 k[PC], q[PC];
#pragma unroll
  for (int j = 0; j < PC; ++j) {
    k[j] = sk[ks + 8 * j];
    q[j] = sq[ks + 8 * j];
  }
#pragma unroll
  for (int p = 0; p < CP; ++p) {
    f32x4 d4 = {0.f, 0.f, 0.f, 0.f}, o4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < PC; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        d4[i] = __builtin_fmaf(S[p][j][i], k[j][i], d4[i]);
        o4[i] = __builtin_fmaf(S[p][j][i], q[j][i], o4[i]);
      }
    const float dot = column_lanes_sum<8>((d4[0] + d4[1]) + (d4[2] + d4[3]));
    const float oq = column_lanes_sum<8>((o4[0] + o4[1]) + (o4[2] + o4[3]));
    const float u = bc * (v[p] - gc * dot);
    const int c = c0 + 64 * p;
    if (c < dv) {
#pragma unroll
      for (int j = 0; j < PC; ++j) {
        f32x4 t;
#pragma unroll
        for (int i = 0; i < 4; ++i) t[i] = __builtin_fmaf(k[j][i], u, gc * S[p][j][i]);
        __builtin_nontemporal_store(t, reinterpret_cast<f32x4*>(s_new + (size_t)c * DK + 32 * j));
      }
      if (ks == 0) so[c] = __builtin_fmaf(kqc, u, gc * oq);
    }
  }
  __syncthreads();
  float ss = 0.f;
  for (int e = lane; e < dv; e += 64) ss = __builtin_fmaf(so[e], so[e], ss);
  const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)dv + eps);
  for (int e = tid; e < dv; e += 512) {
    const size_t at = ((size_t)n * H + h) * dv + e;
    const float z = Num<T>::load(gate + at);
    Num<T>::store(out + at, so[e] * inv * norm_w[e] * (z / (1.0f + expf(-z))));
  }
}

template <typename T>
int launch_single(const T* rows, const float* gates, const float* a_log, const float* dt_bias, const float* norm_w,
                  const T* gate, float* state, const int* state_slots, const int* state_phase, T* out, int R, int H, int G,
                  int dk, int dv, float eps, float floor, hipStream_t s) {
#define JLE_SINGLE(DK_, CP_)                                                                                               \
  hipLaunchKernelGGL((gdr_single_kernel<T, DK_, CP_>), dim3(R, H), dim3(512), 0, s, rows, gates, a_log, dt_bias, norm_w, \
                     gate, state, state_slots, state_phase, out, eps, floor, H, G, dv)
  if (dk == 128) {
    if (dv <= 64) JLE_SINGLE(128, 1);
    else if (dv <= 128) JLE_SINGLE(128, 2);
    else JLE_SINGLE(128, 4);
  } else {
    if (dv <= 64) JLE_SINGLE(64, 1);
    else if (dv <= 128) JLE_SINGLE(64, 2);
    else JLE_SINGLE(64, 4);
  }
#undef JLE_SINGLE
  JLE_LAUNCH_CHECK();
  return 0;
}

template <typename T>
int launch_gdr(const T* rows, const float* gates, const float* a_log, const float* dt_bias, const float* norm_w,
               const T* gate, float* state, const int* cu_seqlens, const int* state_slots, const int* state_phase,
               float* qn, float* kn, float* beta, float* decay, float* kq, float* o_raw, T* out, int N, int R_, int H,
               int G, int dk, int dv, int dkp, float eps, float floor, const ByChunks& by_chunks, hipStream_t s) {
  // lanes a column: the fewest that leave a lane at most 16 rows of it (by the sizes alone)
  int KS = 1;
  while (KS < 64 && (dk + KS - 1) / KS > 16) KS <<= 1;
  const int per = (dk + KS - 1) / KS;
  const int RR = per <= 4 ? 4 : per <= 8 ? 8 : per <= 16 ? 16 : 32;
  if (dkp != KS * RR) return JLE_BAD_ARG;
  hipLaunchKernelGGL(gdr_prepare_kernel<T>, dim3(N, G + 1), dim3(64), 0, s, rows, gates, a_log, dt_bias, qn, kn, beta,
                     decay, kq, floor, H, G, dk, dv, dkp);
  JLE_LAUNCH_CHECK();
  if (by_chunks.num_segs > 0) {
    const int rc = dk == 128 ? launch_chunks<T, 128>(by_chunks, rows, qn, kn, beta, decay, kq, state, cu_seqlens, state_slots,
                                                     state_phase, o_raw, N, H, G, dv, s)
                             : launch_chunks<T, 64>(by_chunks, rows, qn, kn, beta, decay, kq, state, cu_seqlens, state_slots,
                                                    state_phase, o_raw, N, H, G, dv, s);
    if (rc != 0) return rc;
  }
  // A step with few (segment, head) pairs leaves most of the machine idle, and what a token takes is the length of its
  // chain of dependent operations: then a column gets more lanes with fewer rows each (the row's width stays).
  int ks = KS, rr = RR;
  while (rr > 4 && ks < 16 && (long long)R_ * H * ((dv + 64 / ks - 1) / (64 / ks)) < 1024) {  // (up to a row of 16 lanes)
    ks <<= 1;
    rr >>= 1;
  }
  const int cols_ = 64 / ks;
  const dim3 grid(R_, H, (dv + cols_ - 1) / cols_);
#define JLE_SCAN(KS_, RR_)                                                                                          \
  hipLaunchKernelGGL((gdr_scan_kernel<T, KS_, RR_>), grid, dim3(64), 0, s, rows, qn, kn, beta, decay, kq, state, cu_seqlens, \
                     state_slots, state_phase, o_raw, H, G, dk, dv, by_chunks.from)
#define JLE_SCAN_R(KS_)              \
  do {                               \
    if (rr == 4) JLE_SCAN(KS_, 4);   \
    else if (rr == 8) JLE_SCAN(KS_, 8); \
    else if (rr == 16) JLE_SCAN(KS_, 16); \
    else JLE_SCAN(KS_, 32);          \
  } while (0)
  if (by_chunks.others) switch (ks) {
    case 1: JLE_SCAN_R(1); break;
    case 2: JLE_SCAN_R(2); break;
    case 4: JLE_SCAN_R(4); break;
    case 8: JLE_SCAN_R(8); break;
    case 16: JLE_SCAN_R(16); break;
    case 32: JLE_SCAN_R(32); break;
    default: JLE_SCAN_R(64); break;
  }
#undef JLE_SCAN_R
#undef JLE_SCAN
  JLE_LAUNCH_CHECK();
  hipLaunchKernelGGL(gdr_out_kernel<T>, dim3(N, H), dim3(64), 0, s, o_raw, gate, norm_w, out, eps, H, dv);
  JLE_LAUNCH_CHECK();
  return 0;
}

}  // namespace

// The width of a unit vector's row in the scratch arrays: dk rounded up to lanes a column x rows a lane.
JLE_API int jle_gated_delta_padded(int dk) {
  if (dk <= 0 || dk > 2048) return -1;
  int KS = 1;
  while (KS < 64 && (dk + KS - 1) / KS > 16) KS <<= 1;
  const int per = (dk + KS - 1) / KS;
  return KS * (per <= 4 ? 4 : per <= 8 ? 8 : per <= 16 ? 16 : 32);
}

// The chunked form's scratch of one chunk of 64 tokens in KiB; -1: sizes that it is not compiled for.
JLE_API int jle_gated_delta_chunk_kib(int H, int G, int dk, int dv) {
  if ((dk != 64 && dk != 128) || dv <= 0 || dv % 16 || H <= 0 || G <= 0 || H % G || H > 65535) return -1;
  return (int)((chunk_floats(H, G, dk, dv) * sizeof(float) + 1023) / 1024);
}

// rows [N, 2 G dk + H dv] (q | k | v behind convolution and activation) and gate [N, H dv] in the run dtype; gates
// float32 [N, 2 H] (write strengths, then decays, before their biases and squashing); state float32 [slots, 2, H, dv,
// dk]; qn, kn [N, G, dkp] (dkp = jle_gated_delta_padded(dk), 16-byte aligned), beta, decay [N, H], o_raw [N, H, dv]
// and 64 floats behind it: float32 scratch; out [N, H dv] in the run dtype.
// Segments of `from` tokens and more go 64 tokens at a time (num_segs of them, their num_chunks chunks; sizes as
// jle_gated_delta_chunk_kib says; scratch of num_chunks times that many KiB, 16-byte aligned); others: whether shorter
// ones are left.  num_segs = 0: none does.
JLE_API int jle_gated_delta(const void* rows, int is_bf16, const float* gates, const float* a_log, const float* dt_bias,
                            const float* norm_w, const void* gate, float* state, const int* cu_seqlens,
                            const int* state_slots, const int* state_phase, float* qn, float* kn, float* beta,
                            float* decay, float* kq, float* o_raw, void* out, int N, int R, int H, int G, int dk, int dv,
                            float eps, float floor, const int* chunks, int num_chunks, const int* segs, int num_segs,
                            int from, int others, float* ws, hipStream_t s) {
  if (N <= 0) return 0;
  ByChunks b = {chunks, segs, num_chunks, num_segs, 0x7fffffff, 1, ws};
  if (num_segs > 0) {
    if ((dk != 64 && dk != 128) || dv % 16 || chunks == nullptr || segs == nullptr || ws == nullptr || from < 1 ||
        num_chunks < num_segs || num_segs > R || ((uintptr_t)ws | (uintptr_t)state) % 16 ||
        (long long)num_segs * H * (dv / 16) > (1ll << 31) - 1)
      return JLE_BAD_ARG;
    b.from = from;
    b.others = others;
  }
  const int dkp = jle_gated_delta_padded(dk);
  if (dkp <= 0 || ((uintptr_t)qn | (uintptr_t)kn) % 16) return JLE_BAD_ARG;
  if (R <= 0 || H <= 0 || G <= 0 || H % G || dk <= 0 || dk > 2048 || dv <= 0 || H > 65535 || G + 1 > 65535 ||
      rows == nullptr || gates == nullptr || state == nullptr || out == nullptr || gate == nullptr)
    return JLE_BAD_ARG;
  if (is_bf16)
    return launch_gdr<bf16_t>((const bf16_t*)rows, gates, a_log, dt_bias, norm_w, (const bf16_t*)gate, state, cu_seqlens,
                              state_slots, state_phase, qn, kn, beta, decay, kq, o_raw, (bf16_t*)out, N, R, H, G, dk, dv, dkp,
                              eps, floor, b, s);
  return launch_gdr<float>((const float*)rows, gates, a_log, dt_bias, norm_w, (const float*)gate, state, cu_seqlens,
                           state_slots, state_phase, qn, kn, beta, decay, kq, o_raw, (float*)out, N, R, H, G, dk, dv, dkp, eps,
                           floor, b, s);
}

// The sizes at which a step of single tokens is one launch.
JLE_API int jle_gated_delta_single_supported(int H, int G, int dk, int dv) {
  return (dk == 64 || dk == 128) && dv > 0 && dv <= 256 && H > 0 && G > 0 && H % G == 0 && H <= 65535;
}

// jle_gated_delta for a step whose every request has one token (token i is request i's): no scratch.
JLE_API int jle_gated_delta_single(const void* rows, int is_bf16, const float* gates, const float* a_log,
                                   const float* dt_bias, const float* norm_w, const void* gate, float* state,
                                   const int* state_slots, const int* state_phase, void* out, int R, int H, int G, int dk,
                                   int dv, float eps, float floor, hipStream_t s) {
  if (R <= 0) return 0;
  if (!jle_gated_delta_single_supported(H, G, dk, dv) || (uintptr_t)state % 16 || rows == nullptr || gates == nullptr ||
      state == nullptr || out == nullptr || gate == nullptr)
    return JLE_BAD_ARG;
  if (is_bf16)
    return launch_single<bf16_t>((const bf16_t*)rows, gates, a_log, dt_bias, norm_w, (const bf16_t*)gate, state, state_slots,
                                 state_phase, (bf16_t*)out, R, H, G, dk, dv, eps, floor, s);
  return launch_single<float>((const float*)rows, gates, a_log, dt_bias, norm_w, (const float*)gate, state, state_slots,
                              state_phase, (float*)out, R, H, G, dk, dv, eps, floor, s);
}
