// Kernels of the sandwich arrangement (a norm before and behind every branch, a sigmoid gate on the branch's
// output, a token shift before the mixer) and of the polynomial activation.
//
// add_norm_shift: per row
//     t  = (y + y_bias) * sigmoid(g + g_bias)                       the gated branch output (or a plain delta, or none)
//     x' = x + t / sqrt(mean(t^2) + eps_b) * w_b                    the residual sum, float32, into a NEW array
//     h  = x' / sqrt(mean(x'^2) + eps) * w                          the next branch's input
//     hs = h + (h_prev - h) * shift                                 h_prev: the float32 h of the token before
// h_prev of a segment's first row comes from the request's state (zeros at position 0); the h of a segment's last
// row goes into the state's other half.  With few rows a block forms its row and, if that is not a segment's first,
// the h of the row before anew (which is why the sum is not written in place).  With many rows that is twice the
// reading and two more reductions a row, so the first kernel leaves x' and 1 / sqrt(mean(x'^2) + eps) only, and
// shift_rows_kernel streams down the columns of x' with the last row's h in registers.  Every row's arithmetic is the
// same in both, so a token's result does not depend on how its request was cut into steps or batched.
#include "common.h"
#include "rows.h"

using namespace jle;

namespace {

constexpr int kThreads = 256;

template <typename T, int VEC>
__device__ __forceinline__ void load_piece(const T* p, float (&o)[VEC]) {
  if constexpr (VEC == 8 && sizeof(T) == 2) {
    typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
    const u32x4 r = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[2 * e] = __uint_as_float(r[e] << 16);
      o[2 * e + 1] = __uint_as_float(r[e] & 0xffff0000u);
    }
  } else if constexpr (VEC >= 4) {
#pragma unroll
    for (int e = 0; e < VEC; e += 4) {
      const f32x4_t r = load4<T>(p + e);
#pragma unroll
      for (int i = 0; i < 4; ++i) o[e + i] = r[i];
    }
  } else {
    o[0] = Num<T>::load(p);
  }
}
template <typename T, int VEC>
__device__ __forceinline__ void store_piece(T* p, const float (&o)[VEC]) {
  if constexpr (VEC == 8 && sizeof(T) == 2) {
    typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
    *reinterpret_cast<u32x4*>(p) = u32x4{pack_bf16(o[0], o[1]), pack_bf16(o[2], o[3]), pack_bf16(o[4], o[5]), pack_bf16(o[6], o[7])};
  } else if constexpr (VEC >= 4) {
#pragma unroll
    for (int e = 0; e < VEC; e += 4) store4<T>(p + e, f32x4_t{o[e], o[e + 1], o[e + 2], o[e + 3]});
  } else {
    Num<T>::store(p, o[0]);
  }
}
// a vector of weights, which may lie at any float (a slice of a longer vector: a load of four needs no more), or `fill`
// where there is none or the row has ended
template <int VEC>
__device__ __forceinline__ void load_weights(const float* p, int d, bool in, float fill, float (&o)[VEC]) {
  if (p != nullptr && in) {
    typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4_anywhere;
    if constexpr (VEC >= 4) {
#pragma unroll
      for (int e = 0; e < VEC; e += 4) {
        const f32x4_t r = *reinterpret_cast<const f32x4_anywhere*>(p + d + e);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[e + i] = r[i];
      }
    } else {
      o[0] = p[d];
    }
  } else {
#pragma unroll
    for (int e = 0; e < VEC; ++e) o[e] = fill;
  }
}

struct SandwichArgs {
  const float* x;        // [N, D]
  float* x_out;          // [N, D] or null (no delta: the residual stays as it is)
  int delta_kind;        // 0 none, 1 plain [N, D], 2 gated
  const void* y;         // [N, D]
  const float* y_bias;   // [D] or null
  const void* g;         // [N, D]
  const float* g_bias;   // [D] or null
  const float* post_w;   // [D] or null
  float post_eps;
  int do_norm;
  const float* w;        // [D] or null
  float eps;
  void* h_out;           // [N, D] or null
  const float* shift_w;  // [D] or null: no shift
  void* hs_out;          // [N, D]
  float* state;          // [slots, 2, D]
  const int* positions;
  const int* token_segment;
  const int* cu_seqlens;
  const int* state_slots;
  const int* state_phase;
  float* stats;          // [N] or null: 1 / sqrt(mean(x'^2) + eps) and no rows
  int N, D;
};

// A block takes one row.  Everything it reads - the row's three arrays, the weights, the state - is asked for before the
// first sum, where the registers allow it (a thread's 8 elements of rows of up to 8,192: as many threads as that takes):
// each of the chain's stages would otherwise begin with a trip to memory.  8 rows of 2,048: 6.0 us, with the weights loaded
// where they are used, an element at a time, 11.4; 2,048 rows of 4,096 without a shift 26 us (115 MB, 4.5 TB/s), before 36.
template <typename T, int THREADS, int CPT, int VEC>
__global__ __launch_bounds__(THREADS) void add_norm_shift_kernel(SandwichArgs a) {
  __shared__ float red[THREADS / 64];
  constexpr bool HOLD = CPT == 1;
  const int D = a.D;
  const int row = blockIdx.x;
  const bool shift = a.shift_w != nullptr;
  int first = 0, last = 0, slot = 0, phase = 0, pos = 0;
  if (shift) {
    const int seg = a.token_segment[row];
    first = a.cu_seqlens[seg];
    last = a.cu_seqlens[seg + 1] - 1;
    slot = a.state_slots[seg];
    phase = a.state_phase[seg];
    pos = a.positions[row];
  }
  float hprev[CPT][VEC];
  float wy[HOLD ? CPT : 1][VEC], wg[HOLD ? CPT : 1][VEC], wp[HOLD ? CPT : 1][VEC], wn[HOLD ? CPT : 1][VEC],
      ws[HOLD ? CPT : 1][VEC];
#pragma unroll
  for (int i = 0; i < CPT; ++i) {
    const int d = (threadIdx.x + THREADS * i) * VEC;
#pragma unroll
    for (int e = 0; e < VEC; ++e) hprev[i][e] = 0.f;
    if (shift && row == first && pos != 0 && d < D)
      load_piece<float, VEC>(a.state + ((size_t)slot * 2 + phase) * D + d, hprev[i]);
    if constexpr (HOLD) {
      load_weights<VEC>(a.y_bias, d, d < D, 0.f, wy[i]);
      load_weights<VEC>(a.g_bias, d, d < D, 0.f, wg[i]);
      load_weights<VEC>(a.post_w, d, d < D, 1.f, wp[i]);
      load_weights<VEC>(a.w, d, d < D, 1.f, wn[i]);
      load_weights<VEC>(a.shift_w, d, d < D, 0.f, ws[i]);
    }
  }
  // (with a shift: the row before first, if it is the same segment's)
  for (int r = shift && row > first ? row - 1 : row; r <= row; ++r) {
    const bool write = r == row;
    const size_t base = (size_t)r * D;
    float v[CPT][VEC], t[CPT][VEC], gg[CPT][VEC];
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int d = (threadIdx.x + THREADS * i) * VEC;
#pragma unroll
      for (int e = 0; e < VEC; ++e) v[i][e] = t[i][e] = gg[i][e] = 0.f;
      if (d < D) {
        load_piece<float, VEC>(a.x + base + d, v[i]);
        if (a.delta_kind != 0) load_piece<T, VEC>((const T*)a.y + base + d, t[i]);
        if (a.delta_kind == 2) load_piece<T, VEC>((const T*)a.g + base + d, gg[i]);
      }
    }
    if (a.delta_kind == 1) {
#pragma unroll
      for (int i = 0; i < CPT; ++i)
#pragma unroll
        for (int e = 0; e < VEC; ++e) v[i][e] += t[i][e];
    } else if (a.delta_kind == 2) {
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < CPT; ++i) {
        const int d = (threadIdx.x + THREADS * i) * VEC;
        if constexpr (!HOLD) {
          load_weights<VEC>(a.y_bias, d, d < D, 0.f, wy[0]);
          load_weights<VEC>(a.g_bias, d, d < D, 0.f, wg[0]);
        }
        if (d < D) {
#pragma unroll
          for (int e = 0; e < VEC; ++e) {
            const float yb = t[i][e] + wy[HOLD ? i : 0][e];
            const float gb = gg[i][e] + wg[HOLD ? i : 0][e];
            t[i][e] = yb * (1.0f / (1.0f + expf(-gb)));
            ss = __builtin_fmaf(t[i][e], t[i][e], ss);
          }
        }
      }
      const float tot = block_sum<THREADS>(ss, red);
      const float inv = 1.0f / sqrtf(tot / (float)D + a.post_eps);
#pragma unroll
      for (int i = 0; i < CPT; ++i) {
        const int d = (threadIdx.x + THREADS * i) * VEC;
        if constexpr (!HOLD) load_weights<VEC>(a.post_w, d, d < D, 1.f, wp[0]);
#pragma unroll
        for (int e = 0; e < VEC; ++e) v[i][e] += t[i][e] * inv * wp[HOLD ? i : 0][e];
      }
    }
    if (write && a.x_out != nullptr) {
#pragma unroll
      for (int i = 0; i < CPT; ++i) {
        const int d = (threadIdx.x + THREADS * i) * VEC;
        if (d < D) store_piece<float, VEC>(a.x_out + base + d, v[i]);
      }
    }
    if (!a.do_norm) continue;
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < CPT; ++i)
#pragma unroll
      for (int e = 0; e < VEC; ++e) ss = __builtin_fmaf(v[i][e], v[i][e], ss);
    const float tot = block_sum<THREADS>(ss, red);
    const float inv = 1.0f / sqrtf(tot / (float)D + a.eps);
    if (a.stats != nullptr) {
      if (threadIdx.x == 0) a.stats[r] = inv;
      continue;
    }
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int d = (threadIdx.x + THREADS * i) * VEC;
      if (d >= D) continue;
      if constexpr (!HOLD) load_weights<VEC>(a.w, d, true, 1.f, wn[0]);
      float h[VEC];
#pragma unroll
      for (int e = 0; e < VEC; ++e) h[e] = v[i][e] * inv * wn[HOLD ? i : 0][e];
      if (write) {
        if (a.h_out != nullptr) store_piece<T, VEC>((T*)a.h_out + base + d, h);
        if (shift) {
          if constexpr (!HOLD) load_weights<VEC>(a.shift_w, d, true, 0.f, ws[0]);
          float hs[VEC];
#pragma unroll
          for (int e = 0; e < VEC; ++e) hs[e] = h[e] + (hprev[i][e] - h[e]) * ws[HOLD ? i : 0][e];
          store_piece<T, VEC>((T*)a.hs_out + base + d, hs);
          if (r == last) store_piece<float, VEC>(a.state + ((size_t)slot * 2 + (1 - phase)) * D + d, h);
        }
      }
#pragma unroll
      for (int e = 0; e < VEC; ++e) hprev[i][e] = h[e];
    }
  }
}

// The rows from the sums and their statistics: a block takes kShiftRows rows of kThreads * VEC columns, all of whose
// values are asked for before the first is used.  Bound by its bytes (a row of 4,096: 16 KB read, 16 KB written): 2,048 rows
// of 4,096 16 us behind 26 for the sums and statistics, where blocks of four rows and the one before took 90.
constexpr int kShiftRows = 8;
template <typename T, int VEC>
__global__ __launch_bounds__(kThreads) void shift_rows_kernel(SandwichArgs a) {
  const int D = a.D, r0 = blockIdx.x * kShiftRows, r1 = min(a.N, r0 + kShiftRows);
  const int d = (blockIdx.y * kThreads + threadIdx.x) * VEC;
  if (d >= D) return;
  const float* x = a.x_out != nullptr ? a.x_out : a.x;
  float v[kShiftRows + 1][VEC], inv[kShiftRows + 1], w[VEC], sw[VEC], hprev[VEC];
#pragma unroll
  for (int j = 0; j <= kShiftRows; ++j) {  // (place 0: the row before the block's)
    const int r = max(0, min(r0 - 1 + j, r1 - 1));
    load_piece<float, VEC>(x + (size_t)r * D + d, v[j]);
    inv[j] = a.stats[r];
  }
  load_weights<VEC>(a.w, d, true, 1.f, w);
  load_weights<VEC>(a.shift_w, d, true, 0.f, sw);
#pragma unroll
  for (int e = 0; e < VEC; ++e) hprev[e] = v[0][e] * inv[0] * w[e];
#pragma unroll
  for (int j = 1; j <= kShiftRows; ++j) {
    const int r = r0 - 1 + j;
    if (r >= r1) break;
    const int seg = a.token_segment[r];
    if (r == a.cu_seqlens[seg]) {
      if (a.positions[r] == 0) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) hprev[e] = 0.f;
      } else {
        load_piece<float, VEC>(a.state + ((size_t)a.state_slots[seg] * 2 + a.state_phase[seg]) * D + d, hprev);
      }
    }
    float h[VEC], hs[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      h[e] = v[j][e] * inv[j] * w[e];
      hs[e] = h[e] + (hprev[e] - h[e]) * sw[e];
      hprev[e] = h[e];
    }
    if (a.h_out != nullptr) store_piece<T, VEC>((T*)a.h_out + (size_t)r * D + d, h);
    store_piece<T, VEC>((T*)a.hs_out + (size_t)r * D + d, hs);
    if (r == a.cu_seqlens[seg + 1] - 1)
      store_piece<float, VEC>(a.state + ((size_t)a.state_slots[seg] * 2 + (1 - a.state_phase[seg])) * D + d, h);
  }
}

template <typename T, int VEC>
int launch_sandwich(const SandwichArgs& args, hipStream_t s) {
  const int strips = (args.D + kThreads * VEC - 1) / (kThreads * VEC);
  SandwichArgs a = args;
  if (a.stats != nullptr) a.shift_w = nullptr;  // (the first kernel: sums and statistics)
  const dim3 g((unsigned)a.N);
  // (wider rows, up to 8,192: 2 x 4 elements a thread, or 8 or 16 single ones by fewer threads, which have the registers;
  // sums and shift of 2,048 rows of 6,148 in pieces of four 69 us, in single elements 198; of 1,026 by 256 threads 23, by
  // 1,024 that spill 96)
  constexpr int T1 = VEC == 1 ? 256 : 1024, C1 = 8 / VEC, T2 = VEC == 1 ? 512 : T1, C2 = VEC == 1 ? 16 : C1;
#define JLE_SANDWICH_CASE(TH, C) \
  else if (a.D <= TH * C * VEC) hipLaunchKernelGGL((add_norm_shift_kernel<T, TH, C, VEC>), g, dim3(TH), 0, s, a)
  // (narrow rows by as few wavefronts: 4,096 rows of 192 with a gated branch and the shift by one 8.8 us, by four 15.8)
  if (VEC < 8 && a.D <= 64 * VEC) hipLaunchKernelGGL((add_norm_shift_kernel<T, 64, 1, VEC < 8 ? VEC : 1>), g, dim3(64), 0, s, a);
  else if (VEC < 8 && a.D <= 128 * VEC) hipLaunchKernelGGL((add_norm_shift_kernel<T, 128, 1, VEC < 8 ? VEC : 1>), g, dim3(128), 0, s, a);
  JLE_SANDWICH_CASE(256, 1);
  JLE_SANDWICH_CASE(512, 1);
  JLE_SANDWICH_CASE(1024, 1);
  JLE_SANDWICH_CASE(T1, C1);
  JLE_SANDWICH_CASE(T2, C2);
  else return JLE_BAD_ARG;
#undef JLE_SANDWICH_CASE
  if (args.stats != nullptr)
    hipLaunchKernelGGL((shift_rows_kernel<T, VEC>), dim3((unsigned)((a.N + kShiftRows - 1) / kShiftRows), (unsigned)strips), dim3(kThreads),
                       0, s, args);
  return 0;
}

// ------------------------------------------------------------------ polynomial activation
// out = c0 N(u) + c1 N(u^2) + c2 N(u^3) + c3,  u = z + bias,  N(v) = v / sqrt(mean(v^2) + eps) over the row.
// PIECES > 0: the row (up to THREADS * VEC * PIECES wide) stays in registers between the sums and the polynomial;
// PIECES == 0: any width, the row is read twice.
template <typename T, int THREADS, int VEC, int PIECES>
__global__ __launch_bounds__(THREADS) void polynorm_kernel(const T* __restrict__ z, int ldz,
                                                            const float* __restrict__ bias,
                                                            const float* __restrict__ coef, float eps,
                                                            T* __restrict__ out, int F) {
  __shared__ float red[3][THREADS / 64];
  const size_t row = blockIdx.x;
  const float c0 = coef[0], c1 = coef[1], c2 = coef[2], c3 = coef[3];
  const T* zr = z + row * ldz;
  T* o = out + row * F;
  float s1 = 0.f, s2 = 0.f, s3 = 0.f;
  auto sums = [&](const float (&u)[VEC]) {
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const float u2 = u[e] * u[e], u3 = u2 * u[e];
      s1 = __builtin_fmaf(u[e], u[e], s1);
      s2 = __builtin_fmaf(u2, u2, s2);
      s3 = __builtin_fmaf(u3, u3, s3);
    }
  };
  auto fetch = [&](int d, float (&u)[VEC]) {
    load_piece<T, VEC>(zr + d, u);
    float b[VEC];
    load_weights<VEC>(bias, d, true, 0.f, b);
#pragma unroll
    for (int e = 0; e < VEC; ++e) u[e] += b[e];
  };
  constexpr int P = PIECES > 0 ? PIECES : 1;
  float kept[P][VEC];
  if constexpr (PIECES > 0) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int d = (threadIdx.x + THREADS * i) * VEC;
#pragma unroll
      for (int e = 0; e < VEC; ++e) kept[i][e] = 0.f;
      if (d < F) fetch(d, kept[i]);
    }
#pragma unroll
    for (int i = 0; i < PIECES; ++i) sums(kept[i]);  // (zeros beyond the row's end add nothing)
  } else {
    for (int d = threadIdx.x * VEC; d < F; d += THREADS * VEC) {
      float u[VEC];
      fetch(d, u);
      sums(u);
    }
  }
  // (the three sums together: one barrier instead of six)
  s1 = wave_sum(s1);
  s2 = wave_sum(s2);
  s3 = wave_sum(s3);
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = s1;
    red[1][threadIdx.x >> 6] = s2;
    red[2][threadIdx.x >> 6] = s3;
  }
  __syncthreads();
  float t[3] = {0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < THREADS / 64; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) t[j] += red[j][i];
  const float i1 = c0 / sqrtf(t[0] / (float)F + eps);
  const float i2 = c1 / sqrtf(t[1] / (float)F + eps);
  const float i3 = c2 / sqrtf(t[2] / (float)F + eps);
  auto poly = [&](const float (&u)[VEC], float (&v)[VEC]) {
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const float u2 = u[e] * u[e];
      v[e] = u[e] * i1 + u2 * i2 + u2 * u[e] * i3 + c3;
    }
  };
  if constexpr (PIECES > 0) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int d = (threadIdx.x + THREADS * i) * VEC;
      if (d < F) {
        float v[VEC];
        poly(kept[i], v);
        store_piece<T, VEC>(o + d, v);
      }
    }
  } else {
    for (int d = threadIdx.x * VEC; d < F; d += THREADS * VEC) {
      float u[VEC], v[VEC];
      fetch(d, u);
      poly(u, v);
      store_piece<T, VEC>(o + d, v);
    }
  }
}

template <typename T>
void launch_polynorm(const T* z, int ldz, const float* bias, const float* coef, float eps, T* out, int N, int F,
                     int vec, hipStream_t s) {
  // (which form runs depends on the width and on where the arrays lie, not on the step; 2,048 rows of 14,336 in 16-byte
  // pieces, the three sums behind one barrier: 34 us, 3.4 TB/s; in pieces of four with a barrier pair a sum 66; 8 rows of
  // 8,192 7.1 and 12.6; 2,048 rows of 14,340 in pieces of four 28, with the row read twice 32)
#define JLE_POLYNORM(TH, V, P) \
  hipLaunchKernelGGL((polynorm_kernel<T, TH, V, P>), dim3(N), dim3(TH), 0, s, z, ldz, bias, coef, eps, out, F)
  if (vec == 8 && F <= 256 * 8 * 2) JLE_POLYNORM(256, 8, 2);
  else if (vec == 8 && F <= 512 * 8 * 4) JLE_POLYNORM(512, 8, 4);
  else if (vec == 8) JLE_POLYNORM(256, 8, 0);
  else if (vec == 4 && F <= 256 * 4 * 4) JLE_POLYNORM(256, 4, 4);
  else if (vec == 4 && F <= 512 * 4 * 8) JLE_POLYNORM(512, 4, 8);
  else if (vec == 4) JLE_POLYNORM(256, 4, 0);
  else JLE_POLYNORM(256, 1, 0);
#undef JLE_POLYNORM
}

}  // namespace

// stats: null, or N floats of scratch: with a shift, the rows are formed by a second kernel (for many rows).
JLE_API int jle_add_norm_shift(const float* x, float* x_out, int delta_kind, const void* y, const float* y_bias,
                               const void* g, const float* g_bias, const float* post_w, float post_eps, int do_norm,
                               const float* w, float eps, void* h_out, const float* shift_w, void* hs_out,
                               float* state, const int* positions, const int* token_segment, const int* cu_seqlens,
                               const int* state_slots, const int* state_phase, int is_bf16, int N, int D, float* stats,
                               hipStream_t s) {
  if (N <= 0) return 0;
  if (D <= 0 || delta_kind < 0 || delta_kind > 2) return JLE_BAD_ARG;
  if (delta_kind != 0 && (y == nullptr || x_out == nullptr)) return JLE_BAD_ARG;
  if (delta_kind == 2 && g == nullptr) return JLE_BAD_ARG;
  if (shift_w != nullptr && (!do_norm || hs_out == nullptr || state == nullptr || positions == nullptr ||
                             token_segment == nullptr || cu_seqlens == nullptr || state_slots == nullptr ||
                             state_phase == nullptr))
    return JLE_BAD_ARG;
  if (stats != nullptr && shift_w == nullptr) return JLE_BAD_ARG;
  SandwichArgs a{x, x_out, delta_kind, y, y_bias, g, g_bias, post_w, post_eps, do_norm, w, eps, h_out, shift_w,
                 hs_out, state, positions, token_segment, cu_seqlens, state_slots, state_phase, stats, N, D};
  uintptr_t all = 0;
  for (const void* p : {(const void*)x, (const void*)x_out, y, g, (const void*)h_out, (const void*)hs_out, (const void*)state})
    all |= (uintptr_t)p;
  // (pieces of eight leave narrow rows too few threads: 2,048 rows of 1,024, gated branch and shift, 18.9 us, of four 15.0;
  // of float32 they are two loads: 256 rows of 2,048 8.3 and 7.6)
  const int vec = all % 16 ? 1 : D % 8 == 0 && D > (is_bf16 ? 1024 : 2048) ? 8 : D % 4 == 0 ? 4 : 1;
  int rc;
  if (is_bf16)
    rc = vec == 8 ? launch_sandwich<bf16_t, 8>(a, s) : vec == 4 ? launch_sandwich<bf16_t, 4>(a, s) : launch_sandwich<bf16_t, 1>(a, s);
  else
    rc = vec == 8 ? launch_sandwich<float, 8>(a, s) : vec == 4 ? launch_sandwich<float, 4>(a, s) : launch_sandwich<float, 1>(a, s);
  if (rc != 0) return rc;
  JLE_LAUNCH_CHECK();
  return 0;
}

JLE_API int jle_polynorm(const void* z, int ldz, const float* bias, const float* coef, float eps, void* out,
                         int is_bf16, int N, int F, hipStream_t s) {
  if (N <= 0) return 0;
  if (F <= 0 || ldz < F || coef == nullptr) return JLE_BAD_ARG;
  const bool aligned = ((uintptr_t)z | (uintptr_t)out) % 16 == 0;
  const int vec = !aligned ? 1 : F % 8 == 0 && ldz % 8 == 0 ? 8 : F % 4 == 0 && ldz % 4 == 0 ? 4 : 1;
  if (is_bf16)
    launch_polynorm<bf16_t>((const bf16_t*)z, ldz, bias, coef, eps, (bf16_t*)out, N, F, vec, s);
  else
    launch_polynorm<float>((const float*)z, ldz, bias, coef, eps, (float*)out, N, F, vec, s);
  JLE_LAUNCH_CHECK();
  return 0;
}
