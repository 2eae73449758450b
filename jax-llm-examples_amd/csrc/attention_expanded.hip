// Attention over a cached latent for steps of many tokens: every head's keys and values are formed from the latents once
// per step and attended to like any other keys and values,
//     k_j = [W_uk,h c_j, k_r_j]  (128 + 64 numbers),   v_j = W_uv,h c_j  (128),   softmax_j((q . k_j) * scale) v_j.
// A (query, key, head) then costs 640 operations instead of the 2,176 of the form that keeps to the latent's 512 numbers
// (attention_latent.hip); forming a key and a value costs 262,144 per head, once per step, which a few dozen queries a key
// pay for.  Three steps: expanded_gather_kernel brings the visible latents and shared key parts out of their pages, two
// library products form K [S, H * 128] and V^T [H * 128, S] (their rows and columns in the order of the gathered keys),
// expanded_attention_kernel attends.  S: every segment's keys from the first that any of its queries sees, that rounded
// down and their end rounded up to 64, so a step of 64 keys is 64 rows of K and whole 128-byte lines of V^T.
#include "mfma_attention.h"

using namespace jle;

namespace {

// One block per 16 gathered keys.  spans: per 64 of them (segment, first position, first position that is needed, end);
// a key that no query sees becomes a row of zeros, one whose page was given back a row of NaN (as its readers get).
__global__ __launch_bounds__(256) void expanded_gather_kernel(const bf16_t* __restrict__ latent,
                                                              const bf16_t* __restrict__ rope,
                                                              const int* __restrict__ block_table, int table_width,
                                                              const int4* __restrict__ spans, bf16_t* __restrict__ c_out,
                                                              bf16_t* __restrict__ kr_out, int R, int dr, int ps) {
  const int4 span = spans[blockIdx.x >> 2];
  const int row0 = blockIdx.x * 16, pos0 = span.y + (blockIdx.x & 3) * 16;
  const int* table = block_table + (size_t)span.x * table_width;
  const int cp = R / 8, per = cp + dr / 8;  // 16-byte pieces of a row
  for (int idx = threadIdx.x; idx < 16 * per; idx += 256) {
    const int row = idx / per, piece = idx - row * per;
    const int pos = pos0 + row;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (pos >= span.z && pos < span.w) {
      const int page = table[pos / ps];
      if (page < 0) {
        v = u32x4{0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u};
      } else {
        const size_t slot = (size_t)page * ps + pos % ps;
        v = piece < cp ? *reinterpret_cast<const u32x4*>(latent + slot * R + piece * 8)
                       : *reinterpret_cast<const u32x4*>(rope + slot * dr + (piece - cp) * 8);
      }
    }
    bf16_t* dst = piece < cp ? c_out + (size_t)(row0 + row) * R + piece * 8
                             : kr_out + (size_t)(row0 + row) * dr + (piece - cp) * 8;
    *reinterpret_cast<u32x4*>(dst) = v;
  }
}

constexpr int kDN = 128, kDR = 64, kDV = 128;
constexpr int kQC = (kDN + kDR) / 32, kNC = kDN / 32, kVT = kDV / 16;
// a step's 64 keys in shared memory: four tiles of 16 keys x 256 bytes (unrotated part), four of 16 x 128 (rotated part),
// the values as 128 rows (elements) of 64 keys
constexpr int kNopeTile = 16 * kDN * 2, kRopeTile = 16 * kDR * 2;
constexpr int kRopeAt = 4 * kNopeTile, kValueAt = kRopeAt + 4 * kRopeTile, kBuffer = kValueAt + kDV * 128;

// where piece p of row r of a rotated tile lies: p ^ rope_swizzle(r); eight neighbouring lanes read rows that differ in
// r % 4 and r / 8, and so eight different pieces of a 128-byte row
__device__ __forceinline__ int rope_swizzle(int r) { return (r & 3) | ((r >> 3) << 2); }

// The maxima, sums and probabilities of a step's 64 keys, and the values added up with them (see softmax64_and_values in
// attention_mfma.hip; keys and values outside a column's range are numbers here, never unwritten memory).
// masked: some key of the step lies outside some column's range (the same for the whole wavefront).
__device__ __forceinline__ void softmax_step(bool masked, f32x4 (&st)[2][4], int halves,
                                             const unsigned char* sv, uint32_t v_rd, int kb, const int (&lo)[2],
                                             const int (&hi)[2], float sc, float (&m)[2], float (&l)[2],
                                             f32x4 (&acc)[2][kVT]) {
  const int g = (threadIdx.x & 63) >> 4;
  bf16x8 pb[2][2];
  float corr[2];
  bool unchanged = true;
  if (masked) {
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = kb + 32 * (tt >> 1) + 8 * g + 4 * (tt & 1) + i;
          st[ct][tt][i] = key >= lo[ct] && key <= hi[ct] ? st[ct][tt][i] : -INFINITY;
        }
  }
#pragma unroll
  for (int ct = 0; ct < 2; ++ct) {
    float mx = -INFINITY;
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
      for (int i = 0; i < 4; ++i) mx = fmaxf(mx, st[ct][tt][i]);
    mx = column_max(mx);
    const float m_new = fmaxf(m[ct], mx * sc);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    corr[ct] = __builtin_amdgcn_exp2f(m[ct] - m_use);
    unchanged = unchanged && m_new == m[ct];
    float sum = 0.f;
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      float p[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        p[j] = __builtin_amdgcn_exp2f(fmaf(st[ct][2 * hf + (j >> 2)][j & 3], sc, -m_use));
        sum += p[j];
      }
      const u32x4 pk = {pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3]), pack_bf16(p[4], p[5]), pack_bf16(p[6], p[7])};
      pb[ct][hf] = __builtin_bit_cast(bf16x8, pk);
    }
    l[ct] = l[ct] * corr[ct] + sum;
    m[ct] = m_new;
  }
  if (!__all(unchanged)) {
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
      for (int dt = 0; dt < kVT; ++dt) acc[ct][dt] *= corr[ct];
  }
#pragma unroll
  for (int hf = 0; hf < 2; ++hf) {
    if (hf >= halves) break;
    bf16x8 va[kVT];
#pragma unroll
    for (int dt = 0; dt < kVT; ++dt) va[dt] = *reinterpret_cast<const bf16x8*>(sv + (v_rd ^ (hf * 64)) + dt * 2048);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int dt = 0; dt < kVT; ++dt)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct)
        acc[ct][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[dt], pb[ct][hf], acc[ct][dt], 0, 0, 0);
  }
}

// One token's outputs from the keys that it sees and no others, by a wavefront, with the maximum m and the factor inv that
// the steps have found.  In a step's product the values of keys outside a token's range meet zero probabilities, and zero
// times an infinity or NaN is NaN: a token whose outputs are not finite though its probabilities are takes this way.
// off: the gathered row of position 0.
__device__ __forceinline__ void attend_alone(const bf16_t* q, const bf16_t* kn, int kn_ld, const bf16_t* kr,
                                             const bf16_t* vt, int S, int off, int lo, int hi, float scale_log2, float m,
                                             float inv, bf16_t* out) {
  const int lane = threadIdx.x & 63;
  float o[2] = {0.f, 0.f};
  for (int kb = lo; kb <= hi; kb += 64) {
    const int count = min(64, hi - kb + 1);
    const size_t row = (size_t)(kb + min(lane, count - 1) + off);  // (behind the last key: that one again, unused)
    const bf16_t *a = kn + row * kn_ld, *b = kr + row * kDR;
    float s = 0.f;
    for (int e = 0; e < kDN; ++e) s = __builtin_fmaf(bf16_to_float(q[e]), bf16_to_float(a[e]), s);
    for (int e = 0; e < kDR; ++e) s = __builtin_fmaf(bf16_to_float(q[kDN + e]), bf16_to_float(b[e]), s);
    const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s, scale_log2, -m));
    const bf16_t* v = vt + (size_t)lane * S + (kb + off);
    for (int j = 0; j < count; ++j) {
      const float pj = __shfl(p, j, 64);
#pragma unroll
      for (int i = 0; i < 2; ++i) o[i] = __builtin_fmaf(pj, bf16_to_float(v[(size_t)(64 * i) * S + j]), o[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) out[lane + 64 * i] = float_to_bf16(o[i] * inv);
}

// A block takes up to 128 consecutive tokens of a segment and one head, a wavefront 32 of them; the keys in steps of 64
// absolute positions, which the load unit brings into one of two buffers in shared memory while the other is worked on
// (a wavefront a quarter of each of K, k_r and V^T), the score and value products transposed as in attention_mfma.hip.
// Two blocks fill a compute unit's 160 KB of shared memory; a step's 40 KB are read by all four wavefronts: one byte of
// shared memory for 32 operations, which is what bounds it beside the matrix cores.  One prompt of 2,048 tokens, 32 heads:
// 78 us (43 GFLOP, 0.55 PFLOP/s) and 46 for the gather and the two products, against 760 for the same attention over a
// latent of 512 (146 GFLOP) and 60 for its two products and their transposition.  One copy of the softmax for masked and
// unmasked steps: two copies kept the accumulators in two sets of registers and spilled 52 of them.
// blocks: (first token, tokens, gathered row of position 0, -) each; grid: blocks x heads, heads fastest (a head's keys
// and values stay in one chiplet's cache).
__global__ __launch_bounds__(256, 2) void expanded_attention_kernel(
    const bf16_t* __restrict__ q, int q_ld, const bf16_t* __restrict__ kn, const bf16_t* __restrict__ kr,
    const bf16_t* __restrict__ vt, int S, bf16_t* __restrict__ out, const int* __restrict__ positions,
    const int4* __restrict__ blocks, int window, float scale_log2, int H, const float* __restrict__ sink) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
  const int lane = threadIdx.x & 63, wave = wave_index();
  const int c16 = lane & 15, g = lane >> 4;
  const int h = blockIdx.x % H;
  const int4 blk = blocks[blockIdx.x / H];
  const int pos0 = positions[blk.x];
  const int k_lo = window > 0 ? max(0, pos0 - window + 1) : 0, k_hi = pos0 + blk.y - 1;
  const int nt = min(32, blk.y - 32 * wave);  // this wavefront's tokens
  const bool live = nt > 0;
  const int n0 = blk.x + (live ? 32 * wave : 0), p0 = pos0 + (live ? 32 * wave : 0);
  const int my_lo = window > 0 ? max(0, p0 - window + 1) : 0, my_hi = p0 + nt - 1;
  const int all_lo = window > 0 ? max(0, my_hi - window + 1) : 0, all_hi = p0;  // keys that every token sees

  bf16x8 qb[2][kQC];
  float m[2], l[2];
  int lo[2], hi[2];
  f32x4 acc[2][kVT];
#pragma unroll
  for (int ct = 0; ct < 2; ++ct) {
    const int c = ct * 16 + c16;
    const bool ok = c < nt;
    lo[ct] = ok ? (window > 0 ? max(0, p0 + c - window + 1) : 0) : 1;
    hi[ct] = ok ? p0 + c : 0;
    const bf16_t* row = q + (size_t)(n0 + (ok ? c : 0)) * q_ld + (size_t)h * (kDN + kDR) + g * 8;
#pragma unroll
    for (int c2 = 0; c2 < kQC; ++c2) {
      u32x4 v = {0u, 0u, 0u, 0u};
      if (ok) v = *reinterpret_cast<const u32x4*>(row + c2 * 32);
      qb[ct][c2] = __builtin_bit_cast(bf16x8, v);
    }
    m[ct] = -INFINITY;
    l[ct] = 0.f;
#pragma unroll
    for (int dt = 0; dt < kVT; ++dt) acc[ct][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // what this wavefront fetches of a step: byte offsets from its tile's first row, and from its first value element
  uint32_t n_src[4], r_src[2], v_src[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 4 * i + (lane >> 4);
    n_src[i] = (uint32_t)row * (uint32_t)(H * kDN * 2) + (uint32_t)(((lane & 15) ^ key_swizzle(row)) * 16);
    v_src[i] = (uint32_t)(8 * i + (lane >> 3)) * (uint32_t)(S * 2) + (uint32_t)(((lane & 7) ^ (lane >> 3)) * 16);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = 8 * i + (lane >> 3);
    r_src[i] = (uint32_t)(row * kDR * 2 + ((lane & 7) ^ rope_swizzle(row)) * 16);
  }
  // what it reads (rows dealt as in attention_prefill_lds_kernel: a lane's eight probabilities of a half are those of
  // keys 8 g .. 8 g + 7)
  // (tile t = 1 of a half: four rows further; the pieces of a row differ in address bits that the swizzle only flips)
  const int row = 8 * ((c16 >> 2) & 1) + (c16 & 3);
  const uint32_t n_rd = (uint32_t)((c16 >> 3) * kNopeTile + row * 256 + ((g ^ key_swizzle(row)) * 16));
  const uint32_t r_rd = (uint32_t)((c16 >> 3) * kRopeTile + row * 128 + ((g ^ rope_swizzle(row)) * 16));
  const uint32_t v_rd = (uint32_t)(c16 * 128 + ((g ^ (c16 & 7)) * 16));

  const int kb_first = k_lo / 64 * 64, kb_last = k_hi / 64 * 64;
  const bf16_t* v_base = vt + ((size_t)h * kDV + 32 * wave) * S;
  auto load_step = [&](int kb, int buf) {
    const size_t row = (size_t)(min(kb, kb_last) + blk.z);  // (behind the last step: that one again, never read)
    const bf16_t* n_at = kn + (row + 16 * wave) * (size_t)(H * kDN) + (size_t)h * kDN;
    const bf16_t* r_at = kr + (row + 16 * wave) * kDR;
    const uint32_t dst = lds0 + (uint32_t)(buf * kBuffer);
#pragma unroll
    for (int i = 0; i < 4; ++i) load_to_lds16(n_at, n_src[i], dst + (uint32_t)(wave * kNopeTile + i * 1024));
#pragma unroll
    for (int i = 0; i < 2; ++i) load_to_lds16(r_at, r_src[i], dst + (uint32_t)(kRopeAt + wave * kRopeTile + i * 1024));
#pragma unroll
    for (int i = 0; i < 4; ++i) load_to_lds16(v_base + row, v_src[i], dst + (uint32_t)(kValueAt + wave * 4096 + i * 1024));
  };

  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the queries have come; from here on only the steps' loads count
  asm volatile("" ::: "memory");
  load_step(kb_first, 0);
  int buf = 0;
  for (int kb = kb_first; kb <= kb_last; kb += 64) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this step's loads have landed
    __syncthreads();
    load_step(kb + 64, buf ^ 1);  // the next step, into the buffer that every wavefront has just left
    if (live && kb + 63 >= my_lo && kb <= my_hi) {
      const unsigned char* sb = smem + buf * kBuffer;
      const int halves = kb + 32 <= my_hi ? 2 : 1;
      f32x4 st[2][4];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) st[ct][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        if (hf >= halves) break;
#pragma unroll
        for (int t = 0; t < 2; ++t) {  // (a tile's six pieces asked for at once; both tiles' twelve do not fit the registers)
          bf16x8 kt[kQC];
#pragma unroll
          for (int c = 0; c < kNC; ++c) kt[c] = *reinterpret_cast<const bf16x8*>(sb + (n_rd ^ ((t * 1152) ^ (c * 64))) + hf * (2 * kNopeTile));
#pragma unroll
          for (int c = kNC; c < kQC; ++c) kt[c] = *reinterpret_cast<const bf16x8*>(sb + kRopeAt + (r_rd ^ ((c - kNC) * 64)) + t * 512 + hf * (2 * kRopeTile));
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int c = 0; c < kQC; ++c)
#pragma unroll
            for (int ct = 0; ct < 2; ++ct)
              st[ct][2 * hf + t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kt[c], qb[ct][c], st[ct][2 * hf + t], 0, 0, 0);
        }
      }
      softmax_step(kb < all_lo || kb + 63 > all_hi, st, halves, sb + kValueAt, v_rd, kb, lo, hi, scale_log2, m, l, acc);
    }
    buf ^= 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may land in shared memory after the block has gone
  if (!live) return;
#pragma unroll
  for (int ct = 0; ct < 2; ++ct) {
    const int c = ct * 16 + c16;
    float sum = column_sum(l[ct]);
    if (sink != nullptr) sum += exp2f(sink[h] * kLog2e - m[ct]);
    const float inv = 1.0f / sum;
    bool odd = false;
#pragma unroll
    for (int dt = 0; dt < kVT; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) odd |= !(fabsf(acc[ct][dt][i]) <= 3.402823466e38f);
    // (a sum that is not finite is so because of a key that the token sees)
    unsigned long long again = __ballot(odd && fabsf(sum) <= 3.402823466e38f && c < nt);
    again |= again >> 32;
    again |= again >> 16;
    again &= 0xffff;
    if (c < nt && !(again >> c16 & 1)) {
      bf16_t* o = out + ((size_t)(n0 + c) * H + h) * kDV + 4 * g;
#pragma unroll
      for (int dt = 0; dt < kVT; ++dt) {
        const u32x2 v = {pack_bf16(acc[ct][dt][0] * inv, acc[ct][dt][1] * inv),
                         pack_bf16(acc[ct][dt][2] * inv, acc[ct][dt][3] * inv)};
        *reinterpret_cast<u32x2*>(o + dt * 16) = v;
      }
    }
    for (; again != 0; again &= again - 1) {
      const int of = __ffsll((long long)again) - 1, n = n0 + ct * 16 + of;
      attend_alone(q + (size_t)n * q_ld + (size_t)h * (kDN + kDR), kn + (size_t)h * kDN, H * kDN, kr,
                   vt + (size_t)h * kDV * S, S, blk.z, __shfl(lo[ct], of, 64), __shfl(hi[ct], of, 64), scale_log2,
                   __shfl(m[ct], of, 64), __shfl(inv, of, 64), out + ((size_t)n * H + h) * kDV);
    }
  }
}

}  // namespace

// The sizes that the expanded form is compiled for (bfloat16 only).
JLE_API int jle_latent_expanded_supported(int R, int dn, int dr, int dv, int q_ld) {
  return dn == kDN && dr == kDR && dv == kDV && R > 0 && R % 8 == 0 && q_ld % 8 == 0;
}

// c_out [S, R] and kr_out [S, dr], S = 64 * num_spans; spans as the kernel says (four ints each, 16-byte aligned).
JLE_API int jle_latent_expanded_gather(const void* latent_pages, const void* rope_pages, const int* block_table,
                                       int table_width, const int* spans, int num_spans, void* c_out, void* kr_out, int R,
                                       int dr, int ps, hipStream_t s) {
  if (num_spans <= 0) return 0;
  if (R <= 0 || R % 8 || dr <= 0 || dr % 8 || ps <= 0 || table_width <= 0 || num_spans > (1 << 24) ||
      ((uintptr_t)latent_pages | (uintptr_t)rope_pages | (uintptr_t)spans | (uintptr_t)c_out | (uintptr_t)kr_out) % 16)
    return JLE_BAD_ARG;
  hipLaunchKernelGGL(expanded_gather_kernel, dim3((unsigned)num_spans * 4), dim3(256), 0, s, (const bf16_t*)latent_pages,
                     (const bf16_t*)rope_pages, block_table, table_width, (const int4*)spans, (bf16_t*)c_out,
                     (bf16_t*)kr_out, R, dr, ps);
  JLE_LAUNCH_CHECK();
  return 0;
}

// q: rows of q_ld numbers that begin with the heads' [128 unrotated | 64 rotated]; kn [S, H * 128], kr [S, 64], vt
// [H * 128, S], out [N, H * 128]; blocks as the kernel says.
JLE_API int jle_latent_expanded_attention(const void* q, int q_ld, const void* kn, const void* kr, const void* vt, int S,
                                          void* out, const int* positions, const int* blocks, int num_blocks, int window,
                                          float scale, int H, const float* sink, hipStream_t s) {
  if (num_blocks <= 0) return 0;
  if (H <= 0 || q_ld < H * (kDN + kDR) || q_ld % 8 || S <= 0 || S % 64 || window < 0 || !(scale > 0.f) ||
      (long long)num_blocks * H > (1ll << 31) - 1 || (long long)S * 64 > (1ll << 31) - 1 || H > (1 << 16) ||
      ((uintptr_t)q | (uintptr_t)kn | (uintptr_t)kr | (uintptr_t)vt | (uintptr_t)out | (uintptr_t)blocks) % 16)
    return JLE_BAD_ARG;
  constexpr int smem = 2 * kBuffer;
  if (const int rc = allow_lds(expanded_attention_kernel, smem)) return rc;
  hipLaunchKernelGGL(expanded_attention_kernel, dim3((unsigned)(num_blocks * H)), dim3(256), smem, s, (const bf16_t*)q, q_ld,
                     (const bf16_t*)kn, (const bf16_t*)kr, (const bf16_t*)vt, S, (bf16_t*)out, positions,
                     (const int4*)blocks, window, scale * kLog2e, H, sink);
  JLE_LAUNCH_CHECK();
  return 0;
}
