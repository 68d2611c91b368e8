// gfx950 decode attention: one new query token per sequence against a KV cache,
// for KV-cached generation (the reference's TradingModel.generate,
// src/mega_trading/model.py:134-147, recomputes the whole context per token
// instead; the maths is the causal GQA attention of triton_attention.py for the
// last query row, whose keys are all cached positions).
//
// Split-K ("flash decoding"): a wave takes 64 cached keys of one (batch, KV
// head) for all R query heads of the group, so each K/V row is read once; the
// 4 or 8 waves of a workgroup merge their (o, m, l) in LDS, and a second kernel
// merges the workgroups with the log-sum-exp rule (none when one workgroup
// covers the cache).
//
// What bounds it: a long cache streams from HBM once, a short one is a chain of
// dependent steps (at the decoder's shapes a wave's data is a few KB).  Both ask
// for every K and V load of a wave to be issued at entry in as few cache lines
// as possible, and for few instructions after it:
//  * K comes in the A-operand layout of v_mfma_f32_16x16x32 (16 rows x 64
//    adjacent bytes per load), and K q for the group's heads (the B columns) is
//    one MFMA per 16 keys x 32 d: exact 16-bit products, fp32 sums.
//  * V comes a 16-byte chunk per lane (whole rows per load); p V is fp32 FMAs,
//    so the probabilities stay fp32.
//  * the reductions stay inside the wave (DPP within 16-lane rows, permlane
//    swaps across rows); one LDS exchange hands the probabilities from the score
//    layout to the V layout.
// Before, a wave read K a row per lane (64 cache lines a load), formed q . k on
// the vector ALUs, reduced every o value by itself and wrote a partial per 64
// keys.  Measured (bf16, attention + merge, us): 16 sequences of 6001 keys, 32 / 8
// heads of 128: 89.3 -> 79.7 (split 76.4 -> 67.5 = 5.8 TB/s, merge 11.3 -> 4.9);
// 32 of 545, 8 / 2 heads of 64: 8.2 -> 7.8; 32 of 512: 8.6 -> 6.2; 60 of 2000,
// 16 / 2 heads of 32: 20.4 -> 12.7.
//
// A launch with RoPE tables (mt_gqa_attn_decode_append) also rotates the new
// token's q and k and appends k and v: the wave that owns the new position takes
// that row from registers, so nothing waits for the cache write.  In a recorded
// token of the 8-layer decoder (32 sequences, 601 keys) rotation, attention and
// merge took 2.9 + 8.5 + 3.7 us a layer, now 10.9 in one launch.
#pragma once

#include "mt_common.h"

namespace mt {

constexpr int kDecSplit = 64;   // keys per wave
constexpr int kDecMaxR = 8;     // query heads per KV head supported
constexpr int kDecMinWaves = 4; // waves of a workgroup: 4, 8 or (D <= 64) 16

// fp32 floats per partial: o[0..D), m (log2), l, two pad floats (16-byte rows)
template <int D>
constexpr int dec_row() { return D + 4; }

struct DecodeParams {
  const uint16_t* q;  // [B, Hq, 1, D] (rotated when RoPE is used)
  const uint16_t* k;  // [B, Hkv, >= L, D] cache (rotated keys)
  const uint16_t* v;  // [B, Hkv, >= L, D] cache
  uint16_t* out;      // [B, Hq, 1, D]
  float* part;        // [B, Hq, nspan, D + 4] fp32: o (unnormalised), m (log2), l
  int64_t sq[2], sk[3], sv[3], so[2];  // strides (b, h) for q / o, (b, h, t) for the caches
  const int* length_dev;  // when set, L is read from device memory (graph-replayable decode)
  int B, Hq, Hkv, R, L, nspan;  // nspan: workgroups per (batch, KV head) (of the capacity when length_dev is set)
  int span;                     // keys per workgroup
  float scale_log2;  // softmax scale * log2(e)
  // With RoPE tables (cos set) q is not read: the launch takes the new token's
  // unrotated q, k and v, rotates q and k, and appends k and v to the caches.
  const void* xq;  // [B, Hq, D], xk, xv [B, Hkv, D]: the cache's type, or fp32 (in_fp32)
  const void* xk;
  const void* xv;
  int64_t sxq[2], sxk[2], sxv[2];  // strides (b, h)
  const float* cos;    // [>= pos + 1, D/2]
  const float* sin;
  const int* pos_dev;  // when set, the position is read from device memory, clamped to [0, pos]
  int pos, in_fp32;
  uint16_t* kc;        // the caches k and v, written at pos
  uint16_t* vc;
};

// 8 consecutive values of a new token's row at element offset i, rounded to the cache's type
template <class E>
__device__ __forceinline__ u32x4 dec_new8(const void* base, int64_t i, int in_fp32) {
  if (!in_fp32) return *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(base) + i);
  const f32x4* f = reinterpret_cast<const f32x4*>(static_cast<const float*>(base) + i);
  const f32x4 a = f[0], b = f[1];
  return u32x4{pack2<E>(a[0], a[1]), pack2<E>(a[2], a[3]), pack2<E>(b[0], b[1]), pack2<E>(b[2], b[3])};
}

// With length_dev, L holds the capacity and the device value is clamped to [1, capacity].
__device__ __forceinline__ int decode_length(const DecodeParams& p) {
  return p.length_dev ? min(max(*p.length_dev, 1), p.L) : p.L;
}

__device__ __forceinline__ f32x4 mfma_16x16x32(BF16, u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma_16x16x32(FP16, u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Layouts.  Score pass: the 64 keys as 4 tiles of 16; A operand lane l = key
// l % 16 of the tile, d chunk l / 16 of each 32; result lane l = head l % 16,
// keys 4 (l / 16) + i.  V pass: lane = (d chunk c = l % NC, key group l / NC),
// keys l / NC + i G.  Keys past the wave's end load its last key instead (in
// bounds; their probabilities are zero), so the loads need no branches.
template <int D>
struct DecLayout {
  static constexpr int KS = D / 32;         // 32-d steps of a score
  static constexpr int NC = D / 8;          // 16-byte chunks per row
  static constexpr int G = 64 / NC;         // key groups of the V pass
  static constexpr int NV = kDecSplit / G;  // V chunks per lane
  static constexpr int LO = NC == 4 ? 2 : NC == 8 ? 3 : 4;  // log2(NC): lane bits of the d chunk
};

// R (query heads of the KV group) is a template parameter: the per-head loops
// then unroll into straight-line code whose LDS reads issue back to back.
template <class E, int D, int R, int NW>
__global__ __launch_bounds__(64 * NW) void attn_decode_kernel(DecodeParams p) {
  static_assert(D == 32 || D == 64 || D == 128, "head size");
  static_assert(R >= 1 && R <= kDecMaxR, "group size");
  using Ly = DecLayout<D>;
  // a wave's block: its probabilities [R][64], then, once its V pass has read
  // them, its unnormalised o [R][D]
  __shared__ __attribute__((aligned(16))) float buf[NW][R * (D > kDecSplit ? D : kDecSplit)];
  __shared__ __attribute__((aligned(16))) float wm[R][NW], wl[R][NW];  // the waves' m and l
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int s = blockIdx.x % p.nspan;
  const int g = blockIdx.x / p.nspan;
  const int kvh = g % p.Hkv;
  const int b = g / p.Hkv;
  const int L = decode_length(p);
  const int k0 = s * (NW * kDecSplit) + wave * kDecSplit;
  const int n = min(kDecSplit, L - k0);
  const int hn = lane & 15, quad = lane >> 4;
  const int c8 = lane % Ly::NC, kg = lane / Ly::NC;
  // the new token's row of the cache, when this wave's keys hold its position;
  // it is written here and, for the wave's own scores, taken from registers
  const int pos = p.cos ? (p.pos_dev ? min(max(*p.pos_dev, 0), p.pos) : p.pos) : -1;
  const bool owner = pos >= k0 && pos < k0 + kDecSplit;  // wave-uniform
  u32x4 knew[Ly::KS], vnew;
  if (owner) {
    const int64_t xk = b * p.sxk[0] + (int64_t)kvh * p.sxk[1] + 8 * quad;
    const float* cs = p.cos + (int64_t)pos * (D / 2) + 4 * quad;
    const float* sn = p.sin + (int64_t)pos * (D / 2) + 4 * quad;
    uint16_t* kr = p.kc + b * p.sk[0] + (int64_t)kvh * p.sk[1] + (int64_t)pos * p.sk[2] + 8 * quad;
#pragma unroll
    for (int c = 0; c < Ly::KS; ++c) {
      knew[c] = rope_chunk<E>(dec_new8<E>(p.xk, xk + 32 * c, p.in_fp32), *reinterpret_cast<const f32x4*>(cs + 16 * c),
                              *reinterpret_cast<const f32x4*>(sn + 16 * c));
      if (hn == 0) *reinterpret_cast<u32x4*>(kr + 32 * c) = knew[c];
    }
    vnew = dec_new8<E>(p.xv, b * p.sxv[0] + (int64_t)kvh * p.sxv[1] + 8 * c8, p.in_fp32);
    if (kg == 0)
      *reinterpret_cast<u32x4*>(p.vc + b * p.sv[0] + (int64_t)kvh * p.sv[1] + (int64_t)pos * p.sv[2] + 8 * c8) = vnew;
  }
  if (s * (NW * kDecSplit) >= L) return;  // past the current length (device-length launches cover the capacity)
  if (n > 0) {  // wave-uniform
    u32x4 kw[4][Ly::KS], vw[Ly::NV], qf[Ly::KS];
    const uint16_t* kb = p.k + b * p.sk[0] + (int64_t)kvh * p.sk[1] + (int64_t)k0 * p.sk[2] + 8 * quad;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int c = 0; c < Ly::KS; ++c)
        kw[t][c] = *reinterpret_cast<const u32x4*>(kb + (int64_t)min(16 * t + hn, n - 1) * p.sk[2] + 32 * c);
    const uint16_t* vb = p.v + b * p.sv[0] + (int64_t)kvh * p.sv[1] + (int64_t)k0 * p.sv[2] + 8 * c8;
#pragma unroll
    for (int i = 0; i < Ly::NV; ++i)
      vw[i] = *reinterpret_cast<const u32x4*>(vb + (int64_t)min(kg + i * Ly::G, n - 1) * p.sv[2]);
    const int qh = kvh * R + min(hn, R - 1);
    if (p.cos) {
      const int64_t xq = b * p.sxq[0] + (int64_t)qh * p.sxq[1] + 8 * quad;
      const float* cs = p.cos + (int64_t)pos * (D / 2) + 4 * quad;
      const float* sn = p.sin + (int64_t)pos * (D / 2) + 4 * quad;
#pragma unroll
      for (int c = 0; c < Ly::KS; ++c)
        qf[c] = rope_chunk<E>(dec_new8<E>(p.xq, xq + 32 * c, p.in_fp32), *reinterpret_cast<const f32x4*>(cs + 16 * c),
                              *reinterpret_cast<const f32x4*>(sn + 16 * c));
    } else {
      const uint16_t* qb = p.q + b * p.sq[0] + (int64_t)qh * p.sq[1] + 8 * quad;
#pragma unroll
      for (int c = 0; c < Ly::KS; ++c) qf[c] = *reinterpret_cast<const u32x4*>(qb + 32 * c);
    }
    if (owner) {  // every load of the new row, also those of keys past the end: the cache may still hold the old one
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int c = 0; c < Ly::KS; ++c) kw[t][c] = min(16 * t + hn, n - 1) == pos - k0 ? knew[c] : kw[t][c];
#pragma unroll
      for (int i = 0; i < Ly::NV; ++i) vw[i] = min(kg + i * Ly::G, n - 1) == pos - k0 ? vnew : vw[i];
    }
    f32x4 sc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      sc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < Ly::KS; ++c) sc[t] = mfma_16x16x32(E{}, kw[t][c], qf[c], sc[t]);
    }
    // the wave's softmax offset m and sum l of head hn (log2 units)
    float m = -INFINITY;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sc[t][i] = 16 * t + 4 * quad + i < n ? sc[t][i] * p.scale_log2 : -INFINITY;
        m = fmaxf(m, sc[t][i]);
      }
    m = wave_reduce<4, true>(m);
    float l = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sc[t][i] = 16 * t + 4 * quad + i < n ? exp2_fast(sc[t][i] - m) : 0.f;
        l += sc[t][i];
      }
      if (hn < R) *reinterpret_cast<f32x4*>(&buf[wave][hn * kDecSplit + 16 * t + 4 * quad]) = sc[t];
    }
    l = wave_reduce<4, false>(l);
    if (lane < R) {
      wm[lane][wave] = m;
      wl[lane][wave] = l;
    }
    // LDS operations of one wave complete in order: a wave-scope fence (a
    // compiler barrier) suffices between the writes and the reads
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float acc[R][8];
#pragma unroll
    for (int h = 0; h < R; ++h)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[h][e] = 0.f;
#pragma unroll
    for (int i = 0; i < Ly::NV; ++i) {
      const int j = kg + i * Ly::G;
      float vv[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        vv[2 * e] = lo_f<E>(vw[i][e]);
        vv[2 * e + 1] = hi_f<E>(vw[i][e]);
      }
#pragma unroll
      for (int h = 0; h < R; ++h) {
        const float pj = buf[wave][h * kDecSplit + j];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[h][e] = __builtin_fmaf(pj, vv[e], acc[h][e]);
      }
    }
    // the sums over the key groups.  Lane bits 5 and 4 halve the values as they
    // add (a permlane swap of two values leaves the lower half of the wave the
    // two halves of one, the upper half those of the other), so that lane quarter
    // `quad` ends with the flat values [2 R quad, 2 R (quad + 1)) of acc[h][e] at
    // 8 h + e: two instructions a pair instead of a full reduction of each value.
    float r1[4 * R], r2[2 * R];
#pragma unroll
    for (int f = 0; f < 4 * R; ++f) {
      const int f2 = f + 4 * R;
      const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[f / 8][f % 8]),
                                                      __float_as_uint(acc[f2 / 8][f2 % 8]), false, false);
      r1[f] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
    }
#pragma unroll
    for (int f = 0; f < 2 * R; ++f) {
      const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(r1[f]), __float_as_uint(r1[f + 2 * R]), false, false);
      float y = __uint_as_float(x[0]) + __uint_as_float(x[1]);
      if constexpr (Ly::LO <= 2) y += dpp_mov<0x124>(y);  // row_ror:4
      if constexpr (Ly::LO <= 3) y += dpp_mov<0x128>(y);  // row_ror:8
      r2[f] = y;
    }
    // in order behind the wave's own reads of the probabilities
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (hn < Ly::NC) {
#pragma unroll
      for (int f = 0; f < 2 * R; f += 2) {
        const int i = 2 * R * quad + f;
        *reinterpret_cast<f32x2*>(&buf[wave][(i >> 3) * D + 8 * c8 + (i & 7)]) = f32x2{r2[f], r2[f + 1]};
      }
    }
  }
  __syncthreads();
  // merge the waves that held keys (0 .. na - 1, na >= 1):
  // M = max m_w, o = sum_w 2^(m_w - M) o_w, l = sum_w 2^(m_w - M) l_w
  const int na = min(NW, (L - s * (NW * kDecSplit) + kDecSplit - 1) / kDecSplit);
  for (int i = tid; i < R * D; i += 64 * NW) {
    const int h = i / D, d = i % D;
    float mw[NW], M = -INFINITY, o = 0.f, lt = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      mw[w] = w < na ? wm[h][w] : -INFINITY;
      M = fmaxf(M, mw[w]);
    }
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float a = exp2_fast(mw[w] - M);
      o = __builtin_fmaf(a, w < na ? buf[w][h * D + d] : 0.f, o);
      lt = __builtin_fmaf(a, w < na ? wl[h][w] : 0.f, lt);
    }
    if (p.nspan == 1) {
      p.out[b * p.so[0] + (int64_t)(kvh * R + h) * p.so[1] + d] = uint16_t(pack2<E>(o / lt, 0.f) & 0xffffu);
    } else {
      float* dst = p.part + (((int64_t)b * p.Hq + kvh * R + h) * p.nspan + s) * dec_row<D>();
      dst[d] = o;
      if (d == 0) *reinterpret_cast<f32x2*>(dst + D) = f32x2{M, lt};
    }
  }
}

// Merge the workgroups' partials ("splits") of each (batch, query head): M = max m_s,
// O = sum_s 2^(m_s - M) o_s / sum_s 2^(m_s - M) l_s.  One thread per d value;
// the splits are read 16 at a time with every load of a batch issued before
// its first use (one memory round trip per 16 splits).
template <class E, int D>
__global__ __launch_bounds__(256) void attn_decode_combine_kernel(DecodeParams p) {
  constexpr int PER = 256 / D;  // (batch, head) pairs per workgroup
  constexpr int ROW = dec_row<D>();
  constexpr int BATCH = 16;
  const int pair = blockIdx.x * PER + threadIdx.x / D;
  const int d = threadIdx.x % D;
  if (pair >= p.B * p.Hq) return;
  const int b = pair / p.Hq, h = pair % p.Hq;
  const float* src = p.part + (int64_t)pair * p.nspan * ROW;
  const int ns = (decode_length(p) + p.span - 1) / p.span;  // workgroups that held keys
  float M = -INFINITY, o = 0.f, l = 0.f;
  for (int s0 = 0; s0 < ns; s0 += BATCH) {
    float ms[BATCH], os[BATCH], ls[BATCH];
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      const bool in = s0 + i < ns;
      const float* r = src + (int64_t)(in ? s0 + i : 0) * ROW;
      const f32x2 ml = *reinterpret_cast<const f32x2*>(r + D);
      ms[i] = in ? ml[0] : -INFINITY;
      ls[i] = in ? ml[1] : 0.f;
      os[i] = in ? r[d] : 0.f;
    }
    float mn = M;
#pragma unroll
    for (int i = 0; i < BATCH; ++i) mn = fmaxf(mn, ms[i]);
    const float a = exp2_fast(M - mn);  // 0 on the first batch (M = -inf)
    o *= a;
    l *= a;
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      const float w = exp2_fast(ms[i] - mn);
      o = __builtin_fmaf(w, os[i], o);
      l = __builtin_fmaf(w, ls[i], l);
    }
    M = mn;
  }
  const float r = o / l;
  p.out[b * p.so[0] + (int64_t)h * p.so[1] + d] = uint16_t(pack2<E>(r, 0.f) & 0xffffu);
}

// ---------------------------------------------------------------------------
// The new token's RoPE and cache append, in one launch: q_rot = rot(q) (written
// [B, Hq, 1, D]), k_cache[:, :, pos] = rot(k), v_cache[:, :, pos] = v.  The
// inputs (views of the projections, [B, H, D] with strides (b, h), d stride 1)
// are first rounded to the cache's 16-bit type, then rotated in fp32 with the
// fp32 tables row `pos` and rounded again -- the sequence the fused forward
// kernels apply to the prompt, so cached and recomputed keys are identical.
// One thread per interleaved pair (x[2i], x[2i+1]).
// ---------------------------------------------------------------------------
struct RopeAppendParams {
  const void* q;
  const void* k;
  const void* v;
  int64_t sq[2], sk[2], sv[2];
  const float* cos;  // [>= pos + 1, D/2]
  const float* sin;
  uint16_t* q_out;   // [B, Hq, 1, D] contiguous
  uint16_t* kc;      // [B, Hkv, cap, D] with strides (b, h, t)
  uint16_t* vc;
  int64_t skc[3], svc[3];
  const int* pos_dev;  // when set, the position is read from device memory, clamped to [0, pos]
  int B, Hq, Hkv, D, pos;
};

template <class E, int XT>
__device__ __forceinline__ float load_in(const void* base, int64_t i) {
  if constexpr (XT == 2) return E::to_f(uint16_t(pack2<E>(static_cast<const float*>(base)[i], 0.f) & 0xffffu));
  else return E::to_f(static_cast<const uint16_t*>(base)[i]);
}

template <class E, int XT>
__global__ __launch_bounds__(256) void decode_rope_append_kernel(RopeAppendParams p) {
  const int half = p.D / 2;
  const int pos = p.pos_dev ? min(max(*p.pos_dev, 0), p.pos) : p.pos;
  const int64_t nq = (int64_t)p.B * p.Hq * half, nk = (int64_t)p.B * p.Hkv * half;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= nq + 2 * nk) return;
  if (i < nq + nk) {
    const bool isq = i < nq;
    const int64_t j = isq ? i : i - nq;
    const int H = isq ? p.Hq : p.Hkv;
    const int pr = int(j % half);
    const int h = int((j / half) % H);
    const int b = int(j / half / H);
    const void* src = isq ? p.q : p.k;
    const int64_t off = b * (isq ? p.sq[0] : p.sk[0]) + (int64_t)h * (isq ? p.sq[1] : p.sk[1]) + 2 * pr;
    const float x0 = load_in<E, XT>(src, off), x1 = load_in<E, XT>(src, off + 1);
    const float c = p.cos[(int64_t)pos * half + pr], sn = p.sin[(int64_t)pos * half + pr];
    const uint32_t w = pack2<E>(x0 * c - x1 * sn, x0 * sn + x1 * c);
    uint16_t* dst = isq ? p.q_out + ((int64_t)b * p.Hq + h) * p.D + 2 * pr
                        : p.kc + b * p.skc[0] + (int64_t)h * p.skc[1] + (int64_t)pos * p.skc[2] + 2 * pr;
    dst[0] = uint16_t(w & 0xffffu);
    dst[1] = uint16_t(w >> 16);
  } else {
    const int64_t j = i - nq - nk;
    const int pr = int(j % half);
    const int h = int((j / half) % p.Hkv);
    const int b = int(j / half / p.Hkv);
    const int64_t off = b * p.sv[0] + (int64_t)h * p.sv[1] + 2 * pr;
    const uint32_t w = pack2<E>(load_in<E, XT>(p.v, off), load_in<E, XT>(p.v, off + 1));
    uint16_t* dst = p.vc + b * p.svc[0] + (int64_t)h * p.svc[1] + (int64_t)pos * p.svc[2] + 2 * pr;
    dst[0] = uint16_t(w & 0xffffu);
    dst[1] = uint16_t(w >> 16);
  }
}

}  // namespace mt
