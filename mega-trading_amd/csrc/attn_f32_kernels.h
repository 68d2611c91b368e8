// fp32 causal grouped-query attention on fp32 MFMA (v_mfma_f32_32x32x2_f32).
//
// The reference takes fp32 tensors on its Triton path
// (src/mega_trading/kernels/triton_attention.py:16): its forward dots run on
// fp32 inputs (TF32 by Triton's default) and its backward is the dense fp32
// fallback (:88-111).  These kernels compute both in full fp32: the MFMA
// multiplies fp32 operands exactly and accumulates in fp32, P and dS stay fp32
// (the reference casts P to V's dtype, fp32 here, :340), and the softmax runs
// in fp32.
//
// What bounds them is the fp32 MFMA (64 cycles for 32 x 32 x 2 products; a
// library product sustains 154 TFLOP/s).  One wave owns 32 query rows (or 32
// keys) and works on 32 x 32 score tiles; the tiles it multiplies come into its
// own LDS block by asynchronous copies of whole rows, each issued as soon as the
// tile before it has been read for the last time and waited for (by count)
// only where its first operand is read, so a wave needs no barrier and the
// copies run behind the MFMAs of the phases between.  Read straight from global
// memory, a row per lane with 16 bytes from each of 64 cache lines a load, the
// same tiles left the MFMAs idle two thirds of the time.  Measured, forward +
// backward with RoPE: 8 x 512, 16 / 4 heads of 64: 362 -> 238 us; 4 x 1000, 8 / 2
// of 64: 441 -> 285; 2 x 1024, 16 / 4 of 128: 1086 -> 605; 2 x 256, 4 / 2 of 32:
// 48.6 -> 33.0.
//
// MFMA layout (32x32x2, fp32): A[m][k] comes from lane m + 32 k, B[k][n] from
// lane n + 32 k, and lane l holds C[m][n = l % 32] for m = 8 (i / 4) + 4 (l / 32)
// + i % 4, i = 0..15.  A lane's half h = l / 32 feeds contraction slot k = h.
//  * Scores: the contraction runs over d, lane half h supplying the d values
//    [h D/2, (h + 1) D/2) of its row (the pairing is the same on both operands,
//    so the product is the full dot product).
//  * Products that contract over the 32 keys (or rows) of a score tile use the
//    score accumulator itself as the B operand: step j pairs slot k = h with
//    key 8 (j / 4) + 4 h + j % 4, exactly the key that lane holds in its slot
//    j, and the A operand reads the matching row.
#pragma once

#include "attn_kernels.h"

namespace mt {

__device__ __forceinline__ f32x16 mfma_f32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// the row (key) a lane's accumulator slot i refers to, within a 32-row tile
__device__ __forceinline__ int f32_slot_row(int i, int hh) { return 8 * (i >> 2) + 4 * hh + (i & 3); }

// wave task t -> (batch, head, 32-row block), longest causal rows first; the
// four waves of a workgroup share a row block when B * H is a multiple of 4
struct F32Task {
  int b, h, blk;
};
__device__ __forceinline__ F32Task f32_task(int t, int B, int H, int nblk, bool reverse) {
  F32Task r;
  const int bh = t % (B * H);
  r.blk = reverse ? nblk - 1 - t / (B * H) : t / (B * H);
  r.h = bh % H;
  r.b = bh / H;
  return r;
}

__device__ __forceinline__ const float* fptr(const uint16_t* p) { return reinterpret_cast<const float*>(p); }
__device__ __forceinline__ float* fptr(uint16_t* p) { return reinterpret_cast<float*>(p); }

// Y = rot(X) for an fp32 [B, H, T, D] tensor, Y contiguous; one thread per 4
// consecutive d values (two interleaved pairs).
template <int D>
__global__ __launch_bounds__(256) void rope_f32_kernel(const float* x, int64_t s0, int64_t s1, int64_t s2, float* y,
                                                       const float* cos, const float* sin, int H, int T,
                                                       int64_t n4) {
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= n4) return;
  const int d0 = int(c % (D / 4)) * 4;
  const int64_t row = c / (D / 4);
  const int t = int(row % T);
  const int64_t bh = row / T;
  const int h = int(bh % H);
  const int64_t b = bh / H;
  const f32x4 v = *reinterpret_cast<const f32x4*>(x + b * s0 + h * s1 + (int64_t)t * s2 + d0);
  const f32x2 cs = *reinterpret_cast<const f32x2*>(cos + (int64_t)t * (D / 2) + d0 / 2);
  const f32x2 sn = *reinterpret_cast<const f32x2*>(sin + (int64_t)t * (D / 2) + d0 / 2);
  const f32x4 r = {v[0] * cs[0] - v[1] * sn[0], v[0] * sn[0] + v[1] * cs[0], v[2] * cs[1] - v[3] * sn[1],
                   v[2] * sn[1] + v[3] * cs[1]};
  *reinterpret_cast<f32x4*>(y + row * D + d0) = r;
}

// ---------------------------------------------------------------------------
// LDS tiles of fp32 rows: a row of D floats is laid out, swizzled and copied as
// a row of 2 D 16-bit values (lds_tile.h).
// ---------------------------------------------------------------------------
// Copies of 32 rows by one wave (WaveStager, lds_tile.h).
template <int D, bool KEPT = true>
using F32Stager = WaveStager<float, 2 * D, 32, KEPT>;

// Operand reads of such a tile.
//  * row: lane (row l32, half hh) reads d values hh D/2 + 4 j .. + 3 (the score
//    contraction's pairing); 16 consecutive rows of a chunk column cover 256
//    distinct bytes.
//  * tr: lane reads d = 32 dt + l32 of the row its accumulator slot j refers to.
template <int D>
struct F32Tile {
  using TL = Tile<2 * D>;
  int rbase, tbase;
  __device__ __forceinline__ F32Tile(int l32, int hh)
      : rbase(l32 * TL::RB + (((hh * (D / 8)) ^ TL::swz(l32)) << 4)),
        tbase(4 * hh * TL::RB + (((l32 >> 2) ^ hh) << 4) + (l32 & 3) * 4) {}
  __device__ __forceinline__ f32x4 row(const char* lds, int j) const {
    return *reinterpret_cast<const f32x4*>(lds + (rbase ^ (j << 4)));
  }
  // the swizzle of row 8 (j / 4) + 4 hh + j % 4 without hh, which tbase holds
  static constexpr int tr_swz(int j) {
    return TL::NC == 8 ? (((j >> 1) & 1) << 2) | (((j >> 2) & 1) << 1) : ((j & 3) << 2) | (((j >> 2) & 1) << 1);
  }
  __device__ __forceinline__ float tr(const char* lds, int j, int dt) const {
    return *reinterpret_cast<const float*>(lds + (8 * (j >> 2) + (j & 3)) * TL::RB +
                                           (tbase ^ (((8 * dt) ^ tr_swz(j)) << 4)));
  }
};

// The values a wave loaded for itself are here.  Asked before a loop over copied
// tiles: left to the first use, the compiler's wait stands inside the loop and
// drains the copies in flight in every pass.
template <int N>
__device__ __forceinline__ void loads_done(const float (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" ::"v"(v[i]));
}

// ---------------------------------------------------------------------------
// Forward: online softmax over 32-key tiles, O and LSE.  SPLIT = 4: the tiles of
// a row block are dealt to the 4 waves of a workgroup, whose (O, m, l) are
// merged; SPLIT = 1: every wave has a row block of its own.
// ---------------------------------------------------------------------------
template <int D, bool ROPE, int SPLIT>
__global__ __launch_bounds__(256, D <= 64 ? 2 : 1) void attn_fwd_f32_kernel(AttnParams p) {
  constexpr int HD = D / 2;  // d values per lane
  constexpr int DT = D / 32;
  using TL = Tile<2 * D>;
  constexpr int BUF = 2 * 32 * TL::RB;  // a wave's K and V tiles
  __shared__ __attribute__((aligned(1024))) char smem[4 * BUF];
  // after the loop, waves 1-3: unnormalised O [wave - 1][dt, g][lane] and (m, l)
  f32x4 (*red_o)[DT * 4][64] = reinterpret_cast<f32x4 (*)[DT * 4][64]>(smem);
  __shared__ f32x2 red_ml[3][64];
  const int lane = threadIdx.x & 63, l32 = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nblk = (p.T + 31) / 32;
  const int t = SPLIT == 4 ? (int)blockIdx.x : fold_order(blockIdx.x, gridDim.x, p.fwd_fold) * 4 + wave;
  if (t >= p.B * p.Hq * nblk) return;  // (workgroup-uniform with SPLIT = 4; no barriers otherwise)
  const F32Task task = f32_task(t, p.B, p.Hq, nblk, true);
  const int kvh = task.h / p.R;
  const int row = task.blk * 32 + l32;
  const int rc = min(row, p.T - 1);
  const int kt0 = SPLIT == 4 ? wave : 0;
  const float* kbase = fptr(p.k) + task.b * p.sk[0] + (int64_t)kvh * p.sk[1];
  const float* vbase = fptr(p.v) + task.b * p.sv[0] + (int64_t)kvh * p.sv[1];
  F32Stager<D> kst, vst;
  kst.init(p.sk[2], lane);
  vst.init(p.sv[2], lane);
  char* K = smem + wave * BUF;
  char* V = K + 32 * TL::RB;
  if (kt0 <= task.blk) {
    kst.stage(K, kbase, p.sk[2], kt0 * 32, p.T);
    vst.stage(V, vbase, p.sv[2], kt0 * 32, p.T);
  }

  // the lane's half of its query row, rotated if RoPE (and written to q_rot,
  // by wave 0 of a split block)
  float qv[HD];
  {
    const float* qr = fptr(p.q) + task.b * p.sq[0] + (int64_t)task.h * p.sq[1] + (int64_t)rc * p.sq[2] + hh * HD;
#pragma unroll
    for (int j = 0; j < HD / 4; ++j) {
      f32x4 x = *reinterpret_cast<const f32x4*>(qr + 4 * j);
      if constexpr (ROPE) {
        const int d0 = hh * HD + 4 * j;
        const f32x2 cs = *reinterpret_cast<const f32x2*>(p.cos + (int64_t)rc * (D / 2) + d0 / 2);
        const f32x2 sn = *reinterpret_cast<const f32x2*>(p.sin + (int64_t)rc * (D / 2) + d0 / 2);
        x = f32x4{x[0] * cs[0] - x[1] * sn[0], x[0] * sn[0] + x[1] * cs[0], x[2] * cs[1] - x[3] * sn[1],
                  x[2] * sn[1] + x[3] * cs[1]};
        if ((SPLIT == 1 || wave == 0) && row < p.T)
          *reinterpret_cast<f32x4*>(fptr(p.qrot) + (((int64_t)task.b * p.Hq + task.h) * p.T + row) * D + d0) = x;
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) qv[4 * j + c] = x[c];
    }
  }
  const float c2 = p.scale_log2;
  const F32Tile<D> tile(l32, hh);

  f32x16 oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) zero16(oacc[dt]);
  float m = -INFINITY, l = 0.f;
  for (int kt = kt0; kt <= task.blk; kt += SPLIT) {
    const bool more = kt + SPLIT <= task.blk;
    // K is here; V may still be on its way (the first time the wave also has its
    // Q loads and Q_rot stores behind the copies)
    if (kt == kt0) copies_done<0>();
    else copies_done<F32Stager<D>::COPIES>();
    // S^T (lane = query, slots = keys)
    f32x16 s = {};
#pragma unroll
    for (int j = 0; j < HD / 4; ++j) {
      const f32x4 k4 = tile.row(K, j);
#pragma unroll
      for (int c = 0; c < 4; ++c) s = mfma_f32(k4[c], qv[4 * j + c], s);
    }
    reads_done();
    if (more) kst.stage(K, kbase, p.sk[2], (kt + SPLIT) * 32, p.T);
    // scaled before the mask: any scale, 0 and negative ones too, leaves -inf as it is
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] *= c2;
    if (kt == task.blk) {  // the diagonal; tiles left of it have every key <= every row
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (f32_slot_row(i, hh) > l32) s[i] = -INFINITY;
    }
    // the diagonal tile holds key 32 kt <= row, so m is finite after a wave's first tile
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[i]);
    const float mnew = fmaxf(m, max_with_partner(mx));
    const float alpha = exp2_fast(m - mnew);
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = exp2_fast(s[i] - mnew);
      ps += s[i];
    }
    l = l * alpha + ps;
    m = mnew;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) oacc[dt][i] *= alpha;
    // O^T += V^T P^T over the tile's 32 keys
    if (more) copies_done<F32Stager<D>::COPIES>();
    else copies_done<0>();
#pragma unroll
    for (int j = 0; j < 16; ++j)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) oacc[dt] = mfma_f32(tile.tr(V, j, dt), s[j], oacc[dt]);
    reads_done();
    if (more) vst.stage(V, vbase, p.sv[2], (kt + SPLIT) * 32, p.T);
  }
  if constexpr (SPLIT == 4) {
    __syncthreads();  // every wave's tiles are read: the block is reused for the merge
    // merge the four waves' (O, m, l) with the log-sum-exp rule (a wave that
    // had no tile has m = -inf and contributes nothing); m is the same on a
    // lane and its lane^32 partner
    if (wave > 0) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          red_o[wave - 1][dt * 4 + g][lane] =
              f32x4{oacc[dt][4 * g], oacc[dt][4 * g + 1], oacc[dt][4 * g + 2], oacc[dt][4 * g + 3]};
      red_ml[wave - 1][lane] = f32x2{m, l};
    }
    __syncthreads();
    if (wave > 0) return;
    {
      f32x2 ml[3];
      float mm = m;
#pragma unroll
      for (int w = 0; w < 3; ++w) {
        ml[w] = red_ml[w][lane];
        mm = fmaxf(mm, ml[w][0]);
      }
      const float a0 = exp2_fast(m - mm);
      l *= a0;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[dt][i] *= a0;
#pragma unroll
      for (int w = 0; w < 3; ++w) {
        const float aw = exp2_fast(ml[w][0] - mm);
        l = __builtin_fmaf(aw, ml[w][1], l);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const f32x4 o = red_o[w][dt * 4 + g][lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) oacc[dt][4 * g + e] = __builtin_fmaf(aw, o[e], oacc[dt][4 * g + e]);
          }
      }
      m = mm;
    }
  }
  if (row >= p.T) return;
  const float lt = sum_with_partner(l);
  const float inv = 1.f / lt;
  float* ob = fptr(p.out) + task.b * p.so[0] + (int64_t)task.h * p.so[1] + (int64_t)row * p.so[2];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(ob + 32 * dt + 8 * g + 4 * hh) =
          f32x4{oacc[dt][4 * g] * inv, oacc[dt][4 * g + 1] * inv, oacc[dt][4 * g + 2] * inv, oacc[dt][4 * g + 3] * inv};
  if (hh == 0) p.lse[((int64_t)task.b * p.Hq + task.h) * p.T + row] = (m + __builtin_amdgcn_logf(lt)) * kLn2;
}

// ---------------------------------------------------------------------------
// Backward prep: -delta = -rowsum(O * dO) and -LSE log2(e) (fp32 O and dO).
// ---------------------------------------------------------------------------
template <int D>
__global__ __launch_bounds__(256) void attn_bwd_prep_f32_kernel(AttnParams p) {
  constexpr int LPR = D / 4;  // lanes per row, one 16-byte chunk each
  const int64_t rows = (int64_t)p.B * p.Hq * p.T;
  const int64_t row = (int64_t)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
  const int c = threadIdx.x % LPR;
  float sum = 0.f;
  if (row < rows) {
    const int t = int(row % p.T);
    const int64_t bh = row / p.T;
    const int h = int(bh % p.Hq);
    const int64_t b = bh / p.Hq;
    const f32x4 o = *reinterpret_cast<const f32x4*>(fptr(p.o) + b * p.so[0] + h * p.so[1] + (int64_t)t * p.so[2] + 4 * c);
    const f32x4 g =
        *reinterpret_cast<const f32x4*>(fptr(p.dout) + b * p.sdo[0] + h * p.sdo[1] + (int64_t)t * p.sdo[2] + 4 * c);
    sum = o[0] * g[0] + o[1] * g[1] + o[2] * g[2] + o[3] * g[3];
  }
#pragma unroll
  for (int msk = 1; msk < LPR; msk <<= 1) sum += __shfl_xor(sum, msk, LPR);
  if (c == 0 && row < rows) {
    p.ndelta[row] = -sum;
    p.nlse2[row] = -p.lse[row] * kLog2e;
  }
}

// ---------------------------------------------------------------------------
// Backward dQ: per workgroup 32 query rows of one head (SPLIT = 4; SPLIT = 1 as
// in the forward, the tiles of a row block on one wave); the 32-key tiles on
// or left of the diagonal are dealt to the 4 waves in turn (each recomputes
// S^T and dP^T for its tiles, lane = query: P = 2^(S c - LSE2), dS = P (dP -
// delta), dQ^T += K^T dS^T), and the four partial sums are added through LDS.
// ---------------------------------------------------------------------------
template <int D, bool ROPE, int SPLIT>
__global__ __launch_bounds__(256, D <= 64 ? 2 : 1) void attn_bwd_dq_f32_kernel(AttnParams p) {
  constexpr int HD = D / 2;
  constexpr int DT = D / 32;
  using TL = Tile<2 * D>;
  constexpr int BUF = 2 * 32 * TL::RB;  // a wave's K and V tiles
  __shared__ __attribute__((aligned(1024))) char smem[4 * BUF];
  f32x4 (*red)[DT * 4][64] = reinterpret_cast<f32x4 (*)[DT * 4][64]>(smem);  // after the loop: waves 1-3
  const int lane = threadIdx.x & 63, l32 = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nblk = (p.T + 31) / 32;
  const int t = SPLIT == 4 ? (int)blockIdx.x : fold_order(blockIdx.x, gridDim.x, p.fwd_fold) * 4 + wave;
  if (t >= p.B * p.Hq * nblk) return;  // (workgroup-uniform with SPLIT = 4; no barriers otherwise)
  const F32Task task = f32_task(t, p.B, p.Hq, nblk, true);
  const int kvh = task.h / p.R;
  const int row = task.blk * 32 + l32;
  const int rc = min(row, p.T - 1);
  const int64_t rowbase = ((int64_t)task.b * p.Hq + task.h) * p.T;

  const int kt0 = SPLIT == 4 ? wave : 0;
  const float* kbase = fptr(p.k) + task.b * p.sk[0] + (int64_t)kvh * p.sk[1];
  const float* vbase = fptr(p.v) + task.b * p.sv[0] + (int64_t)kvh * p.sv[1];
  F32Stager<D> kst, vst;
  kst.init(p.sk[2], lane);
  vst.init(p.sv[2], lane);
  char* K = smem + wave * BUF;
  char* V = K + 32 * TL::RB;
  if (kt0 <= task.blk) {
    vst.stage(V, vbase, p.sv[2], kt0 * 32, p.T);
    kst.stage(K, kbase, p.sk[2], kt0 * 32, p.T);
  }
  float qv[HD], gv[HD];
  {
    const float* qr = fptr(p.q) + task.b * p.sq[0] + (int64_t)task.h * p.sq[1] + (int64_t)rc * p.sq[2] + hh * HD;
    const float* gr = fptr(p.dout) + task.b * p.sdo[0] + (int64_t)task.h * p.sdo[1] + (int64_t)rc * p.sdo[2] + hh * HD;
#pragma unroll
    for (int j = 0; j < HD / 4; ++j) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(qr + 4 * j);
      const f32x4 b = *reinterpret_cast<const f32x4*>(gr + 4 * j);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        qv[4 * j + c] = a[c];
        gv[4 * j + c] = b[c];
      }
    }
  }
  const float nl2 = p.nlse2[rowbase + rc];
  const float nd = p.ndelta[rowbase + rc];
  const float c2 = p.scale_log2;
  const F32Tile<D> tile(l32, hh);

  f32x16 dq[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) zero16(dq[dt]);
  // dP first, then S: V's next tile is copied behind S and dQ, K's behind the next dP
  for (int kt = kt0; kt <= task.blk; kt += SPLIT) {
    const bool more = kt + SPLIT <= task.blk;
    if (kt == kt0) copies_done<0>();
    else copies_done<F32Stager<D>::COPIES>();
    f32x16 s = {}, dp = {};
#pragma unroll
    for (int j = 0; j < HD / 4; ++j) {
      const f32x4 v4 = tile.row(V, j);
#pragma unroll
      for (int c = 0; c < 4; ++c) dp = mfma_f32(v4[c], gv[4 * j + c], dp);
    }
    reads_done();
    if (more) {
      vst.stage(V, vbase, p.sv[2], (kt + SPLIT) * 32, p.T);
      copies_done<F32Stager<D>::COPIES>();
    } else {
      copies_done<0>();
    }
#pragma unroll
    for (int j = 0; j < HD / 4; ++j) {
      const f32x4 k4 = tile.row(K, j);
#pragma unroll
      for (int c = 0; c < 4; ++c) s = mfma_f32(k4[c], qv[4 * j + c], s);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = exp2_fast(__builtin_fmaf(s[i], c2, nl2));
    if (kt == task.blk) {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (f32_slot_row(i, hh) > l32) s[i] = 0.f;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] *= dp[i] + nd;  // dS
#pragma unroll
    for (int j = 0; j < 16; ++j)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) dq[dt] = mfma_f32(tile.tr(K, j, dt), s[j], dq[dt]);
    reads_done();
    if (more) kst.stage(K, kbase, p.sk[2], (kt + SPLIT) * 32, p.T);
  }
  if constexpr (SPLIT == 4) {
    __syncthreads();  // every wave's tiles are read: the block is reused for the sums
    // the four waves' partial sums: waves 1-3 hand theirs to wave 0
    if (wave > 0) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          red[wave - 1][dt * 4 + g][lane] = f32x4{dq[dt][4 * g], dq[dt][4 * g + 1], dq[dt][4 * g + 2], dq[dt][4 * g + 3]};
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 0; w < 3; ++w)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 a = red[w][dt * 4 + g][lane];
#pragma unroll
          for (int e = 0; e < 4; ++e) dq[dt][4 * g + e] += a[e];
        }
  }
  if (row >= p.T) return;
  float* out = fptr(p.out) + task.b * p.sout[0] + (int64_t)task.h * p.sout[1] + (int64_t)row * p.sout[2];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = 32 * dt + 8 * g + 4 * hh;
      float x0 = dq[dt][4 * g] * p.scale, x1 = dq[dt][4 * g + 1] * p.scale;
      float x2 = dq[dt][4 * g + 2] * p.scale, x3 = dq[dt][4 * g + 3] * p.scale;
      if constexpr (ROPE)
        rope_back4(x0, x1, x2, x3, p.cos + (int64_t)row * (D / 2) + d / 2, p.sin + (int64_t)row * (D / 2) + d / 2);
      *reinterpret_cast<f32x4*>(out + d) = f32x4{x0, x1, x2, x3};
    }
}

// ---------------------------------------------------------------------------
// Backward dK / dV: per workgroup 32 keys of one KV head, K and V in
// registers; the (query head, 32-row tile on or below the diagonal) pairs of
// the block are dealt to the 4 waves in turn (each recomputes S and dP for its
// pairs: lane = key, slots = rows; dV^T += dO^T P, dK^T += Q^T dS), and the
// four partial sums are added through LDS.  A wave per key block would leave
// most of the GPU idle at small shapes (32 waves on 1024
// SIMDs, the longest walking every row of its heads).
// ---------------------------------------------------------------------------
template <int D, bool ROPE>
__global__ __launch_bounds__(256, D <= 64 ? 2 : 1) void attn_bwd_dkv_f32_kernel(AttnParams p) {
  constexpr int HD = D / 2;
  constexpr int DT = D / 32;
  using TL = Tile<2 * D>;
  constexpr int BUF = 2 * 32 * TL::RB + 256;  // a wave's Q rows, dO rows, and their -LSE log2(e) | -delta
  constexpr int RED = 3 * 2 * DT * 4 * 64 * 16;
  __shared__ __attribute__((aligned(1024))) char smem[4 * BUF > RED ? 4 * BUF : RED];
  f32x4 (*red)[2 * DT * 4][64] = reinterpret_cast<f32x4 (*)[2 * DT * 4][64]>(smem);  // after the loop: waves 1-3
  const int lane = threadIdx.x & 63, l32 = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nblk = (p.T + 31) / 32;
  const int t = blockIdx.x;
  if (t >= p.B * p.Hkv * nblk) return;  // (workgroup-uniform)
  const F32Task task = f32_task(t, p.B, p.Hkv, nblk, false);  // smallest key block (most rows) first
  const int key = task.blk * 32 + l32;
  const int kc = min(key, p.T - 1);

  float kv[HD], vv[HD];
  {
    const float* kr = fptr(p.k) + task.b * p.sk[0] + (int64_t)task.h * p.sk[1] + (int64_t)kc * p.sk[2] + hh * HD;
    const float* vr = fptr(p.v) + task.b * p.sv[0] + (int64_t)task.h * p.sv[1] + (int64_t)kc * p.sv[2] + hh * HD;
#pragma unroll
    for (int j = 0; j < HD / 4; ++j) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(kr + 4 * j);
      const f32x4 b = *reinterpret_cast<const f32x4*>(vr + 4 * j);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        kv[4 * j + c] = a[c];
        vv[4 * j + c] = b[c];
      }
    }
  }
  const float c2 = p.scale_log2;
  f32x16 dk[DT], dv[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    zero16(dk[dt]);
    zero16(dv[dt]);
  }
  const int ntile = nblk - task.blk;  // row tiles per head on or below the diagonal
  const int npair = p.R * ntile;
  // Each wave copies the rows of its next pair into its own LDS block: Q behind
  // dV, dO behind the next S.
  char* Qt = smem + wave * BUF;
  char* Gt = Qt + 32 * TL::RB;
  const float* vec = reinterpret_cast<const float*>(Gt + 32 * TL::RB);
  F32Stager<D, D <= 64> qst, gst;
  qst.init(p.sq[2], lane);
  gst.init(p.sdo[2], lane);
  const F32Tile<D> tile(l32, hh);
  auto stage_q = [&](int u) {
    const int head = task.h * p.R + u % p.R, qt = task.blk + u / p.R;
    qst.stage(Qt, fptr(p.q) + task.b * p.sq[0] + (int64_t)head * p.sq[1], p.sq[2], qt * 32, p.T);
  };
  auto stage_g = [&](int u) {
    const int head = task.h * p.R + u % p.R, qt = task.blk + u / p.R;
    gst.stage(Gt, fptr(p.dout) + task.b * p.sdo[0] + (int64_t)head * p.sdo[1], p.sdo[2], qt * 32, p.T);
    // lanes 0-31: the rows' -LSE log2(e), lanes 32-63: -delta
    lds_dma4((hh ? p.ndelta : p.nlse2) + ((int64_t)task.b * p.Hq + head) * p.T + min(qt * 32 + l32, p.T - 1),
             Gt + 32 * TL::RB);
  };
  if (wave < npair) {
    stage_q(wave);
    stage_g(wave);
  }
  // (D = 64, 8 x 512, 16 / 4 heads: 108.5 us without, 106.3 with; at D = 32 the
  // first tile's Q arrives before K and V, 2 x 256, 4 / 2 heads: 13.8 / 14.5)
  if constexpr (D > 32) {
    loads_done(kv);
    loads_done(vv);
  }
  for (int u = wave; u < npair; u += 4) {
    const int qt = task.blk + u / p.R;
    const bool more = u + 4 < npair;
    // S and dP: rows m = the tile's queries, lane = key
    f32x16 s = {}, dp = {};
    copies_done<F32Stager<D>::COPIES + 1>();  // Q (dO and its vectors may still be on their way)
#pragma unroll
    for (int j = 0; j < HD / 4; ++j) {
      const f32x4 q4 = tile.row(Qt, j);
#pragma unroll
      for (int c = 0; c < 4; ++c) s = mfma_f32(q4[c], kv[4 * j + c], s);
      if constexpr (D > 64) {
        if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // a few operands in flight, not all
      }
    }
    copies_done<0>();
#pragma unroll
    for (int j = 0; j < HD / 4; ++j) {
      const f32x4 g4 = tile.row(Gt, j);
#pragma unroll
      for (int c = 0; c < 4; ++c) dp = mfma_f32(g4[c], vv[4 * j + c], dp);
      if constexpr (D > 64) {
        if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const f32x4 nl = *reinterpret_cast<const f32x4*>(vec + 8 * a + 4 * hh);
      const f32x4 nd = *reinterpret_cast<const f32x4*>(vec + 32 + 8 * a + 4 * hh);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int i = 4 * a + c;
        s[i] = exp2_fast(__builtin_fmaf(s[i], c2, nl[c]));
        dp[i] += nd[c];
      }
    }
    if (qt == task.blk || qt * 32 + 32 > p.T) {  // the diagonal, or rows past T
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int qrow = qt * 32 + f32_slot_row(i, hh);
        if (key > qrow || qrow >= p.T) s[i] = 0.f;
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) dp[i] *= s[i];  // dS
#pragma unroll
    for (int j = 0; j < 16; ++j) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) dk[dt] = mfma_f32(tile.tr(Qt, j, dt), dp[j], dk[dt]);
      if constexpr (D > 64) {
        if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
    }
    reads_done();
    if (more) stage_q(u + 4);
#pragma unroll
    for (int j = 0; j < 16; ++j) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) dv[dt] = mfma_f32(tile.tr(Gt, j, dt), s[j], dv[dt]);
      if constexpr (D > 64) {
        if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
    }
    reads_done();
    if (more) stage_g(u + 4);
  }
  __syncthreads();  // every wave's tiles are read: the block is reused for the sums
  // the four waves' partial sums: waves 1-3 hand theirs to wave 0
  if (wave > 0) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        red[wave - 1][dt * 4 + g][lane] = f32x4{dk[dt][4 * g], dk[dt][4 * g + 1], dk[dt][4 * g + 2], dk[dt][4 * g + 3]};
        red[wave - 1][(DT + dt) * 4 + g][lane] =
            f32x4{dv[dt][4 * g], dv[dt][4 * g + 1], dv[dt][4 * g + 2], dv[dt][4 * g + 3]};
      }
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll 1
  for (int w = 0; w < 3; ++w)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 a = red[w][dt * 4 + g][lane], b = red[w][(DT + dt) * 4 + g][lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          dk[dt][4 * g + e] += a[e];
          dv[dt][4 * g + e] += b[e];
        }
      }
  if (key >= p.T) return;
  float* dkr = fptr(p.dk) + task.b * p.sdk[0] + (int64_t)task.h * p.sdk[1] + (int64_t)key * p.sdk[2];
  float* dvr = fptr(p.dv) + task.b * p.sdv[0] + (int64_t)task.h * p.sdv[1] + (int64_t)key * p.sdv[2];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = 32 * dt + 8 * g + 4 * hh;
      float x0 = dk[dt][4 * g] * p.scale, x1 = dk[dt][4 * g + 1] * p.scale;
      float x2 = dk[dt][4 * g + 2] * p.scale, x3 = dk[dt][4 * g + 3] * p.scale;
      if constexpr (ROPE)
        rope_back4(x0, x1, x2, x3, p.cos + (int64_t)key * (D / 2) + d / 2, p.sin + (int64_t)key * (D / 2) + d / 2);
      *reinterpret_cast<f32x4*>(dkr + d) = f32x4{x0, x1, x2, x3};
      *reinterpret_cast<f32x4*>(dvr + d) = f32x4{dv[dt][4 * g], dv[dt][4 * g + 1], dv[dt][4 * g + 2], dv[dt][4 * g + 3]};
    }
}

}  // namespace mt
