// Top-k sampling of one token per row, for generation: the draw that
// TradingModel.generate makes after each decode step (the reference's
// model.py:141-145: keep the logits >= the k-th largest, softmax,
// torch.multinomial for one sample), in the form torch.multinomial uses for
// one sample -- argmax over the row of p / E with E ~ Exponential(1), the
// noise E coming from the caller (drawn by torch from its generator, so the
// same seed gives the same stream).  One launch instead of a dozen library
// kernels (a multi-pass radix top-k, the mask, the softmax, the division, the
// argmax).
//
// One workgroup of 1024 threads per row, the row held in registers
// (EPT values per thread, vocab <= 1024 EPT) as order-preserving 32-bit keys.
// A row lives on one CU, so the kernel is bound by its chain of dependent
// steps, not by bandwidth; what it avoids is block-wide barriers.
//
// k <= 1024: every wave finds the ceil(k / 16)-th and the k-th largest of its 64
// lane maxima (one ballot and count per bit, no barrier).  At least k keys of the
// row are >= the smallest of the 16 first bounds, and >= the largest of the
// second ones, so the k-th key is too.  The keys at or above the larger of the two
// (about 60 of 16384 random ones at k = 16, 110 at k = 50) go to LDS in index
// order of (wave, slot, lane); a candidate is kept when fewer than k candidates
// are larger, which keeps every tie at the k-th value, as the reference's
// `logits < values[:, [-1]]` mask does.  One wave then takes the
// maximum, the sum of exp(x - max), p = exp(x - max) / sum and the first
// index of the largest p / E, reading E for the candidates alone: four
// barriers in all.  32 rows of 16384, k = 16: 24.0 -> 9.7 us a launch,
// k = 50: 24.6 -> 12.5; 45 of 1385, k = 50: 18.7 -> 12.2.
//
// k > 1024, or more than kSampleCand candidates (long runs of equal logits): the
// k-th key bit by bit with block-wide counts (32 of them, two barriers each),
// then block-wide reductions over the row (the 24.0 us).
#pragma once

#include "mt_common.h"

namespace mt {

constexpr int kSampleThreads = 1024;

// order-preserving key of a float (larger float, larger key; NaN excluded)
__device__ __forceinline__ uint32_t sample_key(float x) {
  const uint32_t u = __float_as_uint(x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// block-wide max or sum of one float per thread (every thread gets it);
// `buf` holds kSampleThreads / 64 floats, reused: a barrier guards both ends
template <bool MAX>
__device__ __forceinline__ float block_reduce(float v, float* buf) {
  v = wave_reduce<0, MAX>(v);
  const int wave = threadIdx.x >> 6;
  __syncthreads();  // the previous reduction's reads of buf are done
  if ((threadIdx.x & 63) == 0) buf[wave] = v;
  __syncthreads();
  float r = buf[0];
#pragma unroll
  for (int w = 1; w < kSampleThreads / 64; ++w) r = red_op<MAX>(r, buf[w]);
  return r;
}

constexpr int kSampleCand = 1024;   // candidates held in LDS
constexpr int kSampleWaves = kSampleThreads / 64;
constexpr int kSampleWaveK = 64 * kSampleWaves;  // largest k of the candidate path: the lane maxima hold a k-th

__device__ __forceinline__ float sample_unkey(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? k & 0x7fffffffu : ~k);
}

struct SampleCand {
  uint32_t bound[2][kSampleWaves];
  int count[kSampleWaves];
  uint32_t key[kSampleCand];
  int idx[kSampleCand];  // vocabulary index; -1 once dropped
  float noise[kSampleCand];
};

// The candidate path; false (nothing written) when the row has more than
// kSampleCand candidates.  The result is the same on every thread.
template <int EPT>
__device__ __forceinline__ bool sample_candidates(const uint32_t (&key)[EPT], const float* e, int V, int k,
                                                  SampleCand& s, int64_t* out) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t mx = 0u;
#pragma unroll
  for (int j = 0; j < EPT; ++j) mx = max(mx, key[j]);
  // the k1-th and k-th largest lane maxima (0 where the wave holds fewer values)
  const int k1 = (k + kSampleWaves - 1) / kSampleWaves;
  uint32_t t1 = 0u, t2 = 0u;
  for (int bit = 31; bit >= 0; --bit) {
    const uint32_t c1 = t1 | (1u << bit), c2 = t2 | (1u << bit);
    if (__popcll(__ballot(mx >= c1)) >= k1) t1 = c1;
    if (__popcll(__ballot(mx >= c2)) >= k) t2 = c2;
  }
  if (lane == 0) {
    s.bound[0][wave] = t1;
    s.bound[1][wave] = t2;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kSampleWaves; ++w) {
    t1 = min(t1, s.bound[0][w]);
    t2 = max(t2, s.bound[1][w]);
  }
  const uint32_t t = max(t1, t2);
  int mine = 0;
#pragma unroll
  for (int j = 0; j < EPT; ++j) mine += __popcll(__ballot(key[j] >= t && tid + j * kSampleThreads < V));
  if (lane == 0) s.count[wave] = mine;
  __syncthreads();
  int at = 0, n = 0;
#pragma unroll
  for (int w = 0; w < kSampleWaves; ++w) {
    const int c = s.count[w];
    at += w < wave ? c : 0;
    n += c;
  }
  if (n > kSampleCand) return false;
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int i = tid + j * kSampleThreads;
    const bool in = key[j] >= t && i < V;
    const uint64_t mask = __ballot(in);
    if (in) {
      const int slot = at + __popcll(mask & ((1ull << lane) - 1));
      s.key[slot] = key[j];
      s.idx[slot] = i;
    }
    at += __popcll(mask);
  }
  const int pad = n + tid;  // up to three zero keys complete the last group of four
  if (tid < 3 && pad < kSampleCand) s.key[pad] = 0u;
  __syncthreads();
  if (tid < n) {
    const uint32_t own = s.key[tid];
    const int idx = s.idx[tid];
    const float ev = e[idx];
    int larger = 0;
    for (int c = 0; c < n; c += 4) {
      const u32x4 q = *reinterpret_cast<const u32x4*>(&s.key[c]);
#pragma unroll
      for (int x = 0; x < 4; ++x) larger += q[x] > own ? 1 : 0;
    }
    s.noise[tid] = ev;
    if (larger >= k) s.idx[tid] = -1;
  }
  __syncthreads();
  if (wave > 0) return true;
  float m = -INFINITY;
  for (int c = lane; c < n; c += 64)
    if (s.idx[c] >= 0) m = fmaxf(m, sample_unkey(s.key[c]));
  m = wave_reduce<0, true>(m);
  float sum = 0.f;
  for (int c = lane; c < n; c += 64)
    if (s.idx[c] >= 0) sum += expf(sample_unkey(s.key[c]) - m);
  sum = wave_reduce<0, false>(sum);
  const float inv = 1.f / sum;
  float best = -1.f, bi = (float)V;
  for (int c = lane; c < n; c += 64) {
    const int i = s.idx[c];
    if (i < 0) continue;
    const float q = expf(sample_unkey(s.key[c]) - m) * inv / s.noise[c];
    if (q > best || (q == best && (float)i < bi)) {
      best = q;
      bi = (float)i;
    }
  }
  const float top = wave_reduce<0, true>(best);
  const float first = -wave_reduce<0, true>(best == top ? -bi : -(float)V);
  if (lane == 0) out[blockIdx.x] = (int64_t)first;
  return true;
}

template <int EPT>
__global__ __launch_bounds__(kSampleThreads) void topk_sample_kernel(const float* logits, int64_t ld,
                                                                     const float* noise, int64_t ldn, int V, int k,
                                                                     int64_t* out) {
  __shared__ float buf[kSampleThreads / 64];
  __shared__ __attribute__((aligned(16))) SampleCand cand_lds;
  const int tid = threadIdx.x;
  const float* x = logits + (int64_t)blockIdx.x * ld;
  const float* e = noise + (int64_t)blockIdx.x * ldn;
  float v[EPT];
  uint32_t key[EPT];
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int i = tid + j * kSampleThreads;
    v[j] = i < V ? x[i] : -INFINITY;
    key[j] = i < V ? sample_key(v[j]) : 0u;  // padding: below every real key (k <= V)
  }
  if (k <= kSampleWaveK && sample_candidates<EPT>(key, e, V, k, cand_lds, out)) return;
  // the k-th largest key: the largest t with count(key >= t) >= k
  uint32_t t = 0;
  for (int bit = 31; bit >= 0; --bit) {
    const uint32_t cand = t | (1u << bit);
    float c = 0.f;
#pragma unroll
    for (int j = 0; j < EPT; ++j) c += key[j] >= cand ? 1.f : 0.f;
    if (block_reduce<false>(c, buf) >= (float)k) t = cand;
  }
  float m = -INFINITY;
#pragma unroll
  for (int j = 0; j < EPT; ++j)
    if (key[j] >= t) m = fmaxf(m, v[j]);
  m = block_reduce<true>(m, buf);
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < EPT; ++j)
    if (key[j] >= t) s += expf(v[j] - m);
  s = block_reduce<false>(s, buf);
  const float inv = 1.f / s;
  // the largest p / E, first index among equals
  float best = -1.f, bi = (float)V;
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int i = tid + j * kSampleThreads;
    if (i < V && key[j] >= t) {
      const float q = expf(v[j] - m) * inv / e[i];
      if (q > best) {  // j ascending: the first index wins among this thread's equals
        best = q;
        bi = (float)i;
      }
    }
  }
  const float top = block_reduce<true>(best, buf);
  const float first = -block_reduce<true>(best == top ? -bi : -(float)V, buf);
  if (tid == 0) out[blockIdx.x] = (int64_t)first;
}

}  // namespace mt
