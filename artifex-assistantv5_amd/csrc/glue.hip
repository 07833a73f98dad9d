// Decode-step glue of a Llama-style layer around the quantized projections:
// RMSNorm (optionally fused with the residual add that precedes it), SwiGLU,
// rotate_half RoPE + KV-cache append + GQA attention for one new position,
// and greedy argmax.  Reference shaders: rmsnorm.wgsl:1-9,58-67,
// rope.wgsl:1-10, elementwise.wgsl:96-102 (gate_silu), argmax.wgsl; the
// layer loop is webgpu/src/engine/forward-pass.ts:2925-3297.
//
// All kernels are f32, one row (or one KV head) per workgroup; they are small
// and latency-bound, so the goal is one launch per op with coalesced 16-byte
// accesses, not occupancy.
#include <climits>
#include <mutex>

#include "common.hpp"

namespace gguf {

namespace {

constexpr int kGlueThreads = 256;

// Sum over the workgroup; every thread gets the result.  `red` holds one
// float per wave.
__device__ __forceinline__ float block_sum(float v, float *red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float s = 0.f;
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += red[w];
  return s;
}

__device__ __forceinline__ float block_max(float v, float *red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float s = red[0];
  for (int w = 1; w < (int)(blockDim.x >> 6); ++w) s = fmaxf(s, red[w]);
  return s;
}

// y = x * 1/sqrt(mean(x^2) + eps) * w  (rmsnorm.wgsl:58-67, direct weight);
// with r != null the residual add x += r is applied first and x is updated.
// Rows of up to 4 * 4 * kNormThreads elements are held in registers (one
// read of x); longer rows are read twice.
constexpr int kNormThreads = 1024;
__global__ __launch_bounds__(kNormThreads) void rmsnorm_kernel(float *__restrict__ x,
                                                               const float *__restrict__ r,
                                                               const float *__restrict__ w,
                                                               float eps, float *__restrict__ y,
                                                               int n) {
  __shared__ float red[kNormThreads / 64];
  float *xr = x + (int64_t)blockIdx.x * n;
  const float *rr = r ? r + (int64_t)blockIdx.x * n : nullptr;
  float *yr = y + (int64_t)blockIdx.x * n;
  constexpr int R = 4;
  float4 v[R];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < R; ++c) {
    const int i = 4 * (c * kNormThreads + threadIdx.x);
    v[c] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i < n) {
      v[c] = *(const float4 *)(xr + i);
      if (rr) {
        const float4 a = *(const float4 *)(rr + i);
        v[c].x += a.x;
        v[c].y += a.y;
        v[c].z += a.z;
        v[c].w += a.w;
        *(float4 *)(xr + i) = v[c];
      }
    }
    ss += v[c].x * v[c].x + v[c].y * v[c].y + v[c].z * v[c].z + v[c].w * v[c].w;
  }
  for (int i = 4 * (R * kNormThreads + threadIdx.x); i < n; i += 4 * kNormThreads) {
    float4 a = *(const float4 *)(xr + i);
    if (rr) {
      const float4 b = *(const float4 *)(rr + i);
      a.x += b.x;
      a.y += b.y;
      a.z += b.z;
      a.w += b.w;
      *(float4 *)(xr + i) = a;
    }
    ss += a.x * a.x + a.y * a.y + a.z * a.z + a.w * a.w;
  }
  const float inv = 1.0f / sqrtf(block_sum(ss, red) / (float)n + eps);
#pragma unroll
  for (int c = 0; c < R; ++c) {
    const int i = 4 * (c * kNormThreads + threadIdx.x);
    if (i < n) {
      const float4 g = *(const float4 *)(w + i);
      *(float4 *)(yr + i) = make_float4(v[c].x * inv * g.x, v[c].y * inv * g.y,
                                        v[c].z * inv * g.z, v[c].w * inv * g.w);
    }
  }
  for (int i = 4 * (R * kNormThreads + threadIdx.x); i < n; i += 4 * kNormThreads) {
    const float4 a = *(const float4 *)(xr + i), g = *(const float4 *)(w + i);
    *(float4 *)(yr + i) = make_float4(a.x * inv * g.x, a.y * inv * g.y, a.z * inv * g.z,
                                      a.w * inv * g.w);
  }
}

// out[i] = up[i] * silu(gate[i]) for a row [gate (ffn) | up (ffn)]
// (elementwise.wgsl:96-102 with a = up, b = gate).
__global__ __launch_bounds__(kGlueThreads) void swiglu_kernel(const float *__restrict__ gu,
                                                              float *__restrict__ out, int ffn) {
  const float *g = gu + (int64_t)blockIdx.y * 2 * ffn, *u = g + ffn;
  float *o = out + (int64_t)blockIdx.y * ffn;
  const int i = 4 * (blockIdx.x * kGlueThreads + threadIdx.x);
  if (i >= ffn) return;
  const float4 a = *(const float4 *)(g + i), b = *(const float4 *)(u + i);
  *(float4 *)(o + i) = make_float4(b.x * (a.x / (1.0f + expf(-a.x))), b.y * (a.y / (1.0f + expf(-a.y))),
                                   b.z * (a.z / (1.0f + expf(-a.z))), b.w * (a.w / (1.0f + expf(-a.w))));
}

// Decode attention in one launch, flash-decoding style.  Workgroup (g, sp)
// takes KV head g and cache slots [64 sp, 64 sp + 64) of the causal range
// 0..p, p = *pos; the n = ceil((p + 1) / 64) workgroups of the range take
// part and the others exit.  The workgroup whose range holds p writes slot p
// (k after rotate_half RoPE, v as is) into the cache.
//
// Every global load of a workgroup (its K / V rows, the new k / v, the first
// query row of each wave, the RoPE rows) is issued before any is consumed,
// so the whole input arrives in one latency round.  The K / V rows are
// staged in LDS (K rows at a stride of HD + 4 floats, so that lane t reading
// row t is free of bank conflicts); wave w takes query heads w, w + 4, ...:
// lane t owns slot t0 + t, a wave computes 64 dot products, one wave-wide
// softmax reduction and sum_t p_t v_t reading V rows from LDS.
//
// With n = 1 the workgroup writes the output.  Otherwise it writes its
// partial-softmax record per query head (layout and merge rule next to
// kAttnSplit), and the last of the n workgroups to finish -- an atomic
// counter per KV head, kept in the workspace and left at zero -- merges the n
// records in split order, so the result does not depend on which workgroup
// finishes last.  With out == nullptr every workgroup writes its records and
// nothing is merged: the consumer (the output projection's merge prologue)
// merges them with the same arithmetic.
constexpr int kSplit = kAttnSplit;

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

template <int HD>
__global__ __launch_bounds__(kGlueThreads) void attention_kernel(
    const float *__restrict__ qkv, const int64_t *__restrict__ pos, const float *__restrict__ cs,
    const float *__restrict__ sn, float *__restrict__ kc, float *__restrict__ vc,
    float *__restrict__ out, float *__restrict__ work, unsigned *__restrict__ counters, int nh,
    int nkv, int max_seq) {
  constexpr int half = HD / 2, KLD = HD + 4, C4 = HD / 4;
  constexpr int KV4 = kSplit * C4 / kGlueThreads;  // float4 of K (and of V) per thread
  constexpr int QR = (half + 63) / 64;             // query element pairs per lane
  // K / V rows; row kSplit is a pad that takes the stores of rows outside the range
  __shared__ __align__(16) float ks[(kSplit + 1) * KLD];
  __shared__ __align__(16) float vs[(kSplit + 1) * HD];
  __shared__ __align__(16) float qw[4 * HD];       // per wave: roped, scaled query
  __shared__ float pw[4 * kSplit];                  // per wave: probabilities
  __shared__ int merge;
  const int grp = nh / nkv, g = blockIdx.x, sp = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int S = gridDim.y;
  const int64_t p64 = pos[0];
  if (p64 < 0 || p64 >= max_seq) return;  // no cache slot: write nothing
  const int p = (int)p64, T = p + 1, t0 = sp * kSplit;
  if (t0 >= T) return;                     // beyond the causal range
  const int n = (T + kSplit - 1) / kSplit;
  const int tn = min(kSplit, T - t0);
  const int tp = p - t0;                   // row of slot p in this block when < kSplit
  const bool holds_p = tp < kSplit;
  const bool rec_only = out == nullptr;
  constexpr int RS = attn_record_stride(HD);
  float *kbase = kc + (int64_t)g * max_seq * HD, *vbase = vc + (int64_t)g * max_seq * HD;
  const float *crow = cs + (int64_t)p * half, *srow = sn + (int64_t)p * half;

  // 1. all global loads, straight-line: a row outside [t0, t0 + tn) or slot p
  // (written below) reads row t0 instead (always a valid slot) into the pad
  float4 kr[KV4], vr[KV4];
#pragma unroll
  for (int i = 0; i < KV4; ++i) {
    const int e = tid + i * kGlueThreads, t = e / C4, c = e - t * C4;
    const int row = (t < tn && t != tp) ? t0 + t : t0;
    kr[i] = *(const float4 *)(kbase + (int64_t)row * HD + 4 * c);
    vr[i] = *(const float4 *)(vbase + (int64_t)row * HD + 4 * c);
  }
  const int j0 = wave;
  float qa[QR], qb[QR], qc[QR], qs[QR];
  if (j0 < grp) {
    const float *qin = qkv + (int64_t)(g * grp + j0) * HD;
#pragma unroll
    for (int r = 0; r < QR; ++r) {
      const int i = lane + 64 * r;
      if (i < half) {
        qa[r] = qin[i];
        qb[r] = qin[i + half];
        qc[r] = crow[i];
        qs[r] = srow[i];
      }
    }
  }
  float ka = 0.f, kb = 0.f, kcs = 0.f, ksn = 0.f, vv = 0.f;
  if (holds_p) {
    const float *kin = qkv + (int64_t)nh * HD + g * HD;
    const float *vin = qkv + (int64_t)(nh + nkv) * HD + g * HD;
    if (tid < half) {
      ka = kin[tid];
      kb = kin[tid + half];
      kcs = crow[tid];
      ksn = srow[tid];
    }
    if (tid < HD) vv = vin[tid];
  }

  // keep the loads above ahead of every use below (the scheduler would
  // otherwise sink each load to its store and serialize the round trips)
  __builtin_amdgcn_sched_barrier(0);

  // 2. LDS: the block's K / V rows, slot p (rotate_half RoPE of k, rope.wgsl:1-10;
  // also into the caches) and each wave's first roped, scaled query
#pragma unroll
  for (int i = 0; i < KV4; ++i) {
    const int e = tid + i * kGlueThreads, t = e / C4, c = e - t * C4;
    const int st = (t < tn && t != tp) ? t : kSplit;
    *(float4 *)(ks + st * KLD + 4 * c) = kr[i];
    *(float4 *)(vs + st * HD + 4 * c) = vr[i];
  }
  if (holds_p) {
    float *krow = kbase + (int64_t)p * HD, *vrow = vbase + (int64_t)p * HD;
    if (tid < half) {
      const float k0 = ka * kcs - kb * ksn, k1 = kb * kcs + ka * ksn;
      krow[tid] = k0;
      krow[tid + half] = k1;
      ks[tp * KLD + tid] = k0;
      ks[tp * KLD + tid + half] = k1;
    }
    if (tid < HD) {
      vrow[tid] = vv;
      vs[tp * HD + tid] = vv;
    }
  }
  const float scale = 1.0f / sqrtf((float)HD);
  float *q = qw + wave * HD;
  if (j0 < grp) {
#pragma unroll
    for (int r = 0; r < QR; ++r) {
      const int i = lane + 64 * r;
      if (i < half) {
        q[i] = (qa[r] * qc[r] - qb[r] * qs[r]) * scale;
        q[i + half] = (qb[r] * qc[r] + qa[r] * qs[r]) * scale;
      }
    }
  }
  __syncthreads();

  // 3. per query head: scores, softmax, sum p v
  float *pr = pw + wave * kSplit;
  for (int j = j0; j < grp; j += 4) {
    if (j != j0) {  // later heads of a group larger than four: rope this query now
      const float *qin = qkv + (int64_t)(g * grp + j) * HD;
      for (int i = lane; i < half; i += 64) {
        const float c = crow[i], sv = srow[i], a = qin[i], b = qin[i + half];
        q[i] = (a * c - b * sv) * scale;
        q[i + half] = (b * c + a * sv) * scale;
      }
    }
    // the wave's own LDS writes are visible to it in program order
    float sc = -INFINITY;
    if (lane < tn) {
      const float *kr_ = ks + lane * KLD;
      float a0 = 0.f, a1 = 0.f;
#pragma unroll
      for (int c = 0; c < C4; c += 2) {
        const float4 k0 = *(const float4 *)(kr_ + 4 * c), q0 = *(const float4 *)(q + 4 * c);
        const float4 k1 = *(const float4 *)(kr_ + 4 * c + 4), q1 = *(const float4 *)(q + 4 * c + 4);
        a0 += q0.x * k0.x + q0.y * k0.y + q0.z * k0.z + q0.w * k0.w;
        a1 += q1.x * k1.x + q1.y * k1.y + q1.z * k1.z + q1.w * k1.w;
      }
      sc = a0 + a1;
    }
    const float m = wave_max(sc);
    const float e = lane < tn ? expf(sc - m) : 0.f;
    const float l = wave_sum(e);
    pr[lane] = e;
    const bool direct = n == 1 && !rec_only;
    float *rec = work + ((int64_t)(g * S + sp) * grp + j) * RS;
    float *o_out = direct ? out + (int64_t)(g * grp + j) * HD : rec;
    const float inv = direct ? 1.0f / l : 1.0f;
    for (int i = lane; i < HD; i += 64) {
      float o = 0.f;
#pragma unroll 8
      for (int t = 0; t < tn; ++t) o += pr[t] * vs[t * HD + i];
      o_out[i] = o * inv;
    }
    if (!direct && lane == 0) {
      rec[HD] = m;
      rec[HD + 1] = l;
    }
  }
  if (n == 1 || rec_only) return;

  // 4. the last of the n workgroups of KV head g merges the records
  __threadfence();  // this workgroup's records are visible before it is counted
  __syncthreads();
  if (tid == 0) merge = atomicAdd(counters + g, 1u) == (unsigned)(n - 1);
  __syncthreads();
  if (!merge) return;
  __threadfence();  // every other workgroup's records are visible to the merge
  // wave w merges query heads w, w + 4, ...: lane s reads record s's (m, l),
  // so a chunk of 64 records costs one load round, and the weighted sums of
  // the outputs issue their loads together.  L and the outputs accumulate in
  // split order, as the merge prologue of the output projection does.
  constexpr int QO = HD / 64;  // outputs per lane
  const int64_t stride = (int64_t)grp * RS;
  float *pl = ks;  // the K rows are consumed: per wave, the 64 (w_s, l_s) of a chunk
  for (int j = wave; j < grp; j += 4) {
    const float *base = work + ((int64_t)g * S * grp + j) * RS;
    float M = -INFINITY;
    for (int s0 = 0; s0 < n; s0 += 64)
      if (s0 + lane < n) M = fmaxf(M, base[(s0 + lane) * stride + HD]);
    M = wave_max(M);
    float L = 0.f, o[QO];
#pragma unroll
    for (int r = 0; r < QO; ++r) o[r] = 0.f;
    for (int s0 = 0; s0 < n; s0 += 64) {
      float w = 0.f, lv = 0.f;
      if (s0 + lane < n) {
        const float *rec = base + (s0 + lane) * stride;
        w = expf(rec[HD] - M);
        lv = rec[HD + 1];
      }
      pr[lane] = w;  // wave-local: read back in program order
      pl[wave * 64 + lane] = lv;
      const int cnt = min(64, n - s0);
#pragma unroll 8
      for (int u = 0; u < cnt; ++u) {
        const float wu = pr[u];
        L = fmaf(wu, pl[wave * 64 + u], L);
        const float *ro = base + (s0 + u) * stride + lane;
#pragma unroll
        for (int r = 0; r < QO; ++r) o[r] = fmaf(wu, ro[64 * r], o[r]);
      }
    }
    const float inv = 1.0f / L;
#pragma unroll
    for (int r = 0; r < QO; ++r) out[(int64_t)(g * grp + j) * HD + lane + 64 * r] = o[r] * inv;
  }
  if (tid == 0) counters[g] = 0u;  // ready for the next call
}

// ---------------------------------------------------------------------------
// Prefill attention: M new positions, two launches.
//
// rope_append_kernel: one workgroup per row m.  It applies rotate_half RoPE
// (rope.wgsl:1-10, the same products as the decode kernel) to the row's k
// heads and stores k and v at slot pos[m] of the caches.  A row whose position
// lies outside 0..max_seq-1 writes nothing.
//
// attention_prefill_kernel: causal GQA attention of each row over slots
// 0..pos[m] (attention.wgsl:60-234 with new_seq_len = M), flash-style, in f32
// grade on the f16 matrix cores: an f32 operand, scaled by a power of two,
// enters as f16 hi + lo (22 significant bits) and a product is hi hi + hi lo +
// lo hi, accumulated in f32.
// - A wave takes 32 rows of one query head; a workgroup takes four consecutive
//   (32-row block, head of the group) pairs of one KV head, so that groups of
//   any size fill it.  Blocks are launched last rows first (the longest causal
//   ranges), KV head fastest: with 8 KV heads each XCD keeps one head's K and V
//   in its L2.
// - Keys come in tiles of KT slots.  Wave w converts the w-th quarter (group) of
//   the tile, each group with a power of two of their own (K and V apart), so
//   the conversion needs no cross-wave maximum.  K rows and transposed V rows,
//   hi and lo, are stored in LDS, rows padded by 16 bytes: every fragment read
//   is one base register and an immediate, free of bank conflicts.
// - Two barriers per tile: V's loads are in flight under S = K Q, the next K's
//   under O += V P, so a wave holds one operand's 8 float4 at a time.
// - S^T = K . Q^T (keys x rows): in the 32x32x16 accumulator, lane l holds keys
//   8 (r / 4) + 4 (l / 32) + r % 4 of row l % 32.  V^T is stored with the middle
//   two of each four 4-key blocks exchanged, so that those registers, converted
//   to f16, are the B operand of O^T += V^T . P^T: the probabilities never
//   leave their lane.
// - log2 e is folded into the score factor; the running maximum is rounded up
//   to an integer, so a rescale is by an exact power of two, and it is skipped
//   while no row's maximum moved.
// What bounds it: the vector work of the conversion and the softmax beside the
// matrix cores' three products (per 64 keys and 32 rows about 3900 cycles of VALU
// issue against 3072 of MFMA), and few workgroups.  Against the v_mfma f32 kernel
// it replaces (16 rows per wave, f32 K / V tiles): 1500 rows over 548 cached, 32 / 8
// heads of 128, 584 -> 158 us with the append; 500 rows over 1500, 8 / 2 heads of
// 64 / 128 / 256, 119 -> 85, 218 -> 134, 417 -> 273; 8 rows over 700, 83 -> 54.  The
// error against float64 fell from 7.2e-7 to 4.6e-7 there (fewer, longer f32
// accumulation steps), and is no larger at any of 37 shapes tried.
// A row whose position lies outside 0..max_seq-1, or past M, attends to
// nothing and is not written.
constexpr int kPfRows = 32;   // rows (positions) per wave
constexpr int kPfWaves = 4;   // (row block, head) pairs per workgroup
// key slots per tile, a quarter of them per wave
template <int HD>
constexpr int pf_keys() { return HD <= 128 ? 64 : 32; }

typedef float float16_t __attribute__((ext_vector_type(16)));

template <int HD>
__global__ __launch_bounds__(kGlueThreads) void rope_append_kernel(
    const float *__restrict__ qkv, int64_t ldq, const int64_t *__restrict__ pos,
    const float *__restrict__ cs, const float *__restrict__ sn, float *__restrict__ kc,
    float *__restrict__ vc, int nh, int nkv, int max_seq) {
  constexpr int half = HD / 2;
  const int64_t m = blockIdx.x;
  const int64_t p = pos[m];
  if (p < 0 || p >= max_seq) return;
  const float *kin = qkv + m * ldq + (int64_t)nh * HD, *vin = kin + (int64_t)nkv * HD;
  const float *crow = cs + p * half, *srow = sn + p * half;
  for (int e = threadIdx.x; e < nkv * half; e += kGlueThreads) {
    const int h = e / half, i = e - h * half;
    const float a = kin[h * HD + i], b = kin[h * HD + i + half], c = crow[i], s = srow[i];
    float *krow = kc + ((int64_t)h * max_seq + p) * HD;
    krow[i] = a * c - b * s;
    krow[i + half] = b * c + a * s;
  }
  for (int e = threadIdx.x; e < nkv * HD; e += kGlueThreads) {
    const int h = e / HD, i = e - h * HD;
    vc[((int64_t)h * max_seq + p) * HD + i] = vin[h * HD + i];
  }
}

__device__ __forceinline__ float16_t mfma_h32(half8_t a, half8_t b, float16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// The power of two 2^e that brings a largest magnitude m to [2^13, 2^14), e
// clamped to +-126.
__device__ __forceinline__ int pf_exp(float m) {
  const int e = 140 - (int)((__float_as_uint(m) >> 23) & 255u);
  return max(-126, min(126, e));
}
__device__ __forceinline__ float pf_pow2(int e) {  // 2^e, |e| <= 126
  return __uint_as_float((uint32_t)(e + 127) << 23);
}

// f16 hi + lo parts of eight f32 values times sc
__device__ __forceinline__ void pf_split(const float *x, float sc, half8_t &hi, half8_t &lo) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float v = x[i] * sc;
    asm("" : "+v"(v));  // one product for both parts (else it is folded into each conversion)
    const half_t h = (half_t)v;
    hi[i] = h;
    lo[i] = (half_t)(v - (float)h);
  }
}

// Largest finite magnitude of a wave's n values (an infinity must not take the
// scale from the finite values of its group; NaN never wins).
template <int N>
__device__ __forceinline__ float pf_wave_absmax(const float (&x)[N]) {
  float m = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) m = fmaxf(m, fabsf(x[i]));
  m = max_xor32(max_xor16(max_lanes16(m)));
  if (__builtin_amdgcn_readfirstlane(__float_as_uint(m)) == 0x7f800000u) {
    m = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i) m = fmaxf(m, fabsf(x[i]) < INFINITY ? fabsf(x[i]) : 0.f);
    m = max_xor32(max_xor16(max_lanes16(m)));
  }
  return m;
}

// A wave's 32 query rows of one head, roped and split: qh / ql[s] = the f16 hi /
// lo parts of elements 16 s + 8 (lane / 32) + 0..7 of row lane % 32, times 2^eq
// (the row's own exponent).  Returns log2 e / sqrt(HD) * 2^-eq.  A row is read by
// HD / 8 lanes side by side (a lane per row would read 32 lines per load) and
// turned through the wave's part of LDS, ROWS rows at a time.  `my`: the lane's row's position, or -1 (zeros).
template <int HD>
struct PfQuery {
  static constexpr int LPR = HD / 8, RPG = 64 / LPR;   // lanes per row, rows per load
  static constexpr int ROWS = HD <= 128 ? 32 : 16;     // rows per pass
  static constexpr int RB = 2 * HD + 16, BYTES = 2 * ROWS * RB;
};

template <int HD>
__device__ __forceinline__ float pf_query(const float *__restrict__ qrows, int64_t ldq,
                                          const float *__restrict__ cs,
                                          const float *__restrict__ sn, int my, unsigned char *buf,
                                          half8_t (&qh)[HD / 16], half8_t (&ql)[HD / 16]) {
  using Q = PfQuery<HD>;
  constexpr int half = HD / 2, NG = Q::ROWS / Q::RPG;
  const int lane = threadIdx.x & 63, col = lane & 31, hf = lane >> 5;
  const int i = 4 * (lane % Q::LPR);
  int eq = 0;
  if (Q::ROWS < kPfRows) {  // a pass without rows is left out
#pragma unroll
    for (int k = 0; k < HD / 16; ++k)
#pragma unroll
      for (int e = 0; e < 8; ++e) qh[k][e] = ql[k][e] = (half_t)0.f;
  }
#pragma unroll
  for (int r0 = 0; r0 < kPfRows; r0 += Q::ROWS) {
    if (Q::ROWS < kPfRows && !__any(my >= 0 && col / Q::ROWS * Q::ROWS == r0)) continue;
    float4 a[NG], b[NG], c[NG], s[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int row = r0 + g * Q::RPG + lane / Q::LPR, p = __shfl(my, row);
      a[g] = b[g] = c[g] = s[g] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (p >= 0) {
        const float *q = qrows + row * ldq + i;
        a[g] = *(const float4 *)q;
        b[g] = *(const float4 *)(q + half);
        c[g] = *(const float4 *)(cs + (int64_t)p * half + i);
        s[g] = *(const float4 *)(sn + (int64_t)p * half + i);
      }
    }
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int row = g * Q::RPG + lane / Q::LPR;
      float x[8] = {a[g].x * c[g].x - b[g].x * s[g].x, a[g].y * c[g].y - b[g].y * s[g].y,
                    a[g].z * c[g].z - b[g].z * s[g].z, a[g].w * c[g].w - b[g].w * s[g].w,
                    b[g].x * c[g].x + a[g].x * s[g].x, b[g].y * c[g].y + a[g].y * s[g].y,
                    b[g].z * c[g].z + a[g].z * s[g].z, b[g].w * c[g].w + a[g].w * s[g].w};
      float mx = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(x[e]));
      mx = fmaxf(mx, dpp<kDppXor1>(mx));
      mx = fmaxf(mx, dpp<kDppXor2>(mx));
      mx = fmaxf(mx, dpp<kDppHalfMirror>(mx));
      if (Q::LPR >= 16) mx = fmaxf(mx, dpp<kDppMirror>(mx));
      if (Q::LPR >= 32) mx = max_xor16(mx);
      const int e2 = pf_exp(mx);
      half8_t h, l;
      pf_split(x, pf_pow2(e2), h, l);
      unsigned char *at = buf + row * Q::RB + 2 * i;
      *(half4_t *)at = half4_t{h[0], h[1], h[2], h[3]};
      *(half4_t *)(at + HD) = half4_t{h[4], h[5], h[6], h[7]};
      at += Q::ROWS * Q::RB;
      *(half4_t *)at = half4_t{l[0], l[1], l[2], l[3]};
      *(half4_t *)(at + HD) = half4_t{l[4], l[5], l[6], l[7]};
      if (lane % Q::LPR == 0) *(int *)(buf + row * Q::RB + 2 * HD) = e2;  // in the row's pad
    }
    // the wave's own LDS writes are visible to it in program order
    if (Q::ROWS == kPfRows || col / Q::ROWS * Q::ROWS == r0) {
      const unsigned char *at = buf + (col - r0) * Q::RB;
      eq = *(const int *)(at + 2 * HD);
#pragma unroll
      for (int k = 0; k < HD / 16; ++k) {
        qh[k] = *(const half8_t *)(at + 32 * k + 16 * hf);
        ql[k] = *(const half8_t *)(at + Q::ROWS * Q::RB + 32 * k + 16 * hf);
      }
    }
  }
  return 1.44269504088896340736f / sqrtf((float)HD) * pf_pow2(-eq);
}

template <int HD>
__global__ __launch_bounds__(64 * kPfWaves, HD <= 128 ? 2 : 1) void attention_prefill_kernel(
    const float *__restrict__ qkv, int64_t ldq, const int64_t *__restrict__ pos, int64_t M,
    const float *__restrict__ cs, const float *__restrict__ sn, const float *__restrict__ kc,
    const float *__restrict__ vc, float *__restrict__ out, int64_t ldo, int nh, int nkv,
    int max_seq) {
  constexpr int KS = HD / 16;                 // k steps of S
  constexpr int DT = HD / 32;                 // 32-wide output tiles
  constexpr int KT = pf_keys<HD>(), GK = KT / kPfWaves;  // keys per tile, per wave's group
  constexpr int JT = KT / 32;                 // 32-key score tiles
  constexpr int KRB = 2 * HD + 16, VRB = 2 * KT + 16;  // bytes of a K row and of a V^T row in LDS
  constexpr int KI = GK * HD / 8 / 64;        // 8-element chunks of K per lane
  constexpr int NB = GK / 4;                  // 4-key blocks of a group
  constexpr int VI = NB * HD / 4 / 64;        // 4 x 4 blocks of V per lane
  constexpr int CPR = HD / 8;                 // chunks per K row
  __shared__ __align__(16) unsigned char lds[2 * KT * KRB + 2 * HD * VRB];
  unsigned char *const kh = lds, *const kl = kh + KT * KRB;
  unsigned char *const vh = kl + KT * KRB, *const vl = vh + HD * VRB;
  __shared__ int kex[kPfWaves], vex[kPfWaves], kends[kPfWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 31, hf = lane >> 5;  // MFMA column (row of the block), k half
  const int grp = nh / nkv, kvh = blockIdx.x;
  const int64_t unit = (int64_t)(gridDim.y - 1 - blockIdx.y) * kPfWaves + wave;
  const int64_t rb = unit / grp;
  const int jh = (int)(unit - rb * grp);
  const int64_t m = rb * kPfRows + col;
  int my = -1;  // the row's position; -1: attends to nothing, not written
  if (m < M) {
    const int64_t p = pos[m];
    if (p >= 0 && p < max_seq) my = (int)p;
  }
  // slots 0 .. wend - 1 hold every key of the wave's rows, slots up to wlo are
  // seen by all of them
  int wend = my + 1, wlo = my >= 0 ? my : INT_MAX;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    wend = max(wend, __shfl_xor(wend, o));
    wlo = min(wlo, __shfl_xor(wlo, o));
  }
  if (lane == 0) kends[wave] = wend;
  __syncthreads();
  int kend = 0;
#pragma unroll
  for (int w = 0; w < kPfWaves; ++w) kend = max(kend, kends[w]);
  kend = __builtin_amdgcn_readfirstlane(kend);
  wend = __builtin_amdgcn_readfirstlane(wend);
  wlo = __builtin_amdgcn_readfirstlane(wlo);
  if (kend == 0) return;  // the whole workgroup: no row attends to anything
  const int ntile = (kend + KT - 1) / KT;
  const float *kbase = kc + (int64_t)kvh * max_seq * HD;
  const float *vbase = vc + (int64_t)kvh * max_seq * HD;
  // wave w's share of a tile: keys GK w + ..; a slot past the last key re-reads
  // that key (its score is masked, its probability 0)
  float kr[8 * KI];
  auto load_k = [&](int t0) {
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      const int f = i * 64 + lane, t = GK * wave + f / CPR, c = f % CPR;
      const float *src = kbase + (int64_t)min(t0 + t, kend - 1) * HD + 8 * c;
      *(float4 *)(kr + 8 * i) = *(const float4 *)src;
      *(float4 *)(kr + 8 * i + 4) = *(const float4 *)(src + 4);
    }
  };
  auto store_k = [&]() {
    const int e = pf_exp(pf_wave_absmax(kr));
    if (lane == 0) kex[wave] = e;
    const float sc = pf_pow2(e);
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      const int f = i * 64 + lane, t = GK * wave + f / CPR, c = f % CPR;
      half8_t h, l;
      pf_split(kr + 8 * i, sc, h, l);
      const int at = t * KRB + 16 * c;
      *(half8_t *)(kh + at) = h;
      *(half8_t *)(kl + at) = l;
    }
  };
  // V: 4 keys x 4 elements per block, transposed in registers
  auto load_v = [&](int t0) {
#pragma unroll
    for (int i = 0; i < VI; ++i) {
      const int b = NB * wave + lane % NB, c = lane / NB + 64 / NB * i;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *(float4 *)(kr + 16 * i + 4 * e) =
            *(const float4 *)(vbase + (int64_t)min(t0 + 4 * b + e, kend - 1) * HD + 4 * c);
    }
  };
  auto store_v = [&]() {
    const int e = pf_exp(pf_wave_absmax(kr));
    if (lane == 0) vex[wave] = e;
    const float sc = pf_pow2(e);
#pragma unroll
    for (int i = 0; i < VI; ++i) {
      const int b = NB * wave + lane % NB, c = lane / NB + 64 / NB * i;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        half4_t h, l;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float v = kr[16 * i + 4 * k + d] * sc;
          asm("" : "+v"(v));
          h[k] = (half_t)v;
          l[k] = (half_t)(v - (float)h[k]);
        }
        const int at = (4 * c + d) * VRB + 32 * (b >> 2) + 16 * (b & 1) + 8 * ((b >> 1) & 1);
        *(half4_t *)(vh + at) = h;
        *(half4_t *)(vl + at) = l;
      }
    }
  };

  load_k(0);  // in flight under the query's loads
  half8_t qh[KS], ql[KS];
  const float qf = pf_query<HD>(qkv + rb * kPfRows * ldq + (int64_t)(kvh * grp + jh) * HD, ldq, cs,
                                sn, my, kh + wave * PfQuery<HD>::BYTES, qh, ql);
  static_assert(kPfWaves * PfQuery<HD>::BYTES <= 2 * KT * KRB + 2 * HD * VRB, "fits in the tile");
  __syncthreads();  // the queries' staging is read: the tile may be written
  float16_t o[DT];
#pragma unroll
  for (int a = 0; a < DT; ++a)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[a][r] = 0.f;
  float mrun = -INFINITY, lrun = 0.f;
  int evrun = 126, evmin = 126;  // exponent of the accumulator's V, smallest so far

  store_k();
  for (int it = 0; it < ntile; ++it) {
    const int t0 = it * KT;
    const bool act = t0 < wend;  // wave-uniform
    __syncthreads();             // K of this tile stored, V of the previous one read
    load_v(t0);
    float16_t s[JT];
    float alpha = 1.f;
    if (act) {
      const unsigned char *kp = kh + col * KRB + 16 * hf, *kq = kl + col * KRB + 16 * hf;
      half8_t ah = *(const half8_t *)kp, al = *(const half8_t *)kq;
#pragma unroll
      for (int n = 0; n < JT * KS; ++n) {  // the next fragments are read ahead of the MFMAs
        const int j = n / KS, k = n % KS, n1 = n + 1 < JT * KS ? n + 1 : n;
        const int at = 32 * (n1 / KS) * KRB + 32 * (n1 % KS);
        const half8_t bh = *(const half8_t *)(kp + at), bl = *(const half8_t *)(kq + at);
        if (k == 0)
#pragma unroll
          for (int r = 0; r < 16; ++r) s[j][r] = 0.f;
        s[j] = mfma_h32(al, qh[k], s[j]);
        s[j] = mfma_h32(ah, ql[k], s[j]);
        s[j] = mfma_h32(ah, qh[k], s[j]);
        ah = bh;
        al = bl;
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x8, 3, 0);
      }
      // score factors of the tile's key groups, kept normal (a masked -inf
      // times 0 would be NaN)
      float f[kPfWaves];
#pragma unroll
      for (int g = 0; g < kPfWaves; ++g)
        f[g] = fminf(fmaxf(qf * pf_pow2(-kex[g]), 0x1p-126f), 0x1p126f);
      if (t0 + KT - 1 > wlo) {  // some row does not see the whole tile
#pragma unroll
        for (int j = 0; j < JT; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (t0 + 32 * j + 8 * (r >> 2) + 4 * hf + (r & 3) > my) s[j][r] = -INFINITY;
      }
      float bm = -INFINITY;
#pragma unroll
      for (int j = 0; j < JT; ++j)
#pragma unroll
        for (int r = 0; r < 16; r += 4)
          bm = fmaxf(bm, fmaxf(fmaxf(s[j][r], s[j][r + 1]), fmaxf(s[j][r + 2], s[j][r + 3])) *
                             f[(32 * j + 2 * r) / GK]);
      bm = max_xor32(bm);
      const float mnew = fmaxf(mrun, ceilf(bm));
      const float mu = mnew == -INFINITY ? 0.f : mnew;
      alpha = __builtin_amdgcn_exp2f(mrun - mu);  // an exact power of two, 0 at the start
      mrun = mnew;
      float ls = 0.f;
#pragma unroll
      for (int j = 0; j < JT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float e = __builtin_amdgcn_exp2f(fmaf(s[j][r], f[(32 * j + 8 * (r >> 2)) / GK], -mu));
          s[j][r] = e;
          ls += e;
        }
      lrun = fmaf(lrun, alpha, ls);
    }
    store_v();
    __syncthreads();  // V stored, every wave is done with K
    if (it + 1 < ntile) load_k(t0 + KT);
    if (act) {
      // the accumulator's scale follows V's: down at once when a group holds
      // larger values, up once all are 2^8 smaller (never above 2^60 of the
      // largest seen, so that it cannot overflow)
      int emin = vex[0];
#pragma unroll
      for (int g = 1; g < kPfWaves; ++g) emin = min(emin, vex[g]);
      emin = __builtin_amdgcn_readfirstlane(emin);
      evmin = min(evmin, emin);
      const int en = emin < evrun || emin > evrun + 8 ? min(emin, evmin + 60) : evrun;
      const float rs = ldexpf(alpha, en - evrun);  // exact; 0 at the wave's first tile
      evrun = en;
      if (__any(rs != 1.f)) {
#pragma unroll
        for (int a = 0; a < DT; ++a)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[a][r] *= rs;
      }
      float pf[kPfWaves];
#pragma unroll
      for (int g = 0; g < kPfWaves; ++g)
        pf[g] = ldexpf(0x1p15f, evrun - __builtin_amdgcn_readfirstlane(vex[g]));
      const unsigned char *vp = vh + col * VRB + 16 * hf, *vq = vl + col * VRB + 16 * hf;
      half8_t bh = *(const half8_t *)vp, bl = *(const half8_t *)vq;
      half8_t ph[2], pl[2];
      // probabilities times 2^(15 + evrun - vex) <= 2^15: each group's V has its own exponent
      auto split_p = [&](int g) {
        float p[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
          p[i] = s[g >> 1][8 * (g & 1) + i] * pf[(16 * g + 8 * (i >> 2)) / GK];
        pf_split(p, 1.f, ph[g & 1], pl[g & 1]);
      };
      split_p(0);
#pragma unroll
      for (int n = 0; n < KT / 16 * DT; ++n) {
        const int g = n / DT, a = n % DT, n1 = n + 1 < KT / 16 * DT ? n + 1 : n;
        const int at = 32 * (n1 % DT) * VRB + 32 * (n1 / DT);
        const half8_t ch = *(const half8_t *)(vp + at), cl = *(const half8_t *)(vq + at);
        if (a == 0 && g + 1 < KT / 16) split_p(g + 1);
        o[a] = mfma_h32(bl, ph[g & 1], o[a]);
        o[a] = mfma_h32(bh, pl[g & 1], o[a]);
        o[a] = mfma_h32(bh, ph[g & 1], o[a]);
        bh = ch;
        bl = cl;
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);
        }
      }
    }
    if (it + 1 < ntile) store_k();
  }
  float l = lrun + __shfl_xor(lrun, 32);
  if (my >= 0) {
    const float inv = 1.0f / l;
    float *orow = out + m * ldo + (int64_t)(kvh * grp + jh) * HD + 4 * hf;
#pragma unroll
    for (int a = 0; a < DT; ++a)
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        *(float4 *)(orow + 32 * a + 2 * r) = make_float4(
            ldexpf(o[a][r] * inv, -15 - evrun), ldexpf(o[a][r + 1] * inv, -15 - evrun),
            ldexpf(o[a][r + 2] * inv, -15 - evrun), ldexpf(o[a][r + 3] * inv, -15 - evrun));
  }
}

// Argmax, pass 1: workgroup b scans a contiguous chunk and writes its (value,
// index) with the first index on ties and NaN never winning; pass 2 (one
// workgroup) merges the partials the same way.
constexpr int kArgBlocks = 256;

__device__ __forceinline__ void better(float &v, int64_t &i, float ov, int64_t oi) {
  if (ov > v || (ov == v && oi < i)) {
    v = ov;
    i = oi;
  }
}

__device__ __forceinline__ void block_argmax(float &v, int64_t &idx, float *bv, int64_t *bi) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) better(v, idx, __shfl_xor(v, o), __shfl_xor(idx, o));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    bv[wave] = v;
    bi[wave] = idx;
  }
  __syncthreads();
  if (threadIdx.x == 0)
    for (int w2 = 1; w2 < (int)(blockDim.x >> 6); ++w2) better(v, idx, bv[w2], bi[w2]);
}

__global__ __launch_bounds__(kGlueThreads) void argmax_partial_kernel(const float *__restrict__ x,
                                                                      int64_t n,
                                                                      float *__restrict__ pv,
                                                                      int64_t *__restrict__ pi) {
  __shared__ float bv[kGlueThreads / 64];
  __shared__ int64_t bi[kGlueThreads / 64];
  const int64_t chunk = (n + kArgBlocks - 1) / kArgBlocks;
  const int64_t lo = (int64_t)blockIdx.x * chunk, hi = min(n, lo + chunk);
  float v = -INFINITY;
  int64_t idx = INT64_MAX;  // no candidate yet
  for (int64_t i = lo + threadIdx.x; i < hi; i += kGlueThreads) better(v, idx, x[i], i);
  block_argmax(v, idx, bv, bi);
  if (threadIdx.x == 0) {
    pv[blockIdx.x] = v;
    pi[blockIdx.x] = idx;
  }
}

__global__ __launch_bounds__(kGlueThreads) void argmax_merge_kernel(const float *__restrict__ pv,
                                                                    const int64_t *__restrict__ pi,
                                                                    int64_t *__restrict__ out) {
  __shared__ float bv[kGlueThreads / 64];
  __shared__ int64_t bi[kGlueThreads / 64];
  float v = -INFINITY;
  int64_t idx = INT64_MAX;
  for (int b = threadIdx.x; b < kArgBlocks; b += kGlueThreads) better(v, idx, pv[b], pi[b]);
  block_argmax(v, idx, bv, bi);
  if (threadIdx.x == 0) out[0] = idx == INT64_MAX ? 0 : idx;
}

}  // namespace

hipError_t launch_rmsnorm(float *x, const float *r, const float *w, float eps, float *y,
                          int64_t rows, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(rmsnorm_kernel, dim3((unsigned)rows), dim3(kNormThreads), 0, s, x, r, w, eps,
                     y, (int)n);
  return hipGetLastError();
}

hipError_t launch_swiglu(const float *gu, float *out, int64_t rows, int64_t ffn, hipStream_t s) {
  const unsigned bx = (unsigned)((ffn / 4 + kGlueThreads - 1) / kGlueThreads);
  hipLaunchKernelGGL(swiglu_kernel, dim3(bx, (unsigned)rows), dim3(kGlueThreads), 0, s, gu, out,
                     (int)ffn);
  return hipGetLastError();
}

// The records merged in split order, a wave per 64 columns of a query head; the
// arithmetic and order of attention_kernel's own merge (step 4), so the same bits.
// A lane holds its column of 64 records at once, requested before the position is
// known (records past the range are read and not used): one memory round trip
// for caches of up to 64 splits, one more per further 64.  A position outside the
// cache gives NaN.
// Merged in the output projection's prologue instead, every record past the chunk
// costs each of its workgroups a memory round trip: 94 splits, 4096 x 4096 Q4_K,
// 66.9 us with the projection against 7.4 + 5.6 for this kernel and the plain
// projection.  The records through LDS, 1024 threads per head: 9.3 - 10.7 us.
constexpr int kMergeRecs = 64;

template <int HD>
__global__ __launch_bounds__(64) void attn_merge_kernel(const float *__restrict__ work,
                                                        const int64_t *__restrict__ pos,
                                                        float *__restrict__ out, int grp, int S,
                                                        int max_seq) {
  constexpr int RS = attn_record_stride(HD);
  __shared__ __align__(16) float2 wl[kMergeRecs];
  const int h = blockIdx.x, c = blockIdx.y * 64 + threadIdx.x, lane = threadIdx.x;
  const int64_t stride = (int64_t)grp * RS;
  const float *base = work + ((int64_t)(h / grp) * S * grp + h % grp) * RS;
  float v[kMergeRecs];
  auto load = [&](int s0) {
#pragma unroll
    for (int u = 0; u < kMergeRecs; ++u) v[u] = base[min(s0 + u, S - 1) * stride + c];
  };
  float2 ml = *(const float2 *)(base + min(lane, S - 1) * stride + HD);
  load(0);
  const int64_t p = pos[0];
  const int n = (p >= 0 && p < max_seq) ? (int)(p / kSplit) + 1 : 0;
  float M = lane < n ? ml.x : -INFINITY;
  for (int r = 64 + lane; r < n; r += 64) M = fmaxf(M, base[r * stride + HD]);
  M = wave_max(M);
  float L = 0.f, o = 0.f;
  for (int s0 = 0; s0 < n; s0 += kMergeRecs) {
    if (s0 > 0) {
      ml = *(const float2 *)(base + min(s0 + lane, S - 1) * stride + HD);
      load(s0);
    }
    wl[lane] = make_float2(expf(ml.x - M), ml.y);  // wave-local: read back in program order
    const int cnt = min(kMergeRecs, n - s0);
#pragma unroll
    for (int u = 0; u < kMergeRecs; ++u) {
      if (u < cnt) {
        const float2 w = wl[u];
        L = fmaf(w.x, w.y, L);
        o = fmaf(w.x, v[u], o);
      }
    }
  }
  out[(int64_t)h * HD + c] = o * (1.0f / L);
}

// Workspace: the records [nkv][S][grp][hd + 4] floats, the merged output of
// launch_attn_merge [nh][hd] (more than kMergeChunk splits), then nkv counters.
static int64_t attention_record_bytes(int nh, int nkv, int hd, int64_t max_seq) {
  const int64_t S = (max_seq + kSplit - 1) / kSplit;
  return (int64_t)sizeof(float) * nkv * S * (nh / nkv) * attn_record_stride(hd);
}

// the counters, and all that a call with an output needs
static int64_t attention_counter_bytes(int nkv) { return ((int64_t)nkv * 4 + 15) / 16 * 16; }

int64_t attention_noalloc_bytes(int nh, int nkv, int hd, int64_t max_seq) {
  return attention_record_bytes(nh, nkv, hd, max_seq) + attention_counter_bytes(nkv);
}

int64_t attention_work_bytes(int nh, int nkv, int hd, int64_t max_seq) {
  const bool merge = (max_seq + kSplit - 1) / kSplit > kMergeChunk;  // launch_attn_merge's output
  return attention_noalloc_bytes(nh, nkv, hd, max_seq) + (merge ? (int64_t)sizeof(float) * nh * hd : 0);
}

hipError_t launch_attn_merge(const AttnRecords &ar, const float **merged, hipStream_t s) {
  float *out = (float *)((char *)ar.work +
                         attention_record_bytes(ar.nh, ar.nkv, ar.hd, ar.max_seq));
  const int S = (ar.max_seq + kSplit - 1) / kSplit, grp = ar.nh / ar.nkv;
  const dim3 grid((unsigned)ar.nh, (unsigned)(ar.hd / 64)), block(64);
  if (ar.hd == 64)
    hipLaunchKernelGGL(attn_merge_kernel<64>, grid, block, 0, s, ar.work, ar.pos, out, grp, S,
                       ar.max_seq);
  else if (ar.hd == 128)
    hipLaunchKernelGGL(attn_merge_kernel<128>, grid, block, 0, s, ar.work, ar.pos, out, grp, S,
                       ar.max_seq);
  else
    hipLaunchKernelGGL(attn_merge_kernel<256>, grid, block, 0, s, ar.work, ar.pos, out, grp, S,
                       ar.max_seq);
  *merged = out;
  return hipGetLastError();
}

static hipError_t launch_attention(const float *qkv, const int64_t *pos, const float *cs,
                                   const float *sn, float *kc, float *vc, float *out, float *work,
                                   unsigned *counters, int nh, int nkv, int hd, int64_t max_seq,
                                   hipStream_t s) {
  const int S = (int)((max_seq + kSplit - 1) / kSplit);
  const dim3 grid((unsigned)nkv, (unsigned)S), block(kGlueThreads);
  if (hd == 64)
    hipLaunchKernelGGL(attention_kernel<64>, grid, block, 0, s, qkv, pos, cs, sn, kc, vc, out,
                       work, counters, nh, nkv, (int)max_seq);
  else if (hd == 128)
    hipLaunchKernelGGL(attention_kernel<128>, grid, block, 0, s, qkv, pos, cs, sn, kc, vc, out,
                       work, counters, nh, nkv, (int)max_seq);
  else
    hipLaunchKernelGGL(attention_kernel<256>, grid, block, 0, s, qkv, pos, cs, sn, kc, vc, out,
                       work, counters, nh, nkv, (int)max_seq);
  return hipGetLastError();
}

hipError_t launch_attention_decode(const float *qkv, const int64_t *pos, const float *cs,
                                   const float *sn, float *kc, float *vc, float *out, float *work,
                                   int nh, int nkv, int hd, int64_t max_seq, hipStream_t s) {
  unsigned *counters = (unsigned *)((char *)work + attention_work_bytes(nh, nkv, hd, max_seq) -
                                    attention_counter_bytes(nkv));
  return launch_attention(qkv, pos, cs, sn, kc, vc, out, work, counters, nh, nkv, hd, max_seq, s);
}

template <int HD>
static hipError_t launch_prefill_hd(const float *qkv, int64_t ldq, const int64_t *pos, int64_t m,
                                    const float *cs, const float *sn, float *kc, float *vc,
                                    float *out, int64_t ldo, int nh, int nkv, int max_seq,
                                    hipStream_t s) {
  hipLaunchKernelGGL(rope_append_kernel<HD>, dim3((unsigned)m), dim3(kGlueThreads), 0, s, qkv,
                     ldq, pos, cs, sn, kc, vc, nh, nkv, max_seq);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int64_t units = (m + kPfRows - 1) / kPfRows * (nh / nkv);
  const dim3 grid((unsigned)nkv, (unsigned)((units + kPfWaves - 1) / kPfWaves));
  hipLaunchKernelGGL(attention_prefill_kernel<HD>, grid, dim3(64 * kPfWaves), 0, s, qkv, ldq, pos,
                     m, cs, sn, kc, vc, out, ldo, nh, nkv, max_seq);
  return hipGetLastError();
}

hipError_t launch_attention_prefill(const float *qkv, int64_t ldq, const int64_t *pos, int64_t m,
                                    const float *cs, const float *sn, float *kc, float *vc,
                                    float *out, int64_t ldo, int nh, int nkv, int hd,
                                    int64_t max_seq, hipStream_t s) {
  if (hd == 64)
    return launch_prefill_hd<64>(qkv, ldq, pos, m, cs, sn, kc, vc, out, ldo, nh, nkv,
                                 (int)max_seq, s);
  if (hd == 128)
    return launch_prefill_hd<128>(qkv, ldq, pos, m, cs, sn, kc, vc, out, ldo, nh, nkv,
                                  (int)max_seq, s);
  return launch_prefill_hd<256>(qkv, ldq, pos, m, cs, sn, kc, vc, out, ldo, nh, nkv,
                                (int)max_seq, s);
}

// ---------------------------------------------------------------------------
// Attention without a caller workspace (gguf_hip_attention_decode_noalloc).
// The records and counters live in `scratch`, a file-scope device array that
// every GPU the library runs on holds until the process ends.  Its address is
// taken once per device with hipGetSymbolAddress (the host-side name is only
// a stand-in, not a device address) and passed to the kernels.  Calls that
// overlap on one GPU race on it; each call clears the counters it uses with a
// fill kernel first (no memset, so the call can be captured in a graph).
// ---------------------------------------------------------------------------
namespace {

__device__ __align__(256) unsigned char scratch[kNoAllocAttentionBytes];

std::mutex g_scratch_mu;
constexpr int kMaxDevices = 64;
void *g_scratch[kMaxDevices];  // per device: the device address of `scratch`

__global__ __launch_bounds__(kGlueThreads) void clear_u32_kernel(unsigned *__restrict__ p, int n) {
  for (int i = threadIdx.x; i < n; i += kGlueThreads) p[i] = 0u;
}

hipError_t scratch_ptr(void **out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratch[dev] = p;
  }
  *out = g_scratch[dev];
  return hipSuccess;
}

}  // namespace

hipError_t launch_attention_decode_noalloc(const float *qkv, const int64_t *pos, const float *cs,
                                           const float *sn, float *kc, float *vc, float *out,
                                           int nh, int nkv, int hd, int64_t max_seq,
                                           hipStream_t s) {
  void *ws = nullptr;
  hipError_t e = scratch_ptr(&ws);
  if (e != hipSuccess) return e;
  unsigned *counters = (unsigned *)((char *)ws + attention_record_bytes(nh, nkv, hd, max_seq));
  hipLaunchKernelGGL(clear_u32_kernel, dim3(1), dim3(kGlueThreads), 0, s, counters, nkv);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_attention(qkv, pos, cs, sn, kc, vc, out, (float *)ws, counters, nh, nkv, hd,
                          max_seq, s);
}

int64_t argmax_work_bytes() { return (int64_t)kArgBlocks * (sizeof(float) + sizeof(int64_t)); }

hipError_t launch_argmax(const float *x, int64_t n, int64_t *out, void *work, hipStream_t s) {
  int64_t *pi = (int64_t *)work;
  float *pv = (float *)(pi + kArgBlocks);
  hipLaunchKernelGGL(argmax_partial_kernel, dim3(kArgBlocks), dim3(kGlueThreads), 0, s, x, n, pv,
                     pi);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(argmax_merge_kernel, dim3(1), dim3(kGlueThreads), 0, s, pv, pi, out);
  return hipGetLastError();
}

}  // namespace gguf
