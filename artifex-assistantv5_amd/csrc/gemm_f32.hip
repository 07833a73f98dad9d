// f32-grade GEMM for batches past the 32 rows of the batched decode (33 .. 511
// f32 activation rows of Q4_K, Q5_K and Q6_K weights):
//   y[m, n] = sum_k x[m, k] W[n, k]
// with the arithmetic of the batched decode (decode_mk.hpp).  Each 256-element
// unit of an activation row is scaled by its own power of two and split into f16
// hi + lo parts (22 significant bits); the weight operand is the exact integer
// sc q of a code and its sub-block scale; a unit's products chain in one f32
// accumulator D per output and
//     acc[m, n] += 2^-e[m] (d D - 32 dmin (mins . group sums))
// in f32.  The reference runs its GEMV once per row here
// (webgpu/src/engine/forward-pass.ts:1536-1539).
//
// Run through the batched decode 32 rows at a time, these batches read and
// dequantize the weights in every wave once per 32 rows, for about 8 MFMAs per
// operand.  Here a wave owns 64 rows by 16 NT columns (NT = 4, Q5_K 3, Q6_K 2):
// - A workgroup has four column groups of waves times two halves of its K range
//   (waves 0-3 and 4-7, added through LDS at the end), so that each SIMD has two
//   waves without partial sums in memory.  Larger K splits (grid.y, when the grid
//   leaves CUs idle) write partial sums, added in order.
// - gemm_f32_prep_kernel writes the activations once per call as the image of the
//   LDS stages: per 64 rows and half unit (128 elements) padded hi and lo rows, the
//   group sums and the inverse scales.  A stage is copied by LDS-direct loads, two
//   per K half, one barrier per half unit; K half 1 runs half a unit behind.
// - v_mfma_f32_16x16x32_f16: a fragment read from LDS feeds NT tiles, a weight
//   operand 4 row tiles and both parts.  The operand is the exact f16 integer
//   sc (q - Z) (Q6_K: the sum of two); the codes come straight from memory.
// Measured against the 32-row passes, whole call: Q4_K 128 x 28672 x 4096
// 146 -> 77 us, Q6_K 387 x 4096 x 14336 313 -> 187, Q5_K 200 x 14336 x 4096 415 -> 117,
// Q6_K 500 x 14336 x 4096 424 -> 229, Q4_K 40 x 4096 x 4096 26 -> 22; the error against
// float64 fell (Q4_K 3.0e-7 -> 1.9e-7, Q6_K 1.25e-7 -> 1.09e-7).  What bounds it: the
// vector work of the operands (35 of the 78 us of the first, by leaving it out) and
// the MFMAs beside it (28 us at their full rate) hardly overlap on two waves per SIMD.
#include "decode_impl.hpp"
#include "gguf_hip.h"

namespace gguf {

namespace {

typedef __amdgpu_buffer_rsrc_t rsrc_t;

// A stage for RT row tiles of 16: hi rows, then lo rows of 128 elements, each padded
// by 16 bytes (bank spread; with the unit's second half the pads hold the row's 8
// group sums, hi and lo f16 parts), then an inverse scale per row; whole 1 KB
// pieces, as many for each of 4 waves.
constexpr int kPad = 2 * 128, kLdA = kPad + 16;
template <int RT>
struct FStage {
  static constexpr int ROWS = 16 * RT, L = ROWS * kLdA, F = 2 * L;
  static constexpr int BYTES = (F + ROWS * 4 + 4095) / 4096 * 4096;
};
constexpr int kThr = 512;

__device__ __forceinline__ uint4 bl16(rsrc_t rs, int voff, int soff) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(rs, voff, soff, 0);
  return make_uint4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ uint2 bl8(rsrc_t rs, int voff, int soff) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b64(rs, voff, soff, 0);
  return make_uint2(v[0], v[1]);
}
// A wave-uniform resource.  The base and size go through readfirstlane: the
// compiler otherwise holds them in vector registers and wraps each load in a loop
// over the values they might take.
struct Base {
  uint32_t lo, hi;
  int bytes;
  __device__ __forceinline__ rsrc_t rs() const {
    return __builtin_amdgcn_make_buffer_rsrc((void *)(lo | (uint64_t)hi << 32), 0, bytes,
                                             0x00020000);
  }
};
__device__ __forceinline__ Base make_base(const void *p, int bytes) {
  return Base{(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)p),
              (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)((uintptr_t)p >> 32)),
              __builtin_amdgcn_readfirstlane(bytes)};
}
__device__ __forceinline__ uint32_t pk_fma(half2_t a, half2_t b, half2_t c) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(a, b, c));
}
__device__ __forceinline__ half2_t dup(half_t v) { return half2_t{v, v}; }

// A wave's weights: NT row tiles of 16 weight rows (output columns).  PARTS = 1:
// one exact f16 integer; 2: the sum of two (Q6_K).
// ORDER: the k order of the activations (decode_mk.hpp).
//   load<HF>(u)   request half HF's codes of unit u; header(u) its header
//   begin(act)    the header as the operands use it; the unit adds zero unless act
//   operand(...)  of step n (32 elements) of half HF
template <int TYPE>
struct FW;

// Q4_K / Q5_K.  Step n of a half: chunk n / 2, nibble n & 1.  The operand is
// sc (q - Z), Z the middle of the codes: the products' running sum, and so its f32
// rounding, is half of sc q's; the offset Z d sum(sc S) comes back with the mins.
template <int TYPE>
struct FWK {
  static constexpr int PARTS = 1, ORDER = 1, TU = Fmt<TYPE>::TU, RT = 4, NT = TYPE == 12 ? 4 : 3;
  static constexpr bool MINS = true;
  static constexpr int Z = TYPE == 12 ? 8 : 16, HDR = 1024;
  Base base;
  int ts, vh, vq, vx;   // header, piece and (Q5_K) fifth bits of the lane's row
  uint4 q[2][NT];           // [half][tile]
  unsigned char *hl;        // the wave's 1 KB of LDS: the headers, requested ahead
  uint2 xn[NT], x[NT];      // Q5_K fifth bits, ahead and current
  uint32_t scl[NT], sch[NT], ml[NT], mh[NT], dd[NT];

  __device__ __forceinline__ void init(Base b, int tile_bytes, int lane, unsigned char *headers) {
    base = b;
    hl = headers;
    ts = tile_bytes;
    vh = (lane >> 4) * tile_bytes + 16 * (lane & 15);  // lane l: tile l / 16 (zeros past NT)
    vq = 256 + 16 * lane;
    vx = 2304 + 8 * lane;
  }
  template <int HF>
  __device__ __forceinline__ void load(int u) {
    const rsrc_t rs = base.rs();
#pragma unroll
    for (int j = 0; j < NT; ++j) q[HF][j] = bl16(rs, vq, j * ts + u * TU + 1024 * HF);
  }
  __device__ __forceinline__ void header(int u) {
    const rsrc_t rs = base.rs();
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void *)hl, 16,
                                             vh, u * TU, 0, 0);
    if (TYPE == 13)
#pragma unroll
      for (int j = 0; j < NT; ++j) xn[j] = bl8(rs, vx, j * ts + u * TU);
  }
  __device__ __forceinline__ void begin(bool act) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const uint4 h = *(const uint4 *)(hl + 256 * j + 16 * (threadIdx.x & 15));
      q4k_scales_packed(h.y, h.z, h.w, scl[j], sch[j], ml[j], mh[j]);
      dd[j] = act ? h.x : 0u;
      if (TYPE == 13) x[j] = xn[j];
    }
  }
  template <int HF>
  __device__ __forceinline__ void operand(int n, int j, uint32_t one, half8_t (&b)[PARTS]) const {
    const int c = 2 * HF + (n >> 1), hb = n & 1;
    // (sc of the low nibbles, sc / 16 of the high ones) of chunk c
    const uint32_t two = __builtin_amdgcn_perm(
        0x64646464u, (HF ? sch[j] : scl[j]) >> (16 * (c & 1)), 0x04010400u);
    const half2_t sc =
        (__builtin_bit_cast(half2_t, two) + half2_t{(half_t)-1024.f, (half_t)-1024.f}) *
        half2_t{(half_t)1.f, (half_t)0.0625f};
    const half2_t sp = dup(sc[hb]), off = dup((half_t)(hb ? -1024.f - 16 * Z : -1024.f - Z));
    const uint4 p = q[HF][j];
    const uint32_t w[2] = {n >> 1 ? p.z : p.x, n >> 1 ? p.w : p.y};
    const uint32_t m = hb ? 0x00F000F0u : 0x000F000Fu;
    uint32_t v[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      uint32_t e = and_or(w[i], m, one), o = and_or(w[i] >> 8, m, one);
      if (TYPE == 13) {
        const uint32_t f = i ? x[j].y : x[j].x;
        e |= hb ? q5k_hi_even(f, c) : q5k_lo_even(f, c);
        o |= hb ? q5k_hi_odd(f, c) : q5k_lo_odd(f, c);
      }
      v[2 * i] = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(half2_t, e) + off) * sp);
      v[2 * i + 1] = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(half2_t, o) + off) * sp);
    }
    b[0] = as_h8(v[0], v[1], v[2], v[3]);
  }
  // the mins' and the scales' operands of lane group g: of sub-blocks 4 (g & 1) + (0, 2, 1, 3)
  __device__ __forceinline__ half4_t mins(int j, int g) const {
    constexpr uint32_t nb = neg_base(0);
    const uint32_t w = (g & 1) ? mh[j] : ml[j];
    return as_h4(f16_codes(w, 0x00FF00FFu, nb), f16_codes(w >> 8, 0x00FF00FFu, nb));
  }
  __device__ __forceinline__ half4_t offs(int j, int g) const {
    constexpr uint32_t nb = neg_base(0);
    const uint32_t w = (g & 1) ? sch[j] : scl[j];
    return as_h4(f16_codes(w, 0x00FF00FFu, nb), f16_codes(w >> 8, 0x00FF00FFu, nb));
  }
  __device__ __forceinline__ float d(int j) const { return h2f(dd[j]); }
  __device__ __forceinline__ float dmin(int j) const { return -32.f * h2f(dd[j] >> 16); }
};
template <>
struct FW<12> : FWK<12> {};
template <>
struct FW<13> : FWK<13> {};

// Q6_K: W = sc (q - 32), |W| <= 4096, has up to 13 bits and enters as Wc, W rounded to a
// multiple of 16 (8 bits: with x_hi's 11 the sums hardly round), and W - Wc, both exact:
// four products with the parts of x.  Step n of a half is a window of 32 elements, the
// lane's 8 a quad of each of its two scale groups.
template <>
struct FW<14> {
  static constexpr int PARTS = 2, ORDER = 2, TU = Fmt<14>::TU, RT = 4, NT = 2;
  static constexpr bool MINS = false;
  Base base;
  int ts, vq, vs, vd;
  uint4 q0[NT], q1[NT], q1n[NT], q2[NT];  // the lane's 12 dwords (1n: ahead)
  uint4 sn[NT], sc[NT];
  uint32_t dn[NT], dd[NT];

  __device__ __forceinline__ void init(Base b, int tile_bytes, int lane, unsigned char *) {
    base = b;
    ts = tile_bytes;
    vq = 16 * lane;
    vs = 3072 + 16 * (lane & 15);
    vd = 3328 + 2 * (lane & 15);
  }
  template <int HF>
  __device__ __forceinline__ void load(int u) {
    const rsrc_t rs = base.rs();
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      if (HF == 0) {
        q0[j] = bl16(rs, vq, j * ts + u * TU);
        q1n[j] = bl16(rs, vq, j * ts + u * TU + 1024);
      } else {
        q2[j] = bl16(rs, vq, j * ts + u * TU + 2048);
      }
    }
  }
  __device__ __forceinline__ void header(int u) {
    const rsrc_t rs = base.rs();
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      sn[j] = bl16(rs, vs, j * ts + u * TU);
      dn[j] = __builtin_amdgcn_raw_buffer_load_b16(rs, vd, j * ts + u * TU, 0);
    }
  }
  __device__ __forceinline__ void begin(bool act) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      sc[j] = sn[j];
      q1[j] = q1n[j];
      dd[j] = act ? dn[j] : 0u;
    }
  }
  template <int HF>
  __device__ __forceinline__ void operand(int t, int j, uint32_t one, half8_t (&b)[PARTS]) const {
    const int win = 4 * HF + t;
    const uint4 p = HF ? q2[j] : q0[j], e = q1[j];
    const uint32_t dq[6] = {HF ? e.z : p.x, HF ? e.w : p.y, HF ? p.x : p.z,
                            HF ? p.y : p.w, HF ? p.z : e.x, HF ? p.w : e.y};
    // the window's scales, bytes 2 win, 2 win + 1, as signed f16 integers
    const uint32_t sw = win >> 1 == 0 ? sc[j].x : win >> 1 == 1 ? sc[j].y : win >> 1 == 2 ? sc[j].z : sc[j].w;
    const uint32_t two =
        __builtin_amdgcn_perm(0x64646464u, (sw ^ 0x80808080u) >> (16 * (win & 1)), 0x04010400u);
    const half2_t sv = __builtin_bit_cast(half2_t, two) + half2_t{(half_t)-1152.f, (half_t)-1152.f};
    const half2_t n1056 = {(half_t)-1056.f, (half_t)-1056.f};
    const half2_t magic = {(half_t)24576.f, (half_t)24576.f};  // its ulp is 16
    uint32_t wc[4], wl[4];
#pragma unroll
    for (int lh = 0; lh < 2; ++lh) {
      const uint32_t ql = dq[3 * lh + (t & 1)], qh = dq[3 * lh + 2];
      const uint32_t hi = t == 0 ? (qh << 4) : t == 1 ? (qh << 2) : t == 2 ? qh : (qh >> 2);
      const uint32_t v = ((t >> 1 ? ql >> 4 : ql) & 0x0F0F0F0Fu) | (hi & 0x30303030u);
      const half2_t sp = dup(sv[lh]);
#pragma unroll
      for (int o = 0; o < 2; ++o) {
        const half2_t c = __builtin_bit_cast(half2_t, and_or(o ? v >> 8 : v, 0x00FF00FFu, one)) + n1056;
        const half2_t w = __builtin_elementwise_fma(c, sp, magic) - magic;
        wc[2 * lh + o] = __builtin_bit_cast(uint32_t, w);
        wl[2 * lh + o] = pk_fma(c, sp, -w);
      }
    }
    b[0] = as_h8(wc[0], wc[1], wc[2], wc[3]);
    b[1] = as_h8(wl[0], wl[1], wl[2], wl[3]);
  }
  static constexpr int Z = 0, HDR = 0;
  __device__ __forceinline__ half4_t mins(int, int) const { return half4_t{}; }
  __device__ __forceinline__ half4_t offs(int, int) const { return half4_t{}; }
  __device__ __forceinline__ float d(int j) const { return h2f(dd[j]); }
  __device__ __forceinline__ float dmin(int) const { return 0.f; }
};

// The stages' image, one wave per (unit, activation row), four per workgroup; the
// arithmetic of mk_stage.  Rows past M are not written: their outputs are not stored.
template <int ORDER, bool MINS, int RT>
__global__ __launch_bounds__(256) void gemm_f32_prep_kernel(const float *__restrict__ x,
                                                            int64_t ldx, int M, int nu,
                                                            unsigned char *__restrict__ img) {
  const int u = blockIdx.x, m = 4 * blockIdx.y + (threadIdx.x >> 6), l = threadIdx.x & 63;
  if (m >= M) return;
  const float4 t = *(const float4 *)(x + (int64_t)m * ldx + 256 * u + 4 * l);
  const float v[4] = {t.x, t.y, t.z, t.w};
  const float mx = max_xor32(
      max_xor16(max_lanes16(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))))));
  const int ex = stage_exp(mx);
  const float sc = pow2f(ex);
  half4_t h, lo;
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int pos = (i & 1) << 1 | (i >> 1);  // quad order (0, 2, 1, 3)
    float vi = v[i];
    asm volatile("" : "+v"(vi));  // keep the product out of the f16 conversions (no v_fma_mix)
    const float p = vi * sc;      // exact: a power of two
    const half_t hh = (half_t)p;
    const half_t ll = (half_t)(p - (float)hh);
    h[pos] = hh;
    lo[pos] = ll;
    s += (float)hh + (float)ll;
  }
  // ORDER 2: quad l = 8 w + 4 lh + g of window w goes to quad 8 w + 2 g + lh
  const int dq = ORDER == 2 ? (l & ~7) | ((l & 3) << 1) | ((l >> 2) & 1) : l;
  using St = FStage<RT>;
  const int row = m % St::ROWS;
  unsigned char *blk = img + ((int64_t)(m / St::ROWS) * nu + u) * 2 * St::BYTES;
  unsigned char *a = blk + (dq >> 5) * St::BYTES + row * kLdA + 8 * (dq & 31);
  *(half4_t *)a = h;
  *(half4_t *)(a + St::L) = lo;
  if (MINS) {
    s += dpp<kDppXor1>(s);  // the 8 lanes of a 32-element group
    s += dpp<kDppXor2>(s);
    s += dpp<kDppHalfMirror>(s);
    if ((l & 7) == 0) {
      const int j = l >> 3, k = (j & 4) | ((j & 1) << 1) | ((j >> 1) & 1);  // as the mins
      const float xs = s * 0.03125f;
      const half_t xh = (half_t)xs;
      unsigned char *S = blk + St::BYTES + row * kLdA + kPad + 2 * k;
      *(half_t *)S = xh;
      *(half_t *)(S + St::L) = (half_t)(xs - (float)xh);
    }
  }
  if ((l & 31) == 0) ((float *)(blk + (l >> 5) * St::BYTES + St::F))[row] = pow2f(-ex);
}

// One half unit: 4 steps of 32 elements.  D chains the products of a unit; with
// PARTS = 2 those of the lo parts and residuals chain in E, and the coarse ones by
// halves of a unit (a long f32 chain at the sum's full size is what rounds most).
template <int TYPE>
struct Acc {
  static constexpr int RT = FW<TYPE>::RT, NT = FW<TYPE>::NT, P = FW<TYPE>::PARTS;
  float4_t acc[RT][NT], D[RT][NT], E[P == 2 ? RT : 1][P == 2 ? NT : 1];
  float4_t tot[P == 2 ? RT : 1][P == 2 ? NT : 1];  // the sums of each 4 units, added
};

template <int TYPE, int HF>
__device__ __forceinline__ void half_unit(const FW<TYPE> &w, const unsigned char *stage, int lane,
                                          Acc<TYPE> &a) {
  constexpr int P = FW<TYPE>::PARTS, RT = FW<TYPE>::RT, NT = FW<TYPE>::NT;
  constexpr int NP = 2 * P;  // products
  using St = FStage<RT>;
  const float4_t zero = {0.f, 0.f, 0.f, 0.f};
  uint32_t one = kF16Base;  // 1024.0 x 2 in a register: one v_and_or_b32 per masked pair
  asm volatile("" : "+v"(one));
  const int r = lane & 15, g = lane >> 4;
  const unsigned char *st = stage + r * kLdA + 16 * g;
  half8_t ah[RT], al[RT], b[P], bn[P];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    ah[i] = *(const half8_t *)(st + 16 * i * kLdA);
    al[i] = *(const half8_t *)(st + St::L + 16 * i * kLdA);
  }
  w.template operand<HF>(0, 0, one, b);
#pragma unroll
  for (int n = 0; n < 4; ++n)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const bool last = n == 3 && j == NT - 1, first = HF == 0 && n == 0;
      if (!last) w.template operand<HF>(j + 1 < NT ? n : n + 1, j + 1 < NT ? j + 1 : 0, one, bn);
      // the products of one output tile are RT MFMAs apart
#pragma unroll
      for (int p = P - 1; p >= 0; --p)
#pragma unroll
        for (int i = 0; i < RT; ++i) {
          float4_t &s = P == 2 ? a.E[i % (P == 2 ? RT : 1)][j % (P == 2 ? NT : 1)] : a.D[i][j];
          s = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[i], b[p], first && p == P - 1 ? zero : s, 0,
                                                     0, 0);
        }
      if (j == NT - 1 && n < 3)  // the fragments' last use: the next step's
#pragma unroll
        for (int i = 0; i < RT; ++i)
          al[i] = *(const half8_t *)(st + 64 * (n + 1) + St::L + 16 * i * kLdA);
#pragma unroll
      for (int i = 0; i < RT; ++i)
        a.D[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
            ah[i], b[0], n == 0 && P == 2 ? zero : a.D[i][j], 0, 0, 0);
      if constexpr (P == 2)
#pragma unroll
        for (int i = 0; i < RT; ++i)
          a.E[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[i], b[1], a.E[i][j], 0, 0, 0);
      if (j == NT - 1 && n < 3)
#pragma unroll
        for (int i = 0; i < RT; ++i) ah[i] = *(const half8_t *)(st + 64 * (n + 1) + 16 * i * kLdA);
#pragma unroll
      for (int p = 0; p < P; ++p) b[p] = bn[p];
#pragma unroll
      for (int i = 0; i < RT * NP; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // an MFMA
        if (j == NT - 1 && n < 3 && (i >= RT * (NP - 1) || i < RT))
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // two VALU
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  if constexpr (HF == 0 && P != 2) return;
  // acc += 2^-e (d D + (Z 32 d) scales . sums - (32 dmin) mins . sums)
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const float4 F = *(const float4 *)(stage + St::F + 4 * (16 * i + 4 * g));
    const float f[4] = {F.x, F.y, F.z, F.w};
    half4_t sums = {};
    if (FW<TYPE>::MINS)  // K = 16: the hi, then the lo parts of the 8 sums
      sums = *(const half4_t *)(stage + (16 * i + r) * kLdA + kPad + (g >> 1) * St::L + 8 * (g & 1));
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      float4_t ms = zero, ss = zero;
      if (FW<TYPE>::MINS) {
        ms = __builtin_amdgcn_mfma_f32_16x16x16f16(sums, w.mins(j, g), zero, 0, 0, 0);
        ss = __builtin_amdgcn_mfma_f32_16x16x16f16(sums, w.offs(j, g), zero, 0, 0, 0);
      }
      const float d = w.d(j), dm = w.dmin(j), dz = 32.f * FW<TYPE>::Z * d;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (FW<TYPE>::MINS)
          a.acc[i][j][e] = fmaf(f[e], fmaf(d, a.D[i][j][e], fmaf(dz, ss[e], dm * ms[e])),
                                a.acc[i][j][e]);
        else {  // f d is exact: f is a power of two
          const float E = HF ? a.E[i % (P == 2 ? RT : 1)][j % (P == 2 ? NT : 1)][e] : 0.f;
          a.acc[i][j][e] = fmaf(f[e] * d, HF ? a.D[i][j][e] + E : a.D[i][j][e], a.acc[i][j][e]);
        }
      }
    }
  }
}

template <int TYPE>
__global__ __launch_bounds__(kThr) void gemm_f32_kernel(const unsigned char *__restrict__ img,
                                                        const uint8_t *__restrict__ W, int M, int N,
                                                        int nu, int kunits, int rb,
                                                        float *__restrict__ y, int64_t ldy) {
  constexpr int RT = FW<TYPE>::RT, NT = FW<TYPE>::NT, SB = FStage<RT>::BYTES;
  __shared__ __align__(16) unsigned char lds[4 * SB + 8 * FW<TYPE>::HDR];
  static_assert(4 * SB >= 4 * 64 * 4 * RT * NT * 4, "the K halves' sums are added through it");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kg = __builtin_amdgcn_readfirstlane(wave >> 2);
  const int cw = __builtin_amdgcn_readfirstlane(wave & 3);
  // tiles XCD by XCD (workgroup b runs on XCD b % 8), row blocks fastest: the
  // blocks that share a weight tile share an L2
  const int T = gridDim.x, b = blockIdx.x, xcd = b & 7, rem = T & 7;
  const int t = xcd * (T >> 3) + min(xcd, rem) + (b >> 3);
  const int rblk = t % rb, tile0 = __builtin_amdgcn_readfirstlane((t / rb * 4 + cw) * NT);
  const int ua = blockIdx.y * kunits, un = min(nu - ua, kunits), h0 = (un + 1) >> 1;
  const int u0 = ua + (kg ? h0 : 0), cnt = kg ? un - h0 : h0;  // this K half's units

  // one resource over the wave's row tiles, as far as the weight has them
  const int ts = nu * FW<TYPE>::TU, nt = (N + 15) / 16 - tile0;
  FW<TYPE> w;
  w.init(make_base(W + (int64_t)tile0 * ts, max(0, min(nt, NT)) * ts), ts, lane,
         lds + 4 * SB + __builtin_amdgcn_readfirstlane(wave) * FW<TYPE>::HDR);
  const unsigned char *src = img + (int64_t)rblk * nu * 2 * SB;
  unsigned char *const s0 = lds + kg * 2 * SB, *const s1 = s0 + SB;
  auto stage = [&](int u, int hf, unsigned char *dst) {
    const rsrc_t rs = make_base(src + ((int64_t)u * 2 + hf) * SB, SB).rs();
#pragma unroll
    for (int i = 0; i < SB / 4096; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rs, (__attribute__((address_space(3))) void *)(dst + 1024 * (4 * i + cw)), 16, 16 * lane,
          1024 * (4 * i + cw), 0, 0);
  };

  Acc<TYPE> a;
  constexpr int TR = FW<TYPE>::PARTS == 2 ? RT : 1, TN = FW<TYPE>::PARTS == 2 ? NT : 1;
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      a.acc[i][j] = (float4_t){0.f, 0.f, 0.f, 0.f};
      if (FW<TYPE>::PARTS == 2) a.tot[i % TR][j % TN] = a.acc[i][j];
    }
  // The loop body is straight-line: a K half shorter than the other re-reads its last
  // unit and adds zero, and the loads past the last unit re-read it.  With them under
  // a condition the memory counter's waits assume that they were not issued, and each
  // half unit would wait for its own prefetch.
  // The unit's headers are read before its second half's stage is requested: after that
  // the compiler cannot tell them from the stage and waits for it.  (At a unit's end, where
  // the next stage has been in flight for half a unit, the sums' reads wait for it in Q4_K
  // and Q5_K; Q4_K reloads three of five spilled registers there.)  14336 x 4096, Q5_K, 128
  // rows 64.9 -> 62.0 us, 28672 x 4096, Q4_K, 128 rows 78.8 -> 76.8.
  const int ul = min(ua + un, u0 + max(cnt, 1)) - 1;
  stage(min(u0, ul), 0, s0);
  w.template load<0>(min(u0, ul));
  w.header(min(u0, ul));
  // K half 1 runs half a unit behind K half 0, so that the waves of a SIMD are not at
  // the start or at the sums of a unit together
  if (kg == 1) __syncthreads();
  for (int i = 0; i < h0; ++i) {
    const int u = min(u0 + i, ul), v = min(u0 + i + 1, ul);
    const bool act = i < cnt;
    __syncthreads();  // the first half's stage has arrived, the second's is free
    w.begin(act);
    stage(u, 1, s1);
    w.template load<1>(u);
    half_unit<TYPE, 0>(w, s0, lane, a);
    __syncthreads();
    stage(v, 0, s0);
    w.template load<0>(v);
    w.header(v);
    half_unit<TYPE, 1>(w, s1, lane, a);
    if (FW<TYPE>::PARTS == 2 && ((i & 3) == 3 || i == h0 - 1)) {
#pragma unroll
      for (int p = 0; p < RT; ++p)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          a.tot[p % TR][j % TN] += a.acc[p][j];
          a.acc[p][j] = i == h0 - 1 ? a.tot[p % TR][j % TN] : (float4_t){0.f, 0.f, 0.f, 0.f};
        }
    }
  }

  if (kg == 0) __syncthreads();
  // the second K half's sums, through LDS
  __syncthreads();
  float *x = (float *)lds + cw * 256 * RT * NT + 4 * lane;
  if (kg == 1) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        *(float4 *)(x + 256 * (NT * i + j)) =
            make_float4(a.acc[i][j][0], a.acc[i][j][1], a.acc[i][j][2], a.acc[i][j][3]);
  }
  __syncthreads();
  if (kg == 1) return;
  float *yb = y + (gridDim.y > 1 ? (int64_t)blockIdx.y * M * ldy : 0);
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int n = 16 * (tile0 + j) + (lane & 15);
      const float4 p = *(const float4 *)(x + 256 * (NT * i + j));
      const float pv[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = rblk * 16 * RT + 16 * i + 4 * (lane >> 4) + e;
        if (m < M && n < N) yb[(int64_t)m * ldy + n] = a.acc[i][j][e] + pv[e];
      }
    }
}

struct F32Plan {
  int rb, cb, nu, sp, kunits;
  int64_t img, part;  // floats
};
// K splits by estimated time: rounds of 256 workgroups (one per CU, MI355X), each the
// type's microseconds a unit and K half, 15% more with every CU at work; splitting costs a
// second launch and the partial sums' write and read.  Fitted to 1, 2, 3, 4, 6, 8, 12 and 16
// splits of 11 weights (1024 x 512 to 32000 x 2048 and 4096 x 14336) at 33 to 511 rows, 5 to
// 7% rms; the split chosen is within 0.3% of the best on average and 5% at worst.  In us,
// 1 split / the one chosen: Q4_K 14336 x 4096, 128 rows 68.5 / 48.5 (2); 4096^2, 387 rows
// 70.5 / 50.0 (2); 1024^2, 33 rows 22.6 / 17.7 (2); Q6_K 4096 x 14336, 387 rows 195 (1; 2: 200).
template <int TYPE>
F32Plan plan(int64_t n, int64_t k, int64_t m) {
  F32Plan p;
  p.rb = (int)((m + 16 * FW<TYPE>::RT - 1) / (16 * FW<TYPE>::RT));
  p.cb = (int)((n + 64 * FW<TYPE>::NT - 1) / (64 * FW<TYPE>::NT));
  p.nu = (int)(k / 256);
  p.sp = 1;
  p.kunits = p.nu;
  double best = 0;
  for (int s = 1; s <= 16 && s <= p.nu; ++s) {
    const int ku = (p.nu + s - 1) / s;
    if ((p.nu + ku - 1) / ku != s) continue;  // an empty last split
    const int64_t wgs = (int64_t)p.rb * p.cb * s, rounds = (wgs + 255) / 256;
    const double unit = TYPE == 12 ? 7.0 : TYPE == 13 ? 6.3 : 5.8;
    const double us = rounds * ((ku + 1) / 2) * unit * (1 + 0.15 * (wgs < 256 ? wgs / 256.0 : 1)) +
                      (s > 1 ? 1.8 + s * m * n * 8 / 3.9e6 : 0);
    if (s == 1 || us < best) {
      best = us;
      p.sp = s;
      p.kunits = ku;
    }
  }
  p.img = (int64_t)p.rb * p.nu * 2 * FStage<FW<TYPE>::RT>::BYTES / 4;
  p.part = p.sp > 1 ? p.sp * m * n : 0;
  return p;
}
F32Plan f32_plan(int type, int64_t n, int64_t k, int64_t m) {
  return type == 12 ? plan<12>(n, k, m) : type == 13 ? plan<13>(n, k, m) : plan<14>(n, k, m);
}

template <int TYPE>
hipError_t launch(const float *x, int64_t ldx, const uint8_t *W, int64_t n, int64_t m,
                  const F32Plan &p, float *y, int64_t ldy, float *work, hipStream_t s) {
  unsigned char *img = (unsigned char *)work;
  float *part = work + p.img;
  hipLaunchKernelGGL((gemm_f32_prep_kernel<FW<TYPE>::ORDER, FW<TYPE>::MINS, FW<TYPE>::RT>),
                     dim3((unsigned)p.nu, (unsigned)((m + 3) / 4)), dim3(256), 0, s, x, ldx, (int)m,
                     p.nu, img);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(gemm_f32_kernel<TYPE>, dim3((unsigned)(p.rb * p.cb), (unsigned)p.sp),
                     dim3(kThr), 0, s, img, W, (int)m, (int)n, p.nu, p.kunits, p.rb,
                     p.sp > 1 ? part : y, p.sp > 1 ? n : ldy);
  e = hipGetLastError();
  if (e != hipSuccess || p.sp == 1) return e;
  return launch_gemm_reduce(part, p.sp, (int)m, (int)n, y, ldy, s);
}

}  // namespace

// From 33 rows to the row count from which f32 batches take the fp16 GEMM, at any size; a
// weight's row tile keeps 32-bit byte offsets.  Graph replays in us, 32-row passes / here:
//   rows               33           64           128          511
//   Q4_K 256 x 512     20.9 / 15.4  29.0 / 16.2  57.4 / 16.6  228 / 16.9
//        1024^2        18.9 / 17.6  29.4 / 18.6  58.2 / 19.1  232 / 22.4
//        14336 x 4096  30.4 / 30.5  43.5 / 33.3  86.3 / 48.5  337 / 142
//   Q5_K 1024^2        15.7 / 15.6  22.0 / 16.6  43.7 / 17.0  173 / 20.9
//   Q6_K 256 x 512     21.5 / 12.3  34.3 / 12.9  68.4 / 13.2  272 / 13.8
//        14336 x 4096  37.4 / 39.1  55.4 / 41.0  109 / 64     433 / 236
// 33 rows are one 32-row pass and the one-row kernel there, and the only count where the
// passes are level, by up to 4%, at 58 million weights (256 x 14336 also, 26.0 / 26.4).
bool gemm_f32_serves(int type, int x_type, int64_t n, int64_t k, int64_t m) {
  return x_type == 0 && m > 32 && m < GGUF_HIP_F32_GEMM_MIN_M && (type == 12 || type == 13 || type == 14) && k % 256 == 0 &&
         k <= ((int64_t)1 << 24);
}

int64_t gemm_f32_work(int type, int64_t n, int64_t k, int64_t m) {
  const F32Plan p = f32_plan(type, n, k, m);
  return p.img + p.part;
}

hipError_t launch_gemm_f32(const float *x, int64_t ldx, const uint8_t *tiles, int type, int64_t n,
                           int64_t k, float *y, int64_t ldy, int64_t m, float *work,
                           hipStream_t s) {
  const F32Plan p = f32_plan(type, n, k, m);
  switch (type) {
    case 12: return launch<12>(x, ldx, tiles, n, m, p, y, ldy, work, s);
    case 13: return launch<13>(x, ldx, tiles, n, m, p, y, ldy, work, s);
    default: return launch<14>(x, ldx, tiles, n, m, p, y, ldy, work, s);
  }
}

}  // namespace gguf
