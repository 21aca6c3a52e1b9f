// kv_rotate.h -- element codecs and the re-rotation kernels (flat, pair-task and
// element-wise LDS).
// Part of libdaser_kv: included by kv_move.hip, one translation unit.

#pragma once

#include "kv_flat.h"

namespace {

// ---------------------------------------------------------------------------
// Element codecs for the rotation. Each 16-byte vector holds VE elements.

__device__ __forceinline__ float bf16_to_f32(uint32_t h) {
  return __uint_as_float(h << 16);
}
// Round-to-nearest-even fp32 -> bf16; NaN -> 0x7FC0 with its sign dropped.
__device__ __forceinline__ uint32_t f32_to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0u;
  u += 0x7fffu + ((u >> 16) & 1u);
  return u >> 16;
}

__device__ __forceinline__ float fp16_to_f32(uint32_t h) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}
// fp32 -> fp16 by the hardware conversion (round-to-nearest-even) of the fp32
// value itself; NaN -> 0x7E00.
__device__ __forceinline__ uint32_t f32_to_fp16(float f) {
  if (__builtin_isnan(f)) return 0x7e00u;
  asm("" : "+v"(f));
  return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)f);
}
// a * b + t rounded once, to fp16: the vector kernels' fp16 sums. The compiler
// fuses the conversion in some kernels and not in others; by name, every kernel
// rounds alike, and once.
__device__ __forceinline__ uint32_t fma_fp16(float a, float b, float t) {
  _Float16 h;
  asm("v_fma_mixlo_f16 %0, %1, %2, %3" : "=v"(h) : "v"(a), "v"(b), "v"(t));
  return (uint32_t)__builtin_bit_cast(uint16_t, h);
}
// The two halves of w with NaN -> 0x7E00.
__device__ __forceinline__ uint32_t canonical_fp16(uint32_t w) {
  if ((w & 0x7fffu) > 0x7c00u) w = (w & 0xffff0000u) | 0x7e00u;
  if ((w & 0x7fff0000u) > 0x7c000000u) w = (w & 0xffffu) | 0x7e000000u;
  return w;
}

// OCP e4m3fn (bias 7, no infinities, S.1111.111 = NaN) through the gfx950
// conversion instructions, which use the OCP formats: v_cvt_pk_f32_fp8
// decodes two codes, v_cvt_pk_fp8_f32 encodes two floats with
// round-to-nearest-even (both checked exhaustively against the bit-level
// definition on MI355X: all 256 codes, 200k values incl. every midpoint).
// Encoding saturates by clamping to +-448 first (compare-select keeps NaN);
// the instruction turns NaN into 0xFF, which the clamp range never produces,
// so 0xFF bytes are rewritten to the canonical 0x7F.
typedef float f32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float clamp448(float f) {
  f = f > 448.0f ? 448.0f : f;
  return f < -448.0f ? -448.0f : f;
}
// 0x80 in every byte of w that equals 0xFF.
__device__ __forceinline__ uint32_t ff_bytes(uint32_t w) {
  const uint32_t t = ~w;
  return ~(((t & 0x7f7f7f7fu) + 0x7f7f7f7fu) | t) & 0x80808080u;
}
__device__ __forceinline__ void e4m3x4_to_f32(uint32_t w, float* x) {
  const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, false);
  const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, true);
  x[0] = lo.x;
  x[1] = lo.y;
  x[2] = hi.x;
  x[3] = hi.y;
}
__device__ __forceinline__ uint32_t f32x4_to_e4m3(const float* y) {
  int e = __builtin_amdgcn_cvt_pk_fp8_f32(clamp448(y[0]), clamp448(y[1]), 0, false);
  e = __builtin_amdgcn_cvt_pk_fp8_f32(clamp448(y[2]), clamp448(y[3]), e, true);
  const uint32_t w = (uint32_t)e;
  return w ^ ff_bytes(w);
}

// OCP e5m2 (bias 15, infinities, S.11111.{01,10,11} = NaN) through the
// gfx950 bf8 conversions (v_cvt_pk_f32_bf8 / v_cvt_pk_bf8_f32, round to
// nearest even). Encoding saturates as for e4m3: finite values and
// infinities clamp to +-57344 (compare-select keeps NaN), so an encoded byte
// with an all-ones exponent is NaN, rewritten to torch's canonical 0x7F.
__device__ __forceinline__ float clamp57344(float f) {
  f = f > 57344.0f ? 57344.0f : f;
  return f < -57344.0f ? -57344.0f : f;
}
__device__ __forceinline__ void e5m2x4_to_f32(uint32_t w, float* x) {
  const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_bf8((int)w, false);
  const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_bf8((int)w, true);
  x[0] = lo.x;
  x[1] = lo.y;
  x[2] = hi.x;
  x[3] = hi.y;
}
__device__ __forceinline__ uint32_t f32x4_to_e5m2(const float* y) {
  int e = __builtin_amdgcn_cvt_pk_bf8_f32(clamp57344(y[0]), clamp57344(y[1]), 0, false);
  e = __builtin_amdgcn_cvt_pk_bf8_f32(clamp57344(y[2]), clamp57344(y[3]), e, true);
  const uint32_t w = (uint32_t)e;
  // bytes whose exponent bits (0x7C) are all set: 0x80 in each such byte
  const uint32_t x = (w & 0x7c7c7c7cu) ^ 0x7c7c7c7cu;  // zero byte <=> exponent all ones
  const uint32_t nan = ~(((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x | 0x7f7f7f7fu);
  const uint32_t bytes = (nan >> 7) * 0xffu;
  return (w & ~bytes) | (0x7f7f7f7fu & bytes);
}

// The 8-bit formats: one byte per element, K scaled by the layer's k_scale.
template <int DT>
constexpr bool is_fp8() {
  return DT == DSR_DTYPE_FP8_E4M3 || DT == DSR_DTYPE_FP8_E5M2;
}

// The codecs' quick encoders round by the hardware's conversion alone, and say
// whether a result may need more (NaN, or a value outside the format): those
// vectors go through encode. A rotated page holds next to none of them.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

template <int DT>
struct Codec;

template <>
struct Codec<DSR_DTYPE_BF16> {
  static constexpr int VE = 8;
  __device__ static void decode(u32x4 v, float* x) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      x[2 * k] = bf16_to_f32(v[k] & 0xffffu);
      x[2 * k + 1] = bf16_to_f32(v[k] >> 16);
    }
  }
  __device__ static u32x4 encode(const float* y) {
    u32x4 v;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      v[k] = f32_to_bf16(y[2 * k]) | (f32_to_bf16(y[2 * k + 1]) << 16);
    return v;
  }
  static constexpr uint32_t kSigns = 0x80008000u;
  __device__ static bool encode_quick(const float* y, u32x4* v) {
    uint32_t odd = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const f32x2 f = {y[2 * k], y[2 * k + 1]};
      const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
      odd |= (w & 0x7fff7fffu) + 0x007f007fu;  // past infinity: bit 15
      (*v)[k] = w;
    }
    return odd & kSigns;
  }
};

template <>
struct Codec<DSR_DTYPE_FP16> {
  static constexpr int VE = 8;
  __device__ static void decode(u32x4 v, float* x) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      x[2 * k] = fp16_to_f32(v[k] & 0xffffu);
      x[2 * k + 1] = fp16_to_f32(v[k] >> 16);
    }
  }
  __device__ static u32x4 encode(const float* y) {
    u32x4 v;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      v[k] = f32_to_fp16(y[2 * k]) | (f32_to_fp16(y[2 * k + 1]) << 16);
    return v;
  }
  static constexpr uint32_t kSigns = 0x80008000u;
  // the rotated sums x * c + t themselves; c: the cosine of element e is c[e / per].x
  template <int per>
  __device__ static u32x4 encode_sums(const float* x, const float2* c, const float* t) {
    u32x4 v;
    uint32_t odd = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int e = 2 * k;
      v[k] = fma_fp16(x[e], c[e / per].x, t[e]) |
             fma_fp16(x[e + 1], c[(e + 1) / per].x, t[e + 1]) << 16;
      odd |= (v[k] & 0x7fff7fffu) + 0x03ff03ffu;  // past infinity: bit 15
    }
    if (odd & kSigns)
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = canonical_fp16(v[k]);
    return v;
  }
};

template <>
struct Codec<DSR_DTYPE_FP8_E4M3> {
  static constexpr int VE = 16;
  __device__ static void decode(u32x4 v, float* x) {
#pragma unroll
    for (int k = 0; k < 4; ++k) e4m3x4_to_f32(v[k], x + 4 * k);
  }
  __device__ static u32x4 encode(const float* y) {
    u32x4 v;
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = f32x4_to_e4m3(y + 4 * k);
    return v;
  }
  static constexpr uint32_t kSigns = 0x80808080u;
  // without the clamp, values past +-464 encode as NaN too
  __device__ static bool encode_quick(const float* y, u32x4* v) {
    uint32_t odd = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      int e = __builtin_amdgcn_cvt_pk_fp8_f32(y[4 * k], y[4 * k + 1], 0, false);
      e = __builtin_amdgcn_cvt_pk_fp8_f32(y[4 * k + 2], y[4 * k + 3], e, true);
      odd |= ((uint32_t)e & 0x7f7f7f7fu) + 0x01010101u;  // 0x7F: bit 7
      (*v)[k] = (uint32_t)e;
    }
    return odd & kSigns;
  }
};

template <>
struct Codec<DSR_DTYPE_FP8_E5M2> {
  static constexpr int VE = 16;
  __device__ static void decode(u32x4 v, float* x) {
#pragma unroll
    for (int k = 0; k < 4; ++k) e5m2x4_to_f32(v[k], x + 4 * k);
  }
  __device__ static u32x4 encode(const float* y) {
    u32x4 v;
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = f32x4_to_e5m2(y + 4 * k);
    return v;
  }
  static constexpr uint32_t kSigns = 0x80808080u;
  // without the clamp, values past the largest finite one encode as infinity
  __device__ static bool encode_quick(const float* y, u32x4* v) {
    uint32_t odd = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      int e = __builtin_amdgcn_cvt_pk_bf8_f32(y[4 * k], y[4 * k + 1], 0, false);
      e = __builtin_amdgcn_cvt_pk_bf8_f32(y[4 * k + 2], y[4 * k + 3], e, true);
      odd |= ((uint32_t)e & 0x7c7c7c7cu) + 0x04040404u;  // exponent all ones: bit 7
      (*v)[k] = (uint32_t)e;
    }
    return odd & kSigns;
  }
};

struct RotArgs {
  UnitArgs u;
  const float2* cos_sin;
  const int32_t* rope_idx;
  int32_t n_tables;
  const int32_t* layer_group;  // per record layer: table block, -1 = no RoPE (null: all 0)
  int32_t n_groups;
  int32_t row_vecs;    // 16-byte vectors per K row (head_dim * e / 16)
  int32_t rot_half;    // rot_dim / 2 (pairs per row)
  int32_t task_vecs;   // rotation tasks per row
  int32_t tail_vec0;   // first un-rotated vector of a row
  int32_t tasks_per_row;
  int32_t rot_vecs;   // 16-byte vectors of a row inside the rotated region
  int32_t half_vecs;  // neox: vectors from a first-half vector to its partner
  const float* k_scale;
  // Pair-task kernel only: task columns per table column. 1 for token-major
  // K rows; block_size for the split-x K layout, where a row is one head's
  // [head_dim / X][block_size][X] block and vector c holds dims
  // (c / block_size) * X ... + X - 1 of token c % block_size.
  int32_t col_div = 1;
  // Flat and fan-out kernels on split-x K pages: head blocks of
  // 2^kx_row_shift vectors, block_size 2^kx_bs_shift, neox partners
  // kx_dist vectors apart (0 for gptj).
  int32_t kx_row_shift = 0;
  int32_t kx_bs_shift = 0;
  int32_t kx_dist = 0;
};

// Split-x K: the lane-consecutive vector index i of a page -> the vector it
// moves. Inside a head block the rotated region is walked in 64-vector runs
// whose lanes 0-31 take 32 consecutive first-half vectors and lanes 32-63
// their partners kx_dist vectors on, so a neox partner is always lane ^ 32
// and each half-wave still reads 512 contiguous bytes. Tail vectors (and all
// of gptj) keep their index. Needs kx_dist % 32 == 0 and 64 | block vectors.
__device__ __forceinline__ int kx_phys(const RotArgs& ra, int i) {
  const int q = i & ((1 << ra.kx_row_shift) - 1);
  if (q >= 2 * ra.kx_dist) return i;
  const int w = q & 63;
  return i - q + ((q >> 6) << 5) + (w & 31) + (w >= 32 ? ra.kx_dist : 0);
}

// Table column (dims c * VE ...) of physical K vector p: token-major rows
// have row_vecs vectors of consecutive dims; split-x head blocks hold
// block_size vectors per column.
template <bool KX>
__device__ __forceinline__ int k_column(const RotArgs& ra, int p) {
  return KX ? (p & ((1 << ra.kx_row_shift) - 1)) >> ra.kx_bs_shift : p % ra.row_vecs;
}

// Table of unit (page p, layer l): page p's delta table inside layer l's
// group block (cos_sin holds n_groups blocks of n_tables tables), or -1 when
// the page keeps its position or the layer has no RoPE (K copied as is).
__device__ __forceinline__ int rope_table(const RotArgs& ra, int64_t p, int l) {
  const int ti = ra.rope_idx[p];
  if (ti < 0 || ti >= ra.n_tables) return -1;
  if (!ra.layer_group) return ti;
  const int g = ra.layer_group[ra.u.layer0 + l];
  return g < 0 || g >= ra.n_groups ? -1 : g * ra.n_tables + ti;
}

// First table pair of a row's vector column c (neox: both halves of a row use
// the first half's columns).
template <int DT, int STYLE>
__device__ __forceinline__ int table_column(const RotArgs& ra, int c) {
  if (STYLE == DSR_ROPE_NEOX)
    return (c < ra.half_vecs ? c : c - ra.half_vecs) * Codec<DT>::VE;
  return c * (Codec<DT>::VE / 2);
}

// One K vector after rotation: c is its vector column in the row, own its
// bytes, partner (neox) the bytes of the vector half a rotation away, cs the
// pairs of its column. Vectors past the rotated region are returned unchanged.
// kScaled: the values are multiplied by the layer's scale first and by its
// inverse after. The sums are fused by name (the cosine's product exact), so that
// every kernel rounds alike.
template <int DT, int STYLE, bool kScaled>
__device__ __forceinline__ u32x4 rotate_pairs(const RotArgs& ra, u32x4 own, u32x4 partner, int c,
                                              const float2* cs, float scale, float inv_scale) {
  using C = Codec<DT>;
  constexpr int VE = C::VE;
  constexpr int kPer = STYLE == DSR_ROPE_NEOX ? 1 : 2;  // elements per pair
  float x[VE], t[VE];  // t: the sines' products
  C::decode(own, x);
  if (kScaled) {
#pragma unroll
    for (int e = 0; e < VE; ++e) x[e] *= scale;
  }
  if (STYLE == DSR_ROPE_NEOX) {
    // first half: x c - p s; second half: x c + p s. The sign goes into the
    // partner's bits, which is exact.
    const uint32_t flip = c < ra.half_vecs ? C::kSigns : 0u;
    C::decode(partner ^ flip, t);
#pragma unroll
    for (int e = 0; e < VE; ++e) t[e] = (kScaled ? t[e] * scale : t[e]) * cs[e].y;
  } else {
#pragma unroll
    for (int e = 0; e < VE; e += 2) {
      t[e] = -x[e + 1] * cs[e / 2].y;
      t[e + 1] = x[e] * cs[e / 2].y;
    }
  }
  u32x4 v;
  if constexpr (DT == DSR_DTYPE_FP16) {
    v = C::template encode_sums<kPer>(x, cs, t);
  } else {
#pragma unroll
    for (int e = 0; e < VE; ++e) {
      const float y = __builtin_fmaf(x[e], cs[e / kPer].x, t[e]);
      x[e] = kScaled ? y * inv_scale : y;
    }
    if (C::encode_quick(x, &v)) v = C::encode(x);
  }
  return c >= ra.rot_vecs ? own : v;
}

// An 8-bit layer's scale is multiplied in and its inverse out again: two
// roundings of each value that decide a few ties. A power of two rounds nothing, so
// it is left out (1.0, the scale of uncalibrated caches, among them); the range
// keeps every product normal. The multiplications cost a Llama-3-8B e4m3 load
// nothing, 70B and TP8 loads 1%, Gemma-2-9B head-major ones 2%.
__device__ __forceinline__ bool scale_is_exact(float scale) {
  const uint32_t u = __float_as_uint(scale) & 0x7fffffffu;
  return (u & 0x007fffffu) == 0 && u >= 0x2f800000u && u <= 0x4f800000u;  // 2^-32 to 2^32
}
template <int DT, int STYLE>
__device__ __forceinline__ u32x4 rotate_vec(const RotArgs& ra, u32x4 own, u32x4 partner, int c,
                                            const float2* cs, float scale, float inv_scale) {
  if (is_fp8<DT>() && !scale_is_exact(scale))
    return rotate_pairs<DT, STYLE, true>(ra, own, partner, c, cs, scale, inv_scale);
  return rotate_pairs<DT, STYLE, false>(ra, own, partner, c, cs, scale, inv_scale);
}

// K-page rotation in rounds of kRotUnroll tasks per lane. Task t covers row
// t / tasks_per_row, column c = t % tasks_per_row:
//   neox, c < task_vecs: vector c of the rotated first half and its partner
//                        at +rot_half elements;
//   gptj, c < task_vecs: vector c, whose VE/2 adjacent pairs rotate in place;
//   c >= task_vecs:      one un-rotated 16-byte tail vector, copied.
// The table column of task column c is c / col_div (split-x K: the rows,
// columns and half distance are all counted in vectors of the head block).
template <int DT, int STYLE>
struct KRound {
  static constexpr int VE = Codec<DT>::VE;
  u32x4 a[kRotUnroll], b[kRotUnroll];
  int off[kRotUnroll];
  int kind[kRotUnroll];  // 0 = rotate, 1 = copy, -1 = none
  int c_of[kRotUnroll];

  __device__ __forceinline__ void load(const RotArgs& ra, rsrc_t rs, int base, int ntask,
                                       int row_bytes, int half_off) {
#pragma unroll
    for (int k = 0; k < kRotUnroll; ++k) {
      const int t = base + k * kThreads;
      kind[k] = -1;
      off[k] = 0;
      c_of[k] = 0;
      a[k] = u32x4{0u, 0u, 0u, 0u};
      b[k] = a[k];
      if (t < ntask) {
        const int row = t / ra.tasks_per_row;
        const int c = t - row * ra.tasks_per_row;
        c_of[k] = ra.col_div == 1 ? c : c / ra.col_div;
        if (c < ra.task_vecs) {
          kind[k] = 0;
          off[k] = row * row_bytes + (c << 4);
          a[k] = bload(rs, off[k]);
          if (STYLE == DSR_ROPE_NEOX) b[k] = bload(rs, off[k] + half_off);
        } else {
          kind[k] = 1;
          off[k] = row * row_bytes + ((ra.tail_vec0 + c - ra.task_vecs) << 4);
          a[k] = bload(rs, off[k]);
        }
      }
    }
  }

  __device__ __forceinline__ void store(const RotArgs& ra, rsrc_t rd, const float2* tab,
                                        int half_off, float scale, float inv_scale) {
#pragma unroll
    for (int k = 0; k < kRotUnroll; ++k) {
      if (kind[k] == 1) {
        bstore(rd, off[k], a[k]);
      } else if (kind[k] == 0) {
        const int c = c_of[k];
        const float2* cs = tab + table_column<DT, STYLE>(ra, c);
        bstore(rd, off[k], rotate_vec<DT, STYLE>(ra, a[k], b[k], c, cs, scale, inv_scale));
        if (STYLE == DSR_ROPE_NEOX)
          bstore(rd, off[k] + half_off,
                 rotate_vec<DT, STYLE>(ra, b[k], a[k], c + ra.half_vecs, cs, scale, inv_scale));
      }
    }
  }
};

// One page_bytes run copied in rounds of U vectors per lane.
template <int U>
struct VRound {
  u32x4 r[U];
  __device__ __forceinline__ void load(rsrc_t rs, int base, int nvec) {
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const int i = base + k * kThreads;
      r[k] = i < nvec ? bload(rs, i << 4) : u32x4{0u, 0u, 0u, 0u};
    }
  }
  __device__ __forceinline__ void store(rsrc_t rd, int base, int nvec) {
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const int i = base + k * kThreads;
      if (i < nvec) bstore(rd, i << 4, r[k]);
    }
  }
};

// One workgroup per (page, layer) unit in page-list order. V, and K of pages
// without a table (rope_idx < 0), are copied bit-exactly; K of the others is
// re-rotated row by row with the page's (cos, sin) table staged in LDS. The
// first round of V and K loads is issued before the table is fetched and the
// workgroup synchronises, so the table latency overlaps the page reads.
template <int DT, int STYLE>
__global__ __launch_bounds__(kThreads) void kv_scatter_rerotate_kernel(RotArgs ra) {
  __shared__ float2 tab[kMaxRotHalf];
  uint8_t *cache, *rec;
  int l;
  const int64_t u = layer_major_unit(ra.u.n_units, ra.u.n_layers);
  if (u < 0 || !unit_addresses(ra.u, u, &cache, &rec, &l)) return;
  const int64_t p = udiv32(u, ra.u.n_layers);
  const int ti = rope_table(ra, p, l);
  const int64_t pb = ra.u.page_bytes;
  uint8_t* const vrec = rec + pb;
  uint8_t* const vcache = cache + ra.u.kv_stride;
  if (ti < 0) {
    copy_halves<kRotCopyUnroll>(rec, vrec, cache, vcache, pb);
    return;
  }
  const rsrc_t ks = make_rsrc(rec, pb), kd = make_rsrc(cache, pb);
  const rsrc_t vs = make_rsrc(vrec, pb), vd = make_rsrc(vcache, pb);
  const int nvec = (int)(pb >> 4);
  const int row_bytes = ra.row_vecs << 4;
  const int ntask = (int)(pb / row_bytes) * ra.tasks_per_row;
  const int half_off = ra.rot_half * 16 / Codec<DT>::VE * ra.col_div;

  VRound<kScatterUnroll> v;
  KRound<DT, STYLE> k;
  v.load(vs, threadIdx.x, nvec);
  k.load(ra, ks, threadIdx.x, ntask, row_bytes, half_off);

  const float2* src_tab = ra.cos_sin + (int64_t)ti * ra.rot_half;
  for (int j = threadIdx.x; j < ra.rot_half; j += kThreads) tab[j] = src_tab[j];
  float scale = 1.0f, inv_scale = 1.0f;
  if (is_fp8<DT>()) {
    scale = ra.k_scale[ra.u.layer0 + l];
    inv_scale = 1.0f / scale;
  }
  __syncthreads();

  v.store(vd, threadIdx.x, nvec);
  k.store(ra, kd, tab, half_off, scale, inv_scale);
  for (int base = threadIdx.x + kThreads * kScatterUnroll; base < nvec;
       base += kThreads * kScatterUnroll) {
    v.load(vs, base, nvec);
    v.store(vd, base, nvec);
  }
  for (int base = threadIdx.x + kThreads * kRotUnroll; base < ntask;
       base += kThreads * kRotUnroll) {
    k.load(ra, ks, base, ntask, row_bytes, half_off);
    k.store(ra, kd, tab, half_off, scale, inv_scale);
  }
}

// The re-rotation in the flat form (kv_flat.h): each wave moves one piece of
// a unit, V as it is, K rotated, one 16-byte vector of each per lane. A piece
// is 64 vectors where neox partners sit a power of two of at most 32 vectors
// apart inside a row (and for gptj, whose pairs sit inside one vector), else
// the whole rows that fit in 64 vectors (head_dim 80, 96, 192: 48 to 60 of the
// 64 lanes), so that a vector's partner is always another lane of its wave.
// The page's (cos, sin) table goes through the wave's own part of LDS: no
// barrier, and a wave that copies leaves at once. In LDS every column of pairs
// is followed by 16 bytes, so that the columns a wave reads start in different
// banks (unpadded they are 64 or 128 bytes apart).
// LAYOUT: token-major; split-x K (kx_phys on both sides, partners lane ^ 32);
// head-major cache pages (records token-major, cache vector hnd_vec(i)).
constexpr int kRotNhd = 0, kRotKx = 1, kRotHnd = 2;

template <int DT, int STYLE, int LAYOUT, int POLICY>
__global__ __launch_bounds__(kThreads) void kv_flat_rerotate_kernel(RotArgs ra, FlatMap m,
                                                                    FastDiv row, int piece_vecs) {
  extern __shared__ float2 lds_tab[];
  const UnitArgs& a = ra.u;
  FlatPos u;
  if (!flat_pos<false>(a, m, &u)) return;
  const int lane = (int)threadIdx.x % kWave;
  const int first = (int)u.part * piece_vecs;
  const int nvec = (int)(a.page_bytes >> 4);
  const int i = first + lane;
  const bool whole = LAYOUT != kRotNhd;  // descriptors of the whole page
  const int64_t po = whole ? 0 : (int64_t)first << 4;
  const int64_t left = a.page_bytes - po;
  const int64_t n = whole || left < ((int64_t)piece_vecs << 4) ? left : (int64_t)piece_vecs << 4;
  const bool in = i < nvec && lane < piece_vecs;
  const int out = (int)n;  // an offset outside the descriptors: reads 0, dropped
  const int p = LAYOUT == kRotKx ? kx_phys(ra, i) : i;  // the K vector of the record
  int kr = lane << 4, vr = kr, kc = kr, vc = kr;
  if (whole) {
    kr = in ? p << 4 : out;
    vr = in ? i << 4 : out;
    kc = LAYOUT == kRotHnd ? (in ? hnd_vec(a, i) << 4 : out) : kr;
    vc = LAYOUT == kRotHnd ? kc : vr;
  }
  const u32x4 v = bload(make_rsrc(u.rec + po + a.page_bytes, n), vr);
  const u32x4 k = bload(make_rsrc(u.rec + po, n), kr);
  const rsrc_t kd = make_rsrc(u.cache + po, n), vd = make_rsrc(u.cache + po + a.kv_stride, n);
  const int ti = rope_table(ra, u.page, u.layer);
  if (ti < 0) {
    bstore_as<POLICY>(vd, vc, v);
    bstore_as<POLICY>(kd, kc, k);
    return;
  }
  constexpr int kCol = STYLE == DSR_ROPE_NEOX ? Codec<DT>::VE : Codec<DT>::VE / 2;
  float2* const tab = lds_tab + (threadIdx.x / kWave) * (ra.rot_half + ra.rot_half / kCol * 2);
  const float2* const src_tab = ra.cos_sin + (int64_t)ti * ra.rot_half;
  float scale = 1.0f, inv_scale = 1.0f;
  if (is_fp8<DT>()) {
    scale = ra.k_scale[a.layer0 + u.layer];
    inv_scale = 1.0f / scale;
  }
  for (int j = lane; j < ra.rot_half; j += kWave) tab[j + j / kCol * 2] = src_tab[j];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  bstore_as<POLICY>(vd, vc, v);
  int c;
  if (LAYOUT == kRotKx)
    c = k_column<true>(ra, p);
  else
    c = i - (int)(div_by((uint32_t)i, row) * row.d);
  u32x4 q = k;
  if (STYLE == DSR_ROPE_NEOX) {
    const int h = ra.half_vecs;
    const int from = LAYOUT == kRotKx ? lane ^ 32 : c < h ? lane + h : c < 2 * h ? lane - h : lane;
#pragma unroll
    for (int w = 0; w < 4; ++w) q[w] = (unsigned)__shfl((int)k[w], from);
  }
  const int j0 = c < ra.rot_vecs ? table_column<DT, STYLE>(ra, c) : 0;
  bstore_as<POLICY>(kd, kc, rotate_vec<DT, STYLE>(ra, k, q, c, tab + j0 + j0 / kCol * 2, scale,
                                                  inv_scale));
}

// Any even rot_dim and either style, for rotary widths that do not fill
// whole 16-byte vectors (partial rotary of 24 or 20 dims, ...). A chunk of
// the page's K rows is staged in LDS; each lane decodes one output vector,
// rotates its elements below rot_dim with partners read element by element
// from LDS (a neox partner may straddle vectors), re-encodes, and keeps the
// raw bits of the elements at or past rot_dim through a bit mask. One unit
// per workgroup, layer-major; V is copied alongside.
template <int DT>
__device__ __forceinline__ float elem_decode(uint32_t bits) {
  if (DT == DSR_DTYPE_BF16) return bf16_to_f32(bits);
  if (DT == DSR_DTYPE_FP16) return fp16_to_f32(bits);
  if (DT == DSR_DTYPE_FP8_E5M2) return __builtin_amdgcn_cvt_pk_f32_bf8((int)bits, false)[0];
  return __builtin_amdgcn_cvt_pk_f32_fp8((int)bits, false)[0];
}

template <int DT, int STYLE>
__global__ __launch_bounds__(kThreads) void kv_scatter_rerotate_lds_kernel(RotArgs ra) {
  using C = Codec<DT>;
  constexpr int VE = C::VE;
  constexpr int EB = is_fp8<DT>() ? 8 : 16;  // bits per element
  constexpr int PER = 32 / EB;                           // elements per dword
  constexpr bool kScaled = is_fp8<DT>();
  constexpr int kChunkVecs = 2048;  // 32 KiB of K rows per pass
  __shared__ u32x4 buf[kChunkVecs];
  __shared__ float2 tab[kMaxRotHalf];
  uint8_t *cache, *rec;
  int l;
  const int64_t u = layer_major_unit(ra.u.n_units, ra.u.n_layers);
  if (u < 0 || !unit_addresses(ra.u, u, &cache, &rec, &l)) return;
  const int64_t p = udiv32(u, ra.u.n_layers);
  const int ti = rope_table(ra, p, l);
  const int64_t pb = ra.u.page_bytes;
  uint8_t* const vrec = rec + pb;
  uint8_t* const vcache = cache + ra.u.kv_stride;
  if (ti < 0) {
    copy_halves<kRotCopyUnroll>(rec, vrec, cache, vcache, pb);
    return;
  }
  const rsrc_t ks = make_rsrc(rec, pb), kd = make_rsrc(cache, pb);
  const rsrc_t vs = make_rsrc(vrec, pb), vd = make_rsrc(vcache, pb);
  const int nvec = (int)(pb >> 4);
  {
    VRound<kRotCopyUnroll> v;  // V: a plain copy
    for (int base = threadIdx.x; base < nvec; base += kThreads * kRotCopyUnroll) {
      v.load(vs, base, nvec);
      v.store(vd, base, nvec);
    }
  }
  const float2* src_tab = ra.cos_sin + (int64_t)ti * ra.rot_half;
  for (int j = threadIdx.x; j < ra.rot_half; j += kThreads) tab[j] = src_tab[j];
  float scale = 1.0f, inv_scale = 1.0f;
  if (kScaled) {
    scale = ra.k_scale[ra.u.layer0 + l];
    inv_scale = 1.0f / scale;
    if (scale_is_exact(scale)) scale = inv_scale = 1.0f;
  }
  const uint32_t* bw = reinterpret_cast<const uint32_t*>(buf);
  const int rv = ra.row_vecs, half = ra.rot_half, rot = 2 * ra.rot_half;
  const int rows = nvec / rv, rpc = kChunkVecs / rv;
  for (int r0 = 0; r0 < rows; r0 += rpc) {
    const int nv = (rows - r0 < rpc ? rows - r0 : rpc) * rv;
    __syncthreads();  // the previous chunk's readers are done (and the table is in)
    for (int i = threadIdx.x; i < nv; i += kThreads) buf[i] = bload(ks, (r0 * rv + i) << 4);
    __syncthreads();
    for (int i = threadIdx.x; i < nv; i += kThreads) {
      const int row = i / rv, c = i - row * rv;
      const u32x4 own = buf[i];
      float x[VE];
      C::decode(own, x);
      u32x4 mask = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int e = 0; e < VE; ++e) {
        const int j = c * VE + e;
        if (j >= rot) continue;
        int pj, jj;
        float sg;
        if (STYLE == DSR_ROPE_NEOX) {
          const bool first = j < half;
          pj = first ? j + half : j - half;
          jj = first ? j : j - half;
          sg = first ? -1.0f : 1.0f;
        } else {
          pj = j ^ 1;
          jj = j >> 1;
          sg = (j & 1) ? 1.0f : -1.0f;
        }
        const int pe = pj % VE;
        const uint32_t word = bw[(row * rv + pj / VE) * 4 + pe / PER];
        const float pv = elem_decode<DT>((word >> (EB * (pe % PER))) & ((1u << EB) - 1u));
        const float2 cs = tab[jj];
        const float xo = kScaled ? x[e] * scale : x[e];
        const float xp = kScaled ? pv * scale : pv;
        const float y = __builtin_fmaf(xo, cs.x, sg * xp * cs.y);
        x[e] = kScaled ? y * inv_scale : y;
        mask[e / PER] |= ((1u << EB) - 1u) << (EB * (e % PER));
      }
      const u32x4 enc = C::encode(x);
      bstore(kd, (r0 * rv + i) << 4, (enc & mask) | (own & ~mask));
    }
  }
}

}  // namespace
