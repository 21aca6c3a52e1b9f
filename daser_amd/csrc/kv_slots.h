// kv_slots.h -- token-granular (slot_mapping-driven) gather and scatter.
// Part of libdaser_kv: included by kv_move.hip, one translation unit.
//
// The flat form of the page kernels (kv_flat.h) over tokens: the unit is a run
// of tokens of one layer, cut into pieces of one wave instruction. Rows of 64
// vectors (1 KiB) and more are cut by themselves, so a wave's token is uniform,
// its table entries come by scalar loads and its addresses go into buffer
// descriptors. Shorter rows follow each other in the lanes, 64 vectors of
// whatever tokens come next, each lane with its token's entries and its own
// 64-bit addresses; every row length fills the wave. Invalid tokens (padding,
// out-of-range slots or records) are left out.

#pragma once

#include "kv_flat.h"
#include "kv_rotate.h"

namespace {

struct SlotArgs {
  const uint64_t* layer_base;
  int64_t kv_stride;
  int64_t page_stride;
  int64_t page_bytes;
  int64_t num_blocks;
  int64_t row_bytes;
  const int64_t* slot_mapping;
  const int64_t* row_offsets;
  uint8_t* staging;
  int64_t staging_bytes;
  int64_t layer_bytes;
  int32_t n_tokens;
  int32_t n_layers;
  int32_t layer0;
  int32_t block_size;
  int32_t block_shift;  // log2(block_size) when a power of two, else -1
  int32_t unit_tokens;  // tokens per unit
  int64_t least_row;    // the smallest row offset taken (dsr_gather_slots)
  FastDiv row;          // wide rows: pieces per row; others: vectors per row
};

// Block of a non-negative slot: a shift for power-of-two block sizes (all
// of vLLM's), else a 32-bit division where the slot fits.
__device__ __forceinline__ int64_t slot_block(const SlotArgs& a, int64_t slot) {
  if (a.block_shift >= 0) return slot >> a.block_shift;
  return slot < (int64_t)0xffffffffLL ? udiv32(slot, a.block_size) : slot / a.block_size;
}

// One lane's (short rows) or wave's (wide rows) place: token t, vector v of
// its row, the row's addresses.
struct SlotPos {
  uint8_t* cache;
  uint8_t* rec;
  int64_t t;
  int layer;
  int v;  // wide rows: first vector of the piece
};

// False past the end of the launch or the unit and for invalid tokens. Gather:
// the layers of a run of tokens follow each other (the records are written in
// sequence); scatter: the runs of a layer.
template <bool kGather, bool WIDE>
__device__ __forceinline__ bool slot_pos(const SlotArgs& a, const FlatMap& m, SlotPos* o) {
  const uint32_t w = flat_wave(m);
  if (w >= m.n_waves) return false;
  const uint32_t g = m.wave0 + w;
  const uint32_t q = div_by(g, m.per_unit);
  const uint32_t part = g - q * m.per_unit.d;
  const uint32_t u = m.unit0 + q;
  const uint32_t hi = div_by(u, m.minor);
  const uint32_t lo = u - hi * m.minor.d;
  const uint32_t tb = kGather ? hi : lo, l = kGather ? lo : hi;
  uint32_t in_unit;
  if (WIDE) {
    in_unit = div_by(part, a.row);
    o->v = (int)((part - in_unit * a.row.d) * kWave);
  } else {
    const uint32_t f = part * kWave + (uint32_t)threadIdx.x % kWave;
    in_unit = div_by(f, a.row);
    o->v = (int)(f - in_unit * a.row.d);
    if (in_unit >= (uint32_t)a.unit_tokens) return false;
  }
  const int64_t t = (int64_t)tb * a.unit_tokens + in_unit;
  if (t >= a.n_tokens) return false;
  const int64_t slot = a.slot_mapping[t], row = a.row_offsets[t];
  const int64_t off = row + (int64_t)(a.layer0 + (int)l) * a.layer_bytes;
  const int64_t blk = slot >= 0 ? slot_block(a, slot) : -1;
  if (blk < 0 || blk >= a.num_blocks || row < a.least_row) return false;
  if (off < 0 || off + a.page_bytes + a.row_bytes > a.staging_bytes) return false;
  o->cache = reinterpret_cast<uint8_t*>(a.layer_base[l]) + blk * a.page_stride +
             (slot - blk * a.block_size) * a.row_bytes;
  o->rec = a.staging + off;
  o->t = t;
  o->layer = (int)l;
  return true;
}

__device__ __forceinline__ u32x4 gload(const uint8_t* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
}
__device__ __forceinline__ void gstore(uint8_t* p, u32x4 v) {
  __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(p));
}

template <bool kGather, bool WIDE, int POLICY>
__global__ __launch_bounds__(kThreads) void kv_slots_flat_kernel(SlotArgs a, FlatMap m) {
  SlotPos u;
  if (!slot_pos<kGather, WIDE>(a, m, &u)) return;
  const int64_t po = (int64_t)u.v << 4;
  uint8_t* const src = (kGather ? u.cache : u.rec) + po;
  uint8_t* const dst = (kGather ? u.rec : u.cache) + po;
  const int64_t sv = kGather ? a.kv_stride : a.page_bytes;
  const int64_t dv = kGather ? a.page_bytes : a.kv_stride;
  if (WIDE) {
    const int64_t left = a.row_bytes - po;
    const int64_t n = left < kPiece ? left : kPiece;
    const int o = ((int)threadIdx.x % kWave) << 4;
    const u32x4 k = bload(make_rsrc(src, n), o), v = bload(make_rsrc(src + sv, n), o);
    bstore_as<POLICY>(make_rsrc(dst, n), o, k);
    bstore_as<POLICY>(make_rsrc(dst + dv, n), o, v);
  } else {
    const u32x4 k = gload(src), v = gload(src + sv);
    gstore(dst, k);
    gstore(dst + dv, v);
  }
}

// The load scatter with K re-rotated by each token's own (cos, sin) table.
// Heads are a power-of-two number of vectors (<= 64), so a head never leaves
// its piece and its neox partner sits half_vecs lanes away. Where all tokens of
// a wave use one table (always in wide rows, nearly always in a load of whole
// chunks) it goes through the wave's part of LDS, as in the page kernel; other
// lanes read their token's pairs themselves, 64 or 128 bytes for each 16 that
// they move (one-head e4m3 rows: 2.9 TB/s, 4.2 through LDS). Lanes without a valid
// token take part in the shuffles and move nothing.
// rot_dim <= 256. The kernel takes more (its tables are sized at launch); wider
// ones are refused, unmeasured.
constexpr int kSlotRotMaxHalf = 128;

template <int DT, int STYLE, bool WIDE, int POLICY>
__global__ __launch_bounds__(kThreads) void kv_slots_flat_rerotate_kernel(SlotArgs a, RotArgs ra,
                                                                          FlatMap m) {
  extern __shared__ float2 lds_tab[];
  SlotPos u{};
  const bool ok = slot_pos<false, WIDE>(a, m, &u);
  if (WIDE && !ok) return;
  const int lane = (int)threadIdx.x % kWave;
  int ti = -1;
  u32x4 k = {0u, 0u, 0u, 0u}, v = k;
  uint8_t* dst = nullptr;
  int64_t n = 0;
  if (ok) {
    const int64_t po = (int64_t)u.v << 4;
    const uint8_t* const src = u.rec + po;
    dst = u.cache + po;
    if (WIDE) {
      const int64_t left = a.row_bytes - po;
      n = left < kPiece ? left : kPiece;
      v = bload(make_rsrc(src + a.page_bytes, n), lane << 4);
      k = bload(make_rsrc(src, n), lane << 4);
    } else {
      v = gload(src + a.page_bytes);
      k = gload(src);
    }
    ti = rope_table(ra, u.t, u.layer);
  }
  float scale = 1.0f, inv_scale = 1.0f;
  if (is_fp8<DT>() && ok) {
    scale = ra.k_scale[a.layer0 + u.layer];
    inv_scale = 1.0f / scale;
  }
  constexpr int kCol = STYLE == DSR_ROPE_NEOX ? Codec<DT>::VE : Codec<DT>::VE / 2;
  const int c = (WIDE ? lane : u.v) & (ra.row_vecs - 1);
  const int j0 = c < ra.rot_vecs ? table_column<DT, STYLE>(ra, c) : 0;
  u32x4 q = k;
  if (STYLE == DSR_ROPE_NEOX) {
    const int from = c < ra.half_vecs ? lane + ra.half_vecs : lane - ra.half_vecs;
#pragma unroll
    for (int w = 0; w < 4; ++w) q[w] = (unsigned)__shfl((int)k[w], from);
  }
  const uint64_t valid = __ballot(ok);
  if (valid == 0) return;
  const int ti0 = __builtin_amdgcn_readlane(ti, __builtin_ctzll(valid));
  if (WIDE || __ballot(ok && ti != ti0) == 0) {
    if (ti0 >= 0) {
      float2* const tab = lds_tab + (threadIdx.x / kWave) * (ra.rot_half + ra.rot_half / kCol * 2);
      const float2* const src_tab = ra.cos_sin + (int64_t)ti0 * ra.rot_half;
      for (int j = lane; j < ra.rot_half; j += kWave) tab[j + j / kCol * 2] = src_tab[j];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      k = rotate_vec<DT, STYLE>(ra, k, q, c, tab + j0 + j0 / kCol * 2, scale, inv_scale);
    }
  } else if (ti >= 0) {
    k = rotate_vec<DT, STYLE>(ra, k, q, c, ra.cos_sin + (int64_t)ti * ra.rot_half + j0, scale,
                              inv_scale);
  }
  if (WIDE) {
    bstore_as<POLICY>(make_rsrc(dst + a.kv_stride, n), lane << 4, v);
    bstore_as<POLICY>(make_rsrc(dst, n), lane << 4, k);
  } else if (ok) {
    gstore(dst + a.kv_stride, v);
    gstore(dst, k);
  }
}

}  // namespace
