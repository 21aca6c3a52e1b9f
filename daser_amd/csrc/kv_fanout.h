// kv_fanout.h -- loads in which several pages read the same record (a cached
// chunk placed in several requests): each source record is read once and
// written to every page that loads it, K re-rotated per destination.
// Part of libdaser_kv: included by kv_move.hip, one translation unit.
//
// The per-page scatter reads a shared record once per destination page, so a
// chunk placed in 16 requests is read 16 times (partly from the memory-side
// cache). Here a wave holds one piece (kv_flat.h) of a source's K and V of one
// layer and writes it to each destination, V as is and K rotated by that
// destination's delta table. Reads drop to one pass over the distinct records;
// the writes are the same.

#pragma once

#include "kv_rotate.h"

namespace {

struct FanArgs {
  RotArgs ra;  // caches, staging, geometry, tables, scales (ra.u's page tables unused)
  const int64_t* src_offsets;  // n_src record offsets (layer 0 of the record)
  const int32_t* dst_start;    // n_src + 1: destinations of source s are [start[s], start[s+1])
  const int32_t* dst_pages;    // block id of each destination
  const int32_t* dst_rope;     // table index of each destination (-1: K copied); null: no rotation
  int32_t n_src;
  int32_t n_dst;               // for the launch's shape
};

// A destination's table is fetched while the one before is being written (the
// first 128 pairs; wider tables read the rest when they are needed). ROT false:
// a plain copy. Cache layouts (LAYOUT) as in kv_flat_rerotate_kernel; POLICY: the
// stores' cache policy. A source's destinations may be dealt to several waves
// (`split` shares of each piece): where few waves hold many destinations, each a
// table's way through LDS after the other, that chain bounds the load.
template <int DT, int STYLE, int LAYOUT, bool ROT, int POLICY>
__global__ __launch_bounds__(kThreads) void kv_fanout_kernel(FanArgs fa, FlatMap m, FastDiv row,
                                                             FastDiv pieces, int split,
                                                             bool layer_major) {
  extern __shared__ float2 lds_tab[];
  const RotArgs& ra = fa.ra;
  const UnitArgs& a = ra.u;
  const uint32_t w = flat_wave(m);
  if (w >= m.n_waves) return;
  const uint32_t g = m.wave0 + w;
  const uint32_t qu = div_by(g, m.per_unit);
  const uint32_t share = div_by(g - qu * m.per_unit.d, pieces);
  const uint32_t part = g - qu * m.per_unit.d - share * pieces.d;
  const uint32_t un = m.unit0 + qu;
  const uint32_t hi = div_by(un, m.minor);
  const uint32_t lo = un - hi * m.minor.d;
  const uint32_t s = layer_major ? lo : hi, l = layer_major ? hi : lo;
  const int64_t off = fa.src_offsets[s] + (int64_t)(a.layer0 + (int)l) * a.layer_bytes;
  const int all0 = fa.dst_start[s], all1 = fa.dst_start[s + 1];
  const int each = (all1 - all0 + split - 1) / split;
  const int d0 = all0 + (int)share * each;
  const int d1 = d0 + each < all1 ? d0 + each : all1;
  if (off < 0 || off + 2 * a.page_bytes > a.staging_bytes || d1 <= d0) return;
  const int lane = (int)threadIdx.x % kWave;
  const int first = (int)part * kWave;
  const int nvec = (int)(a.page_bytes >> 4);
  const int i = first + lane;
  const bool whole = LAYOUT != kRotNhd;
  const int64_t po = whole ? 0 : (int64_t)first << 4;
  const int64_t left = a.page_bytes - po;
  const int64_t n = whole || left < kPiece ? left : kPiece;
  const bool in = i < nvec;
  const int out = (int)n;
  const int p = LAYOUT == kRotKx ? kx_phys(ra, i) : i;
  int kr = lane << 4, vr = kr, kc = kr, vc = kr;
  if (whole) {
    kr = in ? p << 4 : out;
    vr = in ? i << 4 : out;
    kc = LAYOUT == kRotHnd ? (in ? hnd_vec(a, i) << 4 : out) : kr;
    vc = LAYOUT == kRotHnd ? kc : vr;
  }
  const uint8_t* const rec = a.staging + off + po;
  const u32x4 k = bload(make_rsrc(rec, n), kr);
  const u32x4 v = bload(make_rsrc(rec + a.page_bytes, n), vr);
  uint8_t* const lbase = reinterpret_cast<uint8_t*>(a.layer_base[l]) + po;
  const int grp = ROT && ra.layer_group ? ra.layer_group[a.layer0 + (int)l] : 0;
  const bool rot_layer = ROT && grp >= 0 && grp < ra.n_groups;
  float scale = 1.0f, inv_scale = 1.0f;
  if (is_fp8<DT>() && rot_layer) {
    scale = ra.k_scale[a.layer0 + (int)l];
    inv_scale = 1.0f / scale;
  }
  constexpr int kCol = STYLE == DSR_ROPE_NEOX ? Codec<DT>::VE : Codec<DT>::VE / 2;
  const int rh = ra.rot_half;
  float2* const tab = lds_tab + (threadIdx.x / kWave) * (rh + rh / kCol * 2);
  int c = 0, j0 = 0;
  u32x4 q = k;
  if (ROT) {
    c = LAYOUT == kRotKx ? k_column<true>(ra, p) : i - (int)(div_by((uint32_t)i, row) * row.d);
    j0 = c < ra.rot_vecs ? table_column<DT, STYLE>(ra, c) : 0;
    if (STYLE == DSR_ROPE_NEOX) {
      const int from = LAYOUT == kRotKx ? lane ^ 32 : lane ^ ra.half_vecs;
#pragma unroll
      for (int x = 0; x < 4; ++x) q[x] = (unsigned)__shfl((int)k[x], from);
    }
  }
  // 64 destinations at a time: lane d holds the d-th one's block and table
  for (int db = d0; db < d1; db += kWave) {
    const int nb = d1 - db < kWave ? d1 - db : kWave;
    const int my_blk = lane < nb ? fa.dst_pages[db + lane] : -1;
    int my_ti = -1;
    if (rot_layer && lane < nb) {
      my_ti = fa.dst_rope[db + lane];
      my_ti = my_ti >= 0 && my_ti < ra.n_tables ? grp * ra.n_tables + my_ti : -1;
    }
    float2 next[ROT ? 2 : 1];  // the next destination's table, this lane's pairs
    auto fetch = [&](int t) {
      const int ti = __builtin_amdgcn_readlane(my_ti, t);
      if (ti >= 0) {
        const float2* src = ra.cos_sin + (int64_t)ti * rh;
#pragma unroll
        for (int x = 0; x < 2; ++x)
          if (lane + x * kWave < rh) next[x] = src[lane + x * kWave];
      }
    };
    if (ROT) fetch(0);
    for (int t = 0; t < nb; ++t) {
      const int64_t blk = __builtin_amdgcn_readlane(my_blk, t);
      const int ti = ROT ? __builtin_amdgcn_readlane(my_ti, t) : -1;
      u32x4 kk = k;
      if (ROT) {
        if (ti >= 0) {
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            const int j = lane + x * kWave;
            if (j < rh) tab[j + j / kCol * 2] = next[x];
          }
          for (int j = lane + 2 * kWave; j < rh; j += kWave)
            tab[j + j / kCol * 2] = ra.cos_sin[(int64_t)ti * rh + j];
        }
        if (t + 1 < nb) fetch(t + 1);
        if (ti >= 0) {
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
          kk = rotate_vec<DT, STYLE>(ra, k, q, c, tab + j0 + j0 / kCol * 2, scale, inv_scale);
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
        }
      }
      if (blk < 0 || blk >= a.num_blocks) continue;  // skipped, as by the page scatter
      uint8_t* const cache = lbase + blk * a.page_stride;
      bstore_as<POLICY>(make_rsrc(cache + a.kv_stride, n), vc, v);
      bstore_as<POLICY>(make_rsrc(cache, n), kc, kk);
    }
  }
}

}  // namespace
