// kv_flat.h -- page gather and scatter as one flat run of 1 KiB pieces.
// Part of libdaser_kv: included by kv_move.hip, one translation unit.
//
// A unit (page, layer) is cut into pieces of one wave instruction, 1 KiB of
// its K run and the same 1 KiB of its V run, and each wave moves one piece: 2
// loads and 2 stores per lane, whatever the page size. What bounds these
// copies is how many different DRAM rows the chip writes at once. Plain write
// streams run at 7.2-7.4 TB/s while the addresses in flight span 4 MiB, 6.9 at 8,
// 6.3 at 16 and 5.6-5.9 TB/s from 32 MiB up, reads at 7.2 or more throughout;
// so waves should hold little each and be dealt out in address order. A
// workgroup that moves a whole 32 KiB page holds 64 KiB, spread over 16
// stretches of the chip's window; 16 waves of one piece per CU hold 8 MiB of
// the destination in all, in order.
// Measured against workgroups of whole units (16 KiB pages 1,127 of 28
// layers, 64 KiB pages 42 layers, both ways in one process): scatter 5.54 ->
// 6.11 and 5.90 -> 6.57 TB/s, gather 5.94 -> 6.26 and 6.57 -> 6.57; 4 KiB pages
// scatter 5.32 -> 5.94; a 16-page load of 24 layers takes 3.4 us, by the
// profiler.

#pragma once

#include "kv_common.h"

namespace {

// Exact division of any 32-bit n by a launch constant (Granlund and
// Montgomery's multiply and shift): the compiler's sequence for a runtime
// divisor is some 20 instructions, and every wave divides twice.
struct FastDiv {
  uint32_t d, m, s1, s2;
};
inline FastDiv fast_div(uint32_t d) {
  uint32_t l = 0;
  while (l < 32 && (1ull << l) < d) ++l;
  FastDiv f;
  f.d = d;
  f.m = (uint32_t)((((1ull << l) - d) << 32) / d + 1);
  f.s1 = l < 1 ? l : 1;
  f.s2 = l > 1 ? l - 1 : 0;
  return f;
}
__device__ __forceinline__ uint32_t div_by(uint32_t n, const FastDiv& f) {
  const uint32_t t = __umulhi(f.m, n);
  return (t + ((n - t) >> f.s1)) >> f.s2;
}

constexpr int kPiece = kWave * 16;  // bytes of one wave instruction

// Consecutive workgroups of a large launch that stay on one XCD: 128 (512 KiB
// of K). Dealt one by one, every XCD translates every page's addresses and
// the same page's lines meet in 8 L2s; in XCD-contiguous eighths, 8 windows
// are written at once. Against chunks of 32, 128 were 0-1% ahead at 4 and 32 KiB
// pages and 1-3% at 64 and 96 KiB ones and at 80 layers of e4m3; of 16, 1-6%;
// of 1,024 and 16,384, 0-2%.
constexpr uint32_t kChunk = 128;
// Launches whose pages share records: each XCD takes one contiguous eighth of
// the waves (copy_shape in kv_move.hip has the figures).
constexpr uint32_t kEighths = ~0u;
constexpr uint32_t kEighthsBit = 1u << 31;

// The waves of one launch: wave w of it moves piece wave0 + w, counted from
// the first piece of unit unit0.
struct FlatMap {
  FastDiv per_unit;  // pieces per unit
  FastDiv minor;     // page-major: layers; layer-major: pages
  uint32_t unit0, wave0, n_waves;
  // workgroups below it are dealt to the XCDs in chunks of kChunk; or kEighthsBit and
  // an eighth of the grid
  uint32_t chunked;
};

struct FlatPos {
  const uint8_t* cache;
  const uint8_t* rec;
  uint32_t page;  // entry of the page tables
  int layer;
  uint32_t part;  // piece of the unit
};

// This wave's number in the launch, in the order of the chunks or eighths. Without a
// branch: with one, the compiler fetches the other arguments in more rounds, and a
// step of 32 gathers of 17 MB takes 167 us, not 159.
__device__ __forceinline__ uint32_t flat_wave(const FlatMap& m) {
  uint32_t b = blockIdx.x;
  const uint32_t x = b % kXcds, j = b / kXcds;
  const uint32_t chunk = b < m.chunked ? (j / kChunk * kXcds + x) * kChunk + j % kChunk : b;
  const uint32_t eighth = x * (m.chunked & ~kEighthsBit) + j;
  b = chunk ^ ((chunk ^ eighth) & -(m.chunked >> 31));
  return b * (kThreads / kWave) +
         (uint32_t)__builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
}

// This wave's piece; false past the end of the launch and where the unit's
// block id or record range is out of bounds (it is then skipped). Page-major:
// the records are written in sequence; layer-major: the destination-ordered
// pages of one layer are. Everything here is uniform over the wave.
template <bool kPageMajor>
__device__ __forceinline__ bool flat_pos(const UnitArgs& a, const FlatMap& m, FlatPos* o) {
  const uint32_t w = flat_wave(m);
  if (w >= m.n_waves) return false;
  const uint32_t g = m.wave0 + w;
  const uint32_t q = div_by(g, m.per_unit);
  o->part = g - q * m.per_unit.d;
  const uint32_t v = m.unit0 + q;
  const uint32_t hi = div_by(v, m.minor);
  const uint32_t lo = v - hi * m.minor.d;
  const uint32_t p = kPageMajor ? hi : lo, l = kPageMajor ? lo : hi;
  const int64_t blk = a.page_ids[p];
  const int64_t off = a.slot_offsets[p] + (int64_t)(a.layer0 + (int)l) * a.layer_bytes;
  if (blk < 0 || blk >= a.num_blocks) return false;
  if (off < 0 || off + 2 * a.page_bytes > a.staging_bytes) return false;
  o->cache = reinterpret_cast<const uint8_t*>(a.layer_base[l]) + blk * a.page_stride;
  o->rec = a.staging + off;
  o->page = p;
  o->layer = (int)l;
  return true;
}

template <int POLICY>
__device__ __forceinline__ void bstore_as(rsrc_t r, int off, u32x4 v) {
  __builtin_amdgcn_raw_buffer_store_b128(v, r, off, 0, POLICY);
}

// Gather (page-major) or scatter (layer-major). U: consecutive pieces per
// wave (1, or 8 in launches that fit the chip once). POLICY: the stores'
// cache policy. HND: head-major cache pages, whose cache side goes through
// hnd_vec; the piece of a page's end is clipped by its descriptors.
template <bool kGather, bool HND, int POLICY, int U = 1>
__global__ __launch_bounds__(kThreads) void kv_flat_copy_kernel(UnitArgs a, FlatMap m) {
  FlatPos u;
  if (!flat_pos<kGather>(a, m, &u)) return;
  const int lane = (int)threadIdx.x % kWave;
  const int64_t first = (int64_t)u.part * (kPiece * U);
  const int64_t po = HND ? 0 : first;
  const int64_t left = a.page_bytes - po;
  const int64_t n = HND || left < kPiece * U ? left : kPiece * U;
  const uint8_t* c = u.cache + po;
  const uint8_t* r = u.rec + po;
  const rsrc_t ck = make_rsrc(c, n), cv = make_rsrc(c + a.kv_stride, n);
  const rsrc_t rk = make_rsrc(r, n), rv = make_rsrc(r + a.page_bytes, n);
  u32x4 xk[U], xv[U];
  int ro[U], co[U];
#pragma unroll
  for (int k = 0; k < U; ++k) {
    ro[k] = co[k] = k * kPiece + (lane << 4);
    if (HND) {
      const int i = (int)(first >> 4) + k * kWave + lane;
      const bool in = i < (int)(a.page_bytes >> 4);
      ro[k] = in ? i << 4 : (int)n;  // n: outside the descriptor, dropped
      co[k] = in ? hnd_vec(a, i) << 4 : (int)n;
    }
    xk[k] = bload(kGather ? ck : rk, kGather ? co[k] : ro[k]);
    xv[k] = bload(kGather ? cv : rv, kGather ? co[k] : ro[k]);
  }
#pragma unroll
  for (int k = 0; k < U; ++k) {
    bstore_as<POLICY>(kGather ? rk : ck, kGather ? ro[k] : co[k], xk[k]);
    bstore_as<POLICY>(kGather ? rv : cv, kGather ? ro[k] : co[k], xv[k]);
  }
}

}  // namespace
