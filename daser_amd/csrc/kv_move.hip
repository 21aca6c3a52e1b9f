// kv_move.hip -- gfx950 kernels and C ABI for DaseR's KV data-movement path.
//
// Three operations, all HBM-bandwidth bound (no contraction, no MFMA):
//   dsr_gather            paged block cache  -> contiguous slot records
//   dsr_scatter           slot records       -> paged block cache
//   dsr_scatter_rerotate  slot records       -> paged block cache, with the K
//                         half of selected pages rotated by a RoPE position
//                         delta in fp32 on the way through.
//
// Work decomposition. A vLLM page (block_size tokens x H heads x D dims) is
// contiguous inside each per-layer cache; only the block index is permuted.
// The unit of work is therefore one (page, layer): two contiguous runs of
// page_bytes (K and V) on each side, moved with 16-byte lane vectors
// (buffer_load_dwordx4 / buffer_store_dwordx4 through descriptors bounded to
// the run) by waves of 1 KiB each way (kv_flat.h). No LDS is needed for the
// copy: both sides are contiguous within a unit. The re-rotation kernels
// keep the unit's (cos, sin) table in LDS.
//
// Kernel choice, by page and row geometry (all inside the entry points):
//   gather / scatter, every page size, token-major and head-major:
//     kv_flat_copy_kernel (1 KiB pieces, one per wave).
//   re-rotation: kv_flat_rerotate_kernel (1 KiB pieces, or the whole rows in 64
//     vectors) for gptj, for neox rows with a power-of-two partner distance
//     and for other neox rows of <= 64 vectors; the pair-task
//     kv_scatter_rerotate_kernel otherwise; rotary widths that are not whole
//     16-byte vectors: kv_scatter_rerotate_lds_kernel.
//   token form (dsr_*_slots): the flat kernels over tokens (kv_slots.h).
//   split-x K pages (dsr_scatter_rerotate_kx): the flat kernel with the
//     split-x vector map, or the pair-task kernel.
//   head-major cache pages (dsr_*_hnd): the same kernels as token-major
//     pages of that size with the HND flag, whose cache-side offsets go
//     through hnd_vec.
// Calls too large for one launch run as several over page (token) ranges.
//
// Reference being replaced: the Python per-(request, block, layer) torch
// copy_ loops of daser/connector/daser_connector.py:536-551 (load) and
// :610-632 (save).

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <mutex>

#include "daser_kv.h"

#include "kv_common.h"
#include "kv_flat.h"
#include "kv_rotate.h"
#include "kv_slots.h"
#include "kv_fanout.h"

namespace {

bool aligned16(int64_t v) { return (v & 15) == 0; }
bool aligned16p(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int check_common(const uint64_t* layer_base, int n_layers, int64_t kv_stride,
                 int64_t page_stride, int64_t page_bytes, int64_t num_blocks,
                 const int32_t* page_ids, const int64_t* slot_offsets,
                 int n_pages, const void* staging, int64_t staging_bytes,
                 int64_t layer_bytes, int layer0) {
  if (n_pages < 0 || n_layers < 0 || layer0 < 0 || num_blocks < 0 ||
      staging_bytes < 0 || page_bytes <= 0)
    return DSR_ERR_ARG;
  if (n_pages == 0 || n_layers == 0) return DSR_OK;
  if (!layer_base || !page_ids || !slot_offsets || !staging) return DSR_ERR_ARG;
  if (layer_bytes < 2 * page_bytes) return DSR_ERR_SHAPE;
  if (page_bytes > 0x7fffffffLL) return DSR_ERR_SHAPE;  // one buffer descriptor per run
  if ((int64_t)n_pages * n_layers > 0x7fffffffLL) return DSR_ERR_ARG;
  if (!aligned16(kv_stride) || !aligned16(page_stride) || !aligned16(page_bytes) ||
      !aligned16(layer_bytes) || !aligned16p(staging))
    return DSR_ERR_ALIGN;
  return DSR_OK;
}

UnitArgs make_unit(const uint64_t* layer_base, int n_layers, int64_t kv_stride,
                   int64_t page_stride, int64_t page_bytes, int64_t num_blocks,
                   const int32_t* page_ids, const int64_t* slot_offsets,
                   int n_pages, const void* staging, int64_t staging_bytes,
                   int64_t layer_bytes, int layer0) {
  UnitArgs a{};
  a.layer_base = layer_base;
  a.kv_stride = kv_stride;
  a.page_stride = page_stride;
  a.page_bytes = page_bytes;
  a.num_blocks = num_blocks;
  a.page_ids = page_ids;
  a.slot_offsets = slot_offsets;
  a.staging = const_cast<uint8_t*>(static_cast<const uint8_t*>(staging));
  a.staging_bytes = staging_bytes;
  a.layer_bytes = layer_bytes;
  a.n_layers = n_layers;
  a.layer0 = layer0;
  a.n_units = (int64_t)n_pages * n_layers;
  return a;
}

// Largest workgroup count of one launch: HIP caps gridDim.x * blockDim.x at
// 2^32 - 1 threads (16.7 M workgroups of 256). The DSR_TUNE_MAX_WG_PER_LAUNCH
// override lowers it, so that tests can exercise the split.
int64_t max_wg_per_launch() {
  int64_t m = 0xffffffffLL / kThreads / kXcds * kXcds;
  if (const int64_t t = tune(DSR_TUNE_MAX_WG_PER_LAUNCH)) {
    const int64_t v = t / kXcds * kXcds;
    if (v >= 2 * kXcds && v < m) m = v;
  }
  return m;
}

// Launches over consecutive page ranges of `a` (one launch unless the pages
// exceed max_wg_per_launch()), each range's tables offset to its first
// page; launch(b, grid) enqueues one kernel. Grids are a whole multiple of
// the XCD count so that the XCD remap covers every unit. Returns the first
// launch error.
template <class F>
int launch_page_ranges(const UnitArgs& a, int n_pages, F launch) {
  const int64_t per = (max_wg_per_launch() - kXcds) / a.n_layers;
  if (per <= 0) return DSR_ERR_ARG;
  for (int64_t p0 = 0; p0 < n_pages; p0 += per) {
    const int64_t n = n_pages - p0 < per ? n_pages - p0 : per;
    UnitArgs b = a;
    b.page_ids += p0;
    b.slot_offsets += p0;
    b.n_units = n * a.n_layers;
    const unsigned grid = (unsigned)((b.n_units + kXcds - 1) / kXcds * kXcds);
    launch(b, grid);
    const int rc = (int)hipGetLastError();
    if (rc != 0) return rc;
  }
  return DSR_OK;
}

// Launches of a flat kernel over every piece of n_units units (one launch
// unless the workgroups exceed max_wg_per_launch()), `minor` the inner extent
// of the unit order: launch(map, grid). `chunk`: consecutive workgroups that stay
// on one XCD (0: dealt one by one; kEighths).
template <class F>
int launch_flat(int64_t n_units, int64_t pieces_per_unit, int64_t minor, uint32_t chunk, F launch) {
  constexpr int kWaves = kThreads / kWave;
  const int64_t total = n_units * pieces_per_unit;
  const int64_t per = max_wg_per_launch() * kWaves;
  for (int64_t g0 = 0; g0 < total; g0 += per) {
    const int64_t n = total - g0 < per ? total - g0 : per;
    unsigned grid = (unsigned)((n + kWaves - 1) / kWaves);
    FlatMap m;
    m.per_unit = fast_div((uint32_t)pieces_per_unit);
    m.minor = fast_div((uint32_t)minor);
    m.unit0 = (uint32_t)(g0 / pieces_per_unit);
    m.wave0 = (uint32_t)(g0 % pieces_per_unit);
    m.n_waves = (uint32_t)n;
    if (chunk == kEighths) grid = (grid + kXcds - 1) / kXcds * kXcds;  // the rest leave at once
    m.chunked = chunk == kEighths ? kEighthsBit | grid / kXcds
                : chunk == kChunk ? grid / (kXcds * kChunk) * (kXcds * kChunk) : 0;
    launch(m, grid);
    const int rc = (int)hipGetLastError();
    if (rc != 0) return rc;
  }
  return DSR_OK;
}

// Workgroups per CU for the pair-task re-rotation kernel, applied with dynamic
// LDS sized from the CU's LDS capacity: 16-bit K (64 KiB per unit at the
// Llama-3-8B shape) ran best at 2-3 per CU, e4m3 (32 KiB) at 4.
template <int DT>
constexpr int rot_wg_per_cu() {
  return is_fp8<DT>() ? 4 : 2;
}
// Dynamic LDS that limits a kernel with `static_lds` bytes of static LDS to
// wg_per_cu workgroups per CU on the current device (0 if the capacity cannot
// be read). The capacity is read once per device.
constexpr int64_t kLdsGranule = 512;
constexpr int kMaxDevices = 64;
std::atomic<int> g_lds_per_cu[kMaxDevices];
size_t occupancy_lds(int wg_per_cu, int64_t static_lds) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || wg_per_cu <= 0) return 0;
  int lds = dev < kMaxDevices ? g_lds_per_cu[dev].load(std::memory_order_relaxed) : 0;
  if (lds <= 0) {
    if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor,
                              dev) != hipSuccess || lds <= 0)
      return 0;
    if (dev < kMaxDevices) g_lds_per_cu[dev].store(lds, std::memory_order_relaxed);
  }
  // a workgroup's LDS (static plus dynamic) is allocated in 512-byte
  // granules: round its share down so that wg_per_cu of them fit
  const int64_t share = (int64_t)lds / wg_per_cu / kLdsGranule * kLdsGranule;
  const int64_t want = share - static_lds;
  return want > 0 ? (size_t)want : 0;
}

// Launch shape of a page copy, by the bytes it moves (read + written).
// Measured per kernel in graphs of some 100 launches on 8 to 16 sets of buffers
// in turn (more than the memory-side cache holds), Llama-3-8B pages, one
// workgroup per unit -> the class's choice:
//   up to 200 MiB: nt stores, which the L2s absorb while the pages are read:
//     one-chunk loads 4.98 -> 2.92 us at 8.4 MB, 5.82 -> 4.52 at 17 MB, 20.9 ->
//     18.1 at 101 MB, 32.7 -> 28.4 at 168 MB (sc0 sc1 stores 3.84, 5.45, 19.5,
//     29.9); a layer's save 4.27 -> 3.17 us at 8.4 MB, 5.49 -> 4.52 at 17 MB;
//   of these, from 20 to 32 MiB, which is one workgroup per CU: each wave holds
//     8 KiB of K and of V, so that no second generation of waves starts: 7.14 ->
//     5.77 us at 29 MB (single pieces 6.53), a layer's save 7.24 -> 6.24 at 34;
//   above: nt sc0 sc1 stores, in chunks of workgroups (kChunk): 50.3 -> 42.1
//     us at 268 MB (nt 42.9), 185 -> 163 at 1.07 GB (nt 169), 738 -> 664 at 4.3
//     GB (nt 681).
// Where the same buffers come again at once and stay in the memory-side cache, the
// replaced kernels' sc0 sc1 stores were 10-20% ahead from 60 to 500 MB moved (8B
// gather of 500 MB 62.1 -> 78.5 us; on four sets in turn 83.4 -> 78.8, scatter 92.2 ->
// 76.3); a load's pages and records are not there.
// Four workgroups of single pieces per CU: 32 KiB of reads in flight there hide
// the latency, and 6 or 8 per CU widen the written window (0-8% slower).
constexpr int kCopyWgPerCu = 4;
//
// Several pages reading the same records (DSR_SHARED_RECORDS): kEighths at every
// size, copies at 6 workgroups per CU. Without the flag -> with it, and the
// per-page kernels of one workgroup per unit: Llama-3-70B, 32,768 pages of 2,048
// records 50.9 -> 49.5 ms (50.2), its TP8 share 6.24 -> 6.14 (6.69); re-rotation
// 50.1 -> 49.0 (50.4) and 6.24 -> 6.20 (6.66); TP8, 64 chunks of 16 pages out of 16:
// 209 -> 176 us (181). Against it: 32 and 64 KiB pages of 10 GB and more in pools
// without a power of two of blocks, copies 1-2% slower (8B, 4,096 pages of 1,024
// records 2,544 -> 2,604 us; 2,862).
constexpr int kSharedWgPerCu = 6;
struct CopyShape {
  bool nt;         // stores: nt, else nt sc0 sc1
  bool whole;      // 8 pieces per wave
  uint32_t chunk;  // workgroups dealt in chunks
};
CopyShape copy_shape(const UnitArgs& a, bool shared) {
  const int64_t moved = 4 * a.page_bytes * a.n_units;
  const bool large = moved > (200 << 20);
  CopyShape c{!large, moved > (20 << 20) && moved <= (32 << 20),
              shared ? kEighths : large ? kChunk : 0};
  if (const int64_t t = tune(DSR_TUNE_COPY_STORES)) c.nt = t == 1;
  if (const int64_t t = tune(DSR_TUNE_COPY_PIECES)) c.whole = t == 8;
  if (a.page_bytes % (8 * kPiece)) c.whole = false;
  return c;
}

template <bool kGather>
int launch_copy(const UnitArgs& a, int n_pages, hipStream_t s, bool shared = false) {
  const CopyShape c = copy_shape(a, shared);
  const int64_t pieces = c.whole ? a.page_bytes / (8 * kPiece) : (a.page_bytes + kPiece - 1) / kPiece;
  const int64_t t = tune(DSR_TUNE_COPY_WG_PER_CU);
  const size_t dyn = occupancy_lds(t ? (int)t : shared ? kSharedWgPerCu : kCopyWgPerCu, 0);
  return launch_flat(a.n_units, pieces, kGather ? a.n_layers : n_pages, c.chunk,
                     [&](const FlatMap& m, unsigned grid) {
#define DSR_COPY(HND, POLICY, U) \
  kv_flat_copy_kernel<kGather, HND, POLICY, U><<<grid, kThreads, dyn, s>>>(a, m)
#define DSR_COPY_U(HND, U)                     \
  if (c.nt) DSR_COPY(HND, kStoreNt, U);        \
  else DSR_COPY(HND, kStoreNtSc, U)
    if (a.hnd_heads && c.whole) DSR_COPY_U(true, 8);
    else if (a.hnd_heads) DSR_COPY_U(true, 1);
    else if (c.whole) DSR_COPY_U(false, 8);
    else DSR_COPY_U(false, 1);
#undef DSR_COPY_U
#undef DSR_COPY
  });
}


// The pair-task kernel: neox rows of more than 64 vectors whose partner distance
// is no power of two, and split-x K pages whose head blocks are none.
template <int DT>
int launch_rerotate_pairs(const RotArgs& ra, int n_pages, int style, hipStream_t s) {
  const size_t dyn =
      occupancy_lds(rot_wg_per_cu<DT>(), (int64_t)sizeof(float2) * kMaxRotHalf);
  return launch_page_ranges(ra.u, n_pages, [&](const UnitArgs& b, unsigned grid) {
    RotArgs rb = ra;
    rb.u = b;
    rb.rope_idx = ra.rope_idx + (b.page_ids - ra.u.page_ids);
    if (style == DSR_ROPE_NEOX)
      kv_scatter_rerotate_kernel<DT, DSR_ROPE_NEOX><<<grid, kThreads, dyn, s>>>(rb);
    else
      kv_scatter_rerotate_kernel<DT, DSR_ROPE_GPTJ><<<grid, kThreads, dyn, s>>>(rb);
  });
}

// Workgroups per CU of the flat re-rotation: 6. A wave lives longer than a
// copying one (its table, its rotation), so 4 keep too little in flight and 8
// widen the written window: Llama-3-8B pages e4m3 5.73 / 5.87 / 5.74 TB/s at 4 / 6
// / 8, Gemma-2-9B bf16 5.96 / 6.46 / 6.45, 70B TP8 bf16 5.99 / 6.13 / 5.84, 8B bf16 of
// 2,900 pages 6.46 / 6.46 / 6.19.
constexpr int kRotFlatWgPerCu = 6;

template <int DT, int LAYOUT>
int launch_flat_rerotate(const RotArgs& ra, int n_pages, int style, int piece_vecs, bool shared,
                         hipStream_t s) {
  const CopyShape c = copy_shape(ra.u, shared);
  const int64_t nvec = ra.u.page_bytes >> 4;
  const FastDiv row = fast_div((uint32_t)ra.row_vecs);
  int wg = kRotFlatWgPerCu;
  if (const int64_t t = tune(DSR_TUNE_ROT_WG_PER_CU)) wg = (int)t;
  const int col = (is_fp8<DT>() ? 16 : 8) / (style == DSR_ROPE_NEOX ? 1 : 2);  // pairs
  const size_t tabs = sizeof(float2) * (ra.rot_half + ra.rot_half / col * 2) * (kThreads / kWave);
  const size_t lds = occupancy_lds(wg, 0);
  const size_t dyn = lds > tabs ? lds : tabs;
  return launch_flat(ra.u.n_units, (nvec + piece_vecs - 1) / piece_vecs, n_pages, c.chunk,
                     [&](const FlatMap& m, unsigned grid) {
#define DSR_ROT(STYLE, POLICY)                                                          \
  kv_flat_rerotate_kernel<DT, STYLE, LAYOUT, POLICY><<<grid, kThreads, dyn, s>>>(ra, m, row, \
                                                                                 piece_vecs)
    if (style == DSR_ROPE_NEOX) {
      if (c.nt) DSR_ROT(DSR_ROPE_NEOX, kStoreNt);
      else DSR_ROT(DSR_ROPE_NEOX, kStoreNtSc);
    } else {
      if (c.nt) DSR_ROT(DSR_ROPE_GPTJ, kStoreNt);
      else DSR_ROT(DSR_ROPE_GPTJ, kStoreNtSc);
    }
#undef DSR_ROT
  });
}

template <int DT>
int launch_rerotate(const RotArgs& ra, int n_pages, int style, bool vec_ok, bool shared,
                    hipStream_t s, int layout) {
  const int h = ra.half_vecs;
  if (!vec_ok) {  // rotary width not in whole vectors: the LDS kernel
    return launch_page_ranges(ra.u, n_pages, [&](const UnitArgs& b, unsigned grid) {
      RotArgs rb = ra;
      rb.u = b;
      rb.rope_idx = ra.rope_idx + (b.page_ids - ra.u.page_ids);
      if (style == DSR_ROPE_NEOX)
        kv_scatter_rerotate_lds_kernel<DT, DSR_ROPE_NEOX><<<grid, kThreads, 0, s>>>(rb);
      else
        kv_scatter_rerotate_lds_kernel<DT, DSR_ROPE_GPTJ><<<grid, kThreads, 0, s>>>(rb);
    });
  }
  // split-x K: the caller checked the kx_phys conditions, which make every
  // neox partner lane ^ 32
  if (layout == kRotKx)
    return launch_flat_rerotate<DT, kRotKx>(ra, n_pages, style, kWave, shared, s);
  if (layout == kRotHnd)
    return launch_flat_rerotate<DT, kRotHnd>(ra, n_pages, style, kWave, shared, s);
  const bool contig = style == DSR_ROPE_GPTJ ||
                      (h > 0 && h <= 32 && (h & (h - 1)) == 0 && ra.row_vecs % (2 * h) == 0);
  // other neox rows of <= 64 vectors: pieces of whole rows
  const bool rows = !contig && ra.row_vecs <= kWave && h > 0 && 2 * h <= ra.row_vecs;
  if ((contig || rows) && tune(DSR_TUNE_ROT_KERNEL) != kRotPairs)
    return launch_flat_rerotate<DT, kRotNhd>(
        ra, n_pages, style, contig ? kWave : kWave / ra.row_vecs * ra.row_vecs, shared, s);
  return launch_rerotate_pairs<DT>(ra, n_pages, style, s);
}

}  // namespace

extern "C" {

int dsr_abi_version(void) { return DSR_ABI_VERSION; }

int dsr_set_tuning(int knob, int64_t value) {
  if (knob < 0 || knob >= DSR_TUNE_COUNT_ || value < 0) return DSR_ERR_ARG;
  g_tuning.v[knob].store(value, std::memory_order_relaxed);
  return DSR_OK;
}

const char* dsr_error_string(int code) {
  switch (code) {
    case DSR_OK:
      return "success";
    case DSR_ERR_ARG:
      return "invalid argument (null pointer, negative count or unknown enum)";
    case DSR_ERR_ALIGN:
      return "pointer, stride or size is not a multiple of 16 bytes";
    case DSR_ERR_SHAPE:
      return "inconsistent page/row/rotation geometry";
    case DSR_ERR_IO:
      return "store file read or write failed (see dsr_ring_last_errno)";
    case DSR_ERR_NOFILE:
      return "store file not found";
    case DSR_ERR_TOO_LARGE:
      return "tables exceed the library's static table area (DSR_STATIC_TABLE_BYTES)";
    case DSR_PLAN_ERR_BLOCK:
      return "block id out of range";
    case DSR_PLAN_ERR_RECORD:
      return "slot record outside the staging buffer";
    case DSR_PLAN_ERR_ALIGN:
      return "slot offsets must be multiples of 16 bytes";
    case DSR_PLAN_ERR_ROPE:
      return "rope_idx outside [-1, n_tables)";
    case DSR_PLAN_ERR_OVERLAP:
      return "slot records of two pages overlap";
    case DSR_PLAN_ERR_SLOT:
      return "slot outside the block pool";
    case DSR_PLAN_ERR_ROW:
      return "token row outside the staging buffer";
    case DSR_PLAN_ERR_ROWALIGN:
      return "row offsets must be multiples of 16 bytes";
    default:
      return code > 0 ? hipGetErrorString((hipError_t)code) : "unknown error";
  }
}

int dsr_gather(const uint64_t* layer_base, int n_layers, int64_t kv_stride,
               int64_t page_stride, int64_t page_bytes, int64_t num_blocks,
               const int32_t* page_ids, const int64_t* slot_offsets,
               int n_pages, void* staging, int64_t staging_bytes,
               int64_t layer_bytes, int layer0, dsr_stream_t stream) {
  int rc = check_common(layer_base, n_layers, kv_stride, page_stride, page_bytes,
                        num_blocks, page_ids, slot_offsets, n_pages, staging,
                        staging_bytes, layer_bytes, layer0);
  if (rc != DSR_OK || n_pages == 0 || n_layers == 0) return rc;
  UnitArgs a = make_unit(layer_base, n_layers, kv_stride, page_stride, page_bytes,
                         num_blocks, page_ids, slot_offsets, n_pages, staging,
                         staging_bytes, layer_bytes, layer0);
  return launch_copy<true>(a, n_pages, (hipStream_t)stream);
}

int dsr_scatter_ex(const uint64_t* layer_base, int n_layers, int64_t kv_stride,
                   int64_t page_stride, int64_t page_bytes, int64_t num_blocks,
                   const int32_t* page_ids, const int64_t* slot_offsets,
                   int n_pages, const void* staging, int64_t staging_bytes,
                   int64_t layer_bytes, int layer0, unsigned flags, dsr_stream_t stream) {
  int rc = check_common(layer_base, n_layers, kv_stride, page_stride, page_bytes,
                        num_blocks, page_ids, slot_offsets, n_pages, staging,
                        staging_bytes, layer_bytes, layer0);
  if (rc != DSR_OK || n_pages == 0 || n_layers == 0) return rc;
  UnitArgs a = make_unit(layer_base, n_layers, kv_stride, page_stride, page_bytes,
                         num_blocks, page_ids, slot_offsets, n_pages, staging,
                         staging_bytes, layer_bytes, layer0);
  return launch_copy<false>(a, n_pages, (hipStream_t)stream, flags & DSR_SHARED_RECORDS);
}

int dsr_scatter(const uint64_t* layer_base, int n_layers, int64_t kv_stride,
                int64_t page_stride, int64_t page_bytes, int64_t num_blocks,
                const int32_t* page_ids, const int64_t* slot_offsets,
                int n_pages, const void* staging, int64_t staging_bytes,
                int64_t layer_bytes, int layer0, dsr_stream_t stream) {
  return dsr_scatter_ex(layer_base, n_layers, kv_stride, page_stride, page_bytes, num_blocks,
                        page_ids, slot_offsets, n_pages, staging, staging_bytes, layer_bytes,
                        layer0, 0u, stream);
}

}  // extern "C"

namespace {

// All K layouts: kx_block = 0 for token-major K rows (block_size x H x D),
// kx_block = block_size for the split-x K layout (H x D/X x block_size x X);
// hnd_block = block_size for head-major cache pages (H x block_size x D,
// records token-major).
int scatter_rerotate_any(const uint64_t* layer_base, int n_layers,
                         int64_t kv_stride, int64_t page_stride,
                         int64_t page_bytes, int64_t num_blocks,
                         const int32_t* page_ids, const int64_t* slot_offsets,
                         int n_pages, const void* staging,
                         int64_t staging_bytes, int64_t layer_bytes,
                         int layer0, const float* cos_sin,
                         const int32_t* rope_idx, int n_tables,
                         const int32_t* layer_group, int n_groups, int head_dim,
                         int rot_dim, int rope_style, int dtype,
                         const float* k_scale, int kx_block, int hnd_block, unsigned flags,
                         dsr_stream_t stream) {
  int rc = check_common(layer_base, n_layers, kv_stride, page_stride, page_bytes,
                        num_blocks, page_ids, slot_offsets, n_pages, staging,
                        staging_bytes, layer_bytes, layer0);
  if (rc != DSR_OK) return rc;
  if (rope_style != DSR_ROPE_NEOX && rope_style != DSR_ROPE_GPTJ) return DSR_ERR_ARG;
  int esize, ve;
  switch (dtype) {
    case DSR_DTYPE_BF16:
    case DSR_DTYPE_FP16:
      esize = 2;
      ve = 8;
      break;
    case DSR_DTYPE_FP8_E4M3:
    case DSR_DTYPE_FP8_E5M2:
      esize = 1;
      ve = 16;
      break;
    default:
      return DSR_ERR_ARG;
  }
  if (n_tables < 0 || (layer_group && n_groups < 1)) return DSR_ERR_ARG;
  if (head_dim <= 0 || rot_dim <= 0 || rot_dim > head_dim || (rot_dim & 1) ||
      rot_dim / 2 > kMaxRotHalf)
    return DSR_ERR_SHAPE;
  const int64_t row_bytes = (int64_t)head_dim * esize;
  if (row_bytes % 16 || page_bytes % row_bytes) return DSR_ERR_SHAPE;
  // Whole 16-byte vectors of rotated (and, neox, half-rotated) elements use
  // the vector kernels; other even rotary widths the LDS kernel.
  const bool vec_ok = ((int64_t)(head_dim - rot_dim) * esize) % 16 == 0 &&
                      (rope_style == DSR_ROPE_NEOX ? (rot_dim / 2) % ve == 0 : rot_dim % ve == 0);
  if (!vec_ok && row_bytes / 16 > 2048) return DSR_ERR_SHAPE;  // one row per LDS chunk
  // split-x K: a head's block of block_size tokens is the rotation "row";
  // only whole-vector rotary widths (the pair-task kernel) are supported
  if (kx_block < 0 || (kx_block > 0 && (!vec_ok || page_bytes % (row_bytes * kx_block))))
    return DSR_ERR_SHAPE;
  const int cd = kx_block > 0 ? kx_block : 1;
  const int task_vecs = !vec_ok ? 0 : rope_style == DSR_ROPE_NEOX ? rot_dim / 2 / ve
                                                                   : rot_dim / ve;
  if (n_pages == 0 || n_layers == 0) return DSR_OK;
  if (!rope_idx || (n_tables > 0 && !cos_sin)) return DSR_ERR_ARG;
  if (esize == 1 && !k_scale) return DSR_ERR_ARG;

  RotArgs ra{};
  ra.u = make_unit(layer_base, n_layers, kv_stride, page_stride, page_bytes,
                   num_blocks, page_ids, slot_offsets, n_pages, staging,
                   staging_bytes, layer_bytes, layer0);
  ra.cos_sin = reinterpret_cast<const float2*>(cos_sin);
  ra.rope_idx = rope_idx;
  ra.n_tables = n_tables;
  ra.layer_group = layer_group;
  ra.n_groups = layer_group ? n_groups : 1;
  ra.row_vecs = (int)(row_bytes / 16) * cd;
  ra.rot_half = rot_dim / 2;
  ra.task_vecs = task_vecs * cd;
  ra.tail_vec0 = rot_dim * esize / 16 * cd;
  ra.tasks_per_row = (task_vecs + (head_dim - rot_dim) * esize / 16) * cd;
  ra.col_div = cd;
  ra.rot_vecs = rot_dim * esize / 16;
  ra.half_vecs = rope_style == DSR_ROPE_NEOX && vec_ok ? rot_dim / 2 * esize / 16 : 0;
  ra.k_scale = k_scale;
  const bool shared = flags & DSR_REROTATE_SHARED_RECORDS;
  hipStream_t s = (hipStream_t)stream;
  if (hnd_block > 0) {
    // head-major pages: rows and partners stay whole in record order, the cache
    // side goes through hnd_vec
    const int h = ra.half_vecs;
    const bool contig = vec_ok && (rope_style == DSR_ROPE_GPTJ ||
                                   (h > 0 && h <= 32 && (h & (h - 1)) == 0 &&
                                    ra.row_vecs % (2 * h) == 0));
    const int64_t rows = page_bytes / row_bytes;
    if (!contig || kx_block > 0 || rows % hnd_block) return DSR_ERR_SHAPE;
    ra.u.hnd_heads = (int)(rows / hnd_block);
    ra.u.hnd_block = hnd_block;
    ra.u.hnd_row_vecs = ra.row_vecs;
    switch (dtype) {
      case DSR_DTYPE_BF16:
        return launch_rerotate<DSR_DTYPE_BF16>(ra, n_pages, rope_style, true, shared, s, kRotHnd);
      case DSR_DTYPE_FP16:
        return launch_rerotate<DSR_DTYPE_FP16>(ra, n_pages, rope_style, true, shared, s, kRotHnd);
      case DSR_DTYPE_FP8_E4M3:
        return launch_rerotate<DSR_DTYPE_FP8_E4M3>(ra, n_pages, rope_style, true, shared, s, kRotHnd);
      default:
        return launch_rerotate<DSR_DTYPE_FP8_E5M2>(ra, n_pages, rope_style, true, shared, s, kRotHnd);
    }
  }
  if (kx_block > 0) {
    // vector kernels when the head block is a power-of-two number of
    // vectors (>= one wave), block_size a power of two and the neox partner
    // distance a multiple of 32 vectors (kx_phys); the pair-task kernel else
    const int64_t hv = row_bytes / 16 * kx_block;  // vectors per head block
    const int dist = rope_style == DSR_ROPE_NEOX ? task_vecs * kx_block : 0;
    const bool pow2 = (hv & (hv - 1)) == 0 && (kx_block & (kx_block - 1)) == 0;
    if (pow2 && hv >= kWave && dist % 32 == 0 && page_bytes % 1024 == 0 &&
        tune(DSR_TUNE_ROT_KERNEL) != kRotPairs) {
      ra.kx_row_shift = __builtin_ctzll((unsigned long long)hv);
      ra.kx_bs_shift = __builtin_ctz((unsigned)kx_block);
      ra.kx_dist = dist;
      ra.row_vecs = (int)hv;
      switch (dtype) {
        case DSR_DTYPE_BF16:
          return launch_rerotate<DSR_DTYPE_BF16>(ra, n_pages, rope_style, true, shared, s, kRotKx);
        case DSR_DTYPE_FP16:
          return launch_rerotate<DSR_DTYPE_FP16>(ra, n_pages, rope_style, true, shared, s, kRotKx);
        case DSR_DTYPE_FP8_E4M3:
          return launch_rerotate<DSR_DTYPE_FP8_E4M3>(ra, n_pages, rope_style, true, shared, s, kRotKx);
        default:
          return launch_rerotate<DSR_DTYPE_FP8_E5M2>(ra, n_pages, rope_style, true, shared, s, kRotKx);
      }
    }
    switch (dtype) {
      case DSR_DTYPE_BF16:
        return launch_rerotate_pairs<DSR_DTYPE_BF16>(ra, n_pages, rope_style, s);
      case DSR_DTYPE_FP16:
        return launch_rerotate_pairs<DSR_DTYPE_FP16>(ra, n_pages, rope_style, s);
      case DSR_DTYPE_FP8_E4M3:
        return launch_rerotate_pairs<DSR_DTYPE_FP8_E4M3>(ra, n_pages, rope_style, s);
      default:
        return launch_rerotate_pairs<DSR_DTYPE_FP8_E5M2>(ra, n_pages, rope_style, s);
    }
  }
  switch (dtype) {
    case DSR_DTYPE_BF16:
      return launch_rerotate<DSR_DTYPE_BF16>(ra, n_pages, rope_style, vec_ok, shared, s, kRotNhd);
    case DSR_DTYPE_FP16:
      return launch_rerotate<DSR_DTYPE_FP16>(ra, n_pages, rope_style, vec_ok, shared, s, kRotNhd);
    case DSR_DTYPE_FP8_E4M3:
      return launch_rerotate<DSR_DTYPE_FP8_E4M3>(ra, n_pages, rope_style, vec_ok, shared, s, kRotNhd);
    default:
      return launch_rerotate<DSR_DTYPE_FP8_E5M2>(ra, n_pages, rope_style, vec_ok, shared, s, kRotNhd);
  }
}

}  // namespace

extern "C" {

int dsr_scatter_rerotate(const uint64_t* layer_base, int n_layers,
                         int64_t kv_stride, int64_t page_stride,
                         int64_t page_bytes, int64_t num_blocks,
                         const int32_t* page_ids, const int64_t* slot_offsets,
                         int n_pages, const void* staging,
                         int64_t staging_bytes, int64_t layer_bytes,
                         int layer0, const float* cos_sin,
                         const int32_t* rope_idx, int n_tables,
                         const int32_t* layer_group, int n_groups, int head_dim,
                         int rot_dim, int rope_style, int dtype,
                         const float* k_scale, unsigned flags, dsr_stream_t stream) {
  return scatter_rerotate_any(layer_base, n_layers, kv_stride, page_stride, page_bytes,
                              num_blocks, page_ids, slot_offsets, n_pages, staging,
                              staging_bytes, layer_bytes, layer0, cos_sin, rope_idx, n_tables,
                              layer_group, n_groups, head_dim, rot_dim, rope_style, dtype,
                              k_scale, 0, 0, flags, stream);
}

int dsr_scatter_rerotate_kx(const uint64_t* layer_base, int n_layers,
                            int64_t kv_stride, int64_t page_stride,
                            int64_t page_bytes, int64_t num_blocks,
                            const int32_t* page_ids, const int64_t* slot_offsets,
                            int n_pages, const void* staging,
                            int64_t staging_bytes, int64_t layer_bytes,
                            int layer0, const float* cos_sin,
                            const int32_t* rope_idx, int n_tables,
                            const int32_t* layer_group, int n_groups, int head_dim,
                            int rot_dim, int rope_style, int dtype,
                            const float* k_scale, int block_size, unsigned flags,
                            dsr_stream_t stream) {
  if (block_size <= 0) return DSR_ERR_ARG;
  return scatter_rerotate_any(layer_base, n_layers, kv_stride, page_stride, page_bytes,
                              num_blocks, page_ids, slot_offsets, n_pages, staging,
                              staging_bytes, layer_bytes, layer0, cos_sin, rope_idx, n_tables,
                              layer_group, n_groups, head_dim, rot_dim, rope_style, dtype,
                              k_scale, block_size, 0, flags, stream);
}

int dsr_scatter_rerotate_hnd(const uint64_t* layer_base, int n_layers,
                             int64_t kv_stride, int64_t page_stride,
                             int64_t page_bytes, int64_t num_blocks,
                             const int32_t* page_ids, const int64_t* slot_offsets,
                             int n_pages, const void* staging,
                             int64_t staging_bytes, int64_t layer_bytes,
                             int layer0, const float* cos_sin,
                             const int32_t* rope_idx, int n_tables,
                             const int32_t* layer_group, int n_groups, int head_dim,
                             int rot_dim, int rope_style, int dtype,
                             const float* k_scale, int block_size, unsigned flags,
                             dsr_stream_t stream) {
  if (block_size <= 0) return DSR_ERR_ARG;
  return scatter_rerotate_any(layer_base, n_layers, kv_stride, page_stride, page_bytes,
                              num_blocks, page_ids, slot_offsets, n_pages, staging,
                              staging_bytes, layer_bytes, layer0, cos_sin, rope_idx, n_tables,
                              layer_group, n_groups, head_dim, rot_dim, rope_style, dtype,
                              k_scale, 0, block_size, flags, stream);
}

}  // extern "C"

namespace {

// Head-major copies: the unit geometry, then the flat copies.
int copy_hnd(bool gather, const uint64_t* layer_base, int n_layers, int64_t kv_stride,
             int64_t page_stride, int64_t page_bytes, int64_t num_blocks,
             const int32_t* page_ids, const int64_t* slot_offsets, int n_pages,
             const void* staging, int64_t staging_bytes, int64_t layer_bytes, int layer0,
             int block_size, int num_heads, dsr_stream_t stream) {
  if (block_size <= 0 || num_heads <= 0) return DSR_ERR_ARG;
  int rc = check_common(layer_base, n_layers, kv_stride, page_stride, page_bytes,
                        num_blocks, page_ids, slot_offsets, n_pages, staging,
                        staging_bytes, layer_bytes, layer0);
  if (rc != DSR_OK) return rc;
  const int64_t rows = (int64_t)block_size * num_heads;
  if (page_bytes % (rows * 16)) return DSR_ERR_SHAPE;
  if (n_pages == 0 || n_layers == 0) return DSR_OK;
  UnitArgs a = make_unit(layer_base, n_layers, kv_stride, page_stride, page_bytes,
                         num_blocks, page_ids, slot_offsets, n_pages, staging,
                         staging_bytes, layer_bytes, layer0);
  a.hnd_heads = num_heads;
  a.hnd_block = block_size;
  a.hnd_row_vecs = (int)(page_bytes / rows / 16);
  return gather ? launch_copy<true>(a, n_pages, (hipStream_t)stream)
                : launch_copy<false>(a, n_pages, (hipStream_t)stream);
}

}  // namespace

extern "C" {

int dsr_gather_hnd(const uint64_t* layer_base, int n_layers, int64_t kv_stride,
                   int64_t page_stride, int64_t page_bytes, int64_t num_blocks,
                   const int32_t* page_ids, const int64_t* slot_offsets, int n_pages,
                   void* staging, int64_t staging_bytes, int64_t layer_bytes, int layer0,
                   int block_size, int num_heads, dsr_stream_t stream) {
  return copy_hnd(true, layer_base, n_layers, kv_stride, page_stride, page_bytes, num_blocks,
                  page_ids, slot_offsets, n_pages, staging, staging_bytes, layer_bytes, layer0,
                  block_size, num_heads, stream);
}

int dsr_scatter_hnd(const uint64_t* layer_base, int n_layers, int64_t kv_stride,
                    int64_t page_stride, int64_t page_bytes, int64_t num_blocks,
                    const int32_t* page_ids, const int64_t* slot_offsets, int n_pages,
                    const void* staging, int64_t staging_bytes, int64_t layer_bytes,
                    int layer0, int block_size, int num_heads, dsr_stream_t stream) {
  return copy_hnd(false, layer_base, n_layers, kv_stride, page_stride, page_bytes,
                  num_blocks, page_ids, slot_offsets, n_pages, staging, staging_bytes,
                  layer_bytes, layer0, block_size, num_heads, stream);
}

}  // extern "C"

namespace {

// The token form's pieces: rows of 64 vectors and more are cut by themselves,
// `wide_tokens` tokens to a unit; of shorter rows a unit holds at least 256 vectors, one
// workgroup's.
struct SlotShape {
  bool wide;
  int64_t pieces;  // per unit
  int64_t units;   // per layer
};
SlotShape slot_shape(SlotArgs* a, int wide_tokens = 16) {
  const int64_t vpr = a->row_bytes >> 4;
  SlotShape h{vpr >= kWave, 0, 0};
  a->unit_tokens = (int32_t)(h.wide ? wide_tokens : vpr >= 16 ? 16 : 16 * ((16 + vpr - 1) / vpr));
  const int64_t per_row = h.wide ? (vpr + kWave - 1) / kWave : vpr;
  a->row = fast_div((uint32_t)per_row);
  h.pieces = h.wide ? a->unit_tokens * per_row : (a->unit_tokens * vpr + kWave - 1) / kWave;
  h.units = ((int64_t)a->n_tokens + a->unit_tokens - 1) / a->unit_tokens;
  return h;
}

// Stores and order of a token-form launch, by the bytes it moves, as for the
// page copies (copy_shape).
int64_t slots_moved(const SlotArgs& a) { return 4 * a.row_bytes * a.n_tokens * a.n_layers; }
bool slots_large(const SlotArgs& a) { return slots_moved(a) > (200 << 20); }

// Workgroups per CU: 6, wide rows' scatters 4 (8B bf16 rows 5.92 TB/s at 4, 5.78 at
// 6; one-head e4m3 rows 5.78 at 4, 5.88 at 6, gathers 5.75 and 5.89).
int slots_wg_per_cu(bool gather, bool wide) {
  const int64_t t = tune(DSR_TUNE_SLOTS_WG_PER_CU);
  return t ? (int)t : wide && !gather ? 4 : 6;
}

// Gathers of rows up to 4 KiB that move more than 16 GiB: sc0 sc1 stores, workgroups
// dealt one by one, and of rows up to 2 KiB the layers of 2 tokens at a time, not of 16.
// The kernel of 16 tokens per workgroup that this one replaced / this with units of 16 /
// of 2: 2 KiB rows of 32 layers 70,000 tokens 2,866 / 2,905 / 2,873 us, 283,000 11,259 / 11,522 /
// 11,282, of 80 layers 70,000 7,157 / 7,240 / 7,114; 1.5 KiB rows 171,000 5,333 / 5,475 / 5,348; 1
// KiB rows 283,000 7,150 / 6,069 / 5,803; 4 KiB rows of 42 layers 108,000 11,842 / 11,404 /
// 11,523. Without it (chunks, nt sc0 sc1): 2 KiB rows 283,000 tokens 11,533 -> 11,682, of 80
// layers 70,000 7,481 -> 7,433 against 7,218 with it. Smaller gathers: within 1% either way, 1
// KiB rows of 11,000 tokens 294 / 236 / 241; rows of 6 KiB 13,387 / 11,694 / 12,568. (One piece
// per wave throughout: 2, 4 and 8 were 1-10% behind.)
constexpr int64_t kSlotsHugeBytes = 16ll << 30;
constexpr int64_t kSlotsHugeRow = 4 << 10;
constexpr int64_t kSlotsPairRow = 2 << 10;

int slots_launch(bool gather, const uint64_t* layer_base, int n_layers, int64_t kv_stride,
                 int64_t page_stride, int64_t page_bytes, int64_t num_blocks, int block_size,
                 int64_t row_bytes, const int64_t* slot_mapping, const int64_t* row_offsets,
                 int n_tokens, const void* staging, int64_t staging_bytes,
                 int64_t layer_bytes, int layer0, dsr_stream_t stream) {
  if (n_tokens < 0 || n_layers < 0 || layer0 < 0 || num_blocks < 0 || staging_bytes < 0 ||
      block_size <= 0 || row_bytes <= 0 || page_bytes <= 0)
    return DSR_ERR_ARG;
  if (n_tokens == 0 || n_layers == 0) return DSR_OK;
  if (!layer_base || !slot_mapping || !row_offsets || !staging) return DSR_ERR_ARG;
  if (page_bytes < (int64_t)block_size * row_bytes || layer_bytes < 2 * page_bytes ||
      row_bytes > 0x7fffffffLL)
    return DSR_ERR_SHAPE;
  if (!aligned16(kv_stride) || !aligned16(page_stride) || !aligned16(page_bytes) ||
      !aligned16(row_bytes) || !aligned16(layer_bytes) || !aligned16p(staging))
    return DSR_ERR_ALIGN;
  SlotArgs a{};
  a.layer_base = layer_base;
  a.kv_stride = kv_stride;
  a.page_stride = page_stride;
  a.page_bytes = page_bytes;
  a.num_blocks = num_blocks;
  a.row_bytes = row_bytes;
  a.slot_mapping = slot_mapping;
  a.row_offsets = row_offsets;
  a.staging = const_cast<uint8_t*>(static_cast<const uint8_t*>(staging));
  a.staging_bytes = staging_bytes;
  a.layer_bytes = layer_bytes;
  a.n_tokens = n_tokens;
  a.n_layers = n_layers;
  a.layer0 = layer0;
  a.block_size = block_size;
  a.block_shift = (block_size & (block_size - 1)) == 0 ? __builtin_ctz((unsigned)block_size) : -1;
  const int64_t vpr = row_bytes >> 4;
  a.least_row = vpr <= 8 && (vpr & (vpr - 1)) == 0 && a.block_shift >= 0 ? 0 : INT64_MIN;
  const bool large = slots_large(a);
  const bool huge = gather && vpr >= kWave && row_bytes <= kSlotsHugeRow &&
                    slots_moved(a) > kSlotsHugeBytes;
  const bool pairs = huge && row_bytes <= kSlotsPairRow &&
                     ((int64_t)n_tokens + 1) / 2 * n_layers <= 0x7fffffffLL;
  const SlotShape h = slot_shape(&a, pairs ? 2 : 16);
  if (h.units * n_layers > 0x7fffffffLL) return DSR_ERR_ARG;
  const hipStream_t s = (hipStream_t)stream;
  const size_t dyn = occupancy_lds(slots_wg_per_cu(gather, h.wide), 0);
  return launch_flat(h.units * n_layers, h.pieces, gather ? n_layers : h.units,
                     large && !huge ? kChunk : 0,
                     [&](const FlatMap& m, unsigned grid) {
#define DSR_SLOTS(WIDE, POLICY)                                                              \
  (gather ? kv_slots_flat_kernel<true, WIDE, POLICY><<<grid, kThreads, dyn, s>>>(a, m)       \
          : kv_slots_flat_kernel<false, WIDE, POLICY><<<grid, kThreads, dyn, s>>>(a, m))
    if (!h.wide) DSR_SLOTS(false, kStoreNt);
    else if (huge) kv_slots_flat_kernel<true, true, kStorePolicy><<<grid, kThreads, dyn, s>>>(a, m);
    else if (large) DSR_SLOTS(true, kStoreNtSc);
    else DSR_SLOTS(true, kStoreNt);
#undef DSR_SLOTS
  });
}

// Token-form scatter with re-rotation: argument checks, then the flat kernel.
int slots_rerotate_launch(const uint64_t* layer_base, int n_layers, int64_t kv_stride,
                          int64_t page_stride, int64_t page_bytes, int64_t num_blocks,
                          int block_size, int64_t row_bytes, const int64_t* slot_mapping,
                          const int64_t* row_offsets, int n_tokens, const void* staging,
                          int64_t staging_bytes, int64_t layer_bytes, int layer0,
                          const float* cos_sin, const int32_t* rope_idx, int n_tables,
                          const int32_t* layer_group, int n_groups, int head_dim, int rot_dim,
                          int rope_style, int dtype, const float* k_scale, dsr_stream_t stream) {
  if (n_tokens < 0 || n_layers < 0 || layer0 < 0 || num_blocks < 0 || staging_bytes < 0 ||
      block_size <= 0 || row_bytes <= 0 || page_bytes <= 0 || n_tables < 0 ||
      (layer_group && n_groups < 1))
    return DSR_ERR_ARG;
  if (rope_style != DSR_ROPE_NEOX && rope_style != DSR_ROPE_GPTJ) return DSR_ERR_ARG;
  const int esize = dtype == DSR_DTYPE_BF16 || dtype == DSR_DTYPE_FP16 ? 2
                    : dtype == DSR_DTYPE_FP8_E4M3 || dtype == DSR_DTYPE_FP8_E5M2 ? 1 : 0;
  if (!esize) return DSR_ERR_ARG;
  if (n_tokens == 0 || n_layers == 0) return DSR_OK;
  if (!layer_base || !slot_mapping || !row_offsets || !staging || !rope_idx ||
      (n_tables > 0 && !cos_sin) || (esize == 1 && !k_scale))
    return DSR_ERR_ARG;
  // heads of a power-of-two number of vectors <= 64, rotary width in whole
  // vectors (both halves for neox), at most 256 rotated dims
  const int64_t head_bytes = (int64_t)head_dim * esize;
  const int ve = 16 / esize;
  const int hv = (int)(head_bytes / 16);
  if (head_dim <= 0 || rot_dim <= 0 || rot_dim > head_dim || rot_dim % 2 ||
      head_bytes % 16 || row_bytes % head_bytes || hv > kWave || (hv & (hv - 1)) ||
      rot_dim / 2 > kSlotRotMaxHalf ||
      (rope_style == DSR_ROPE_NEOX ? (rot_dim / 2) % ve : rot_dim % ve))
    return DSR_ERR_SHAPE;
  if (page_bytes < (int64_t)block_size * row_bytes || layer_bytes < 2 * page_bytes ||
      row_bytes > 0x7fffffffLL)
    return DSR_ERR_SHAPE;
  if (!aligned16(kv_stride) || !aligned16(page_stride) || !aligned16(page_bytes) ||
      !aligned16(row_bytes) || !aligned16(layer_bytes) || !aligned16p(staging))
    return DSR_ERR_ALIGN;
  SlotArgs a{};
  a.layer_base = layer_base;
  a.kv_stride = kv_stride;
  a.page_stride = page_stride;
  a.page_bytes = page_bytes;
  a.num_blocks = num_blocks;
  a.row_bytes = row_bytes;
  a.slot_mapping = slot_mapping;
  a.row_offsets = row_offsets;
  a.staging = const_cast<uint8_t*>(static_cast<const uint8_t*>(staging));
  a.staging_bytes = staging_bytes;
  a.layer_bytes = layer_bytes;
  a.n_tokens = n_tokens;
  a.n_layers = n_layers;
  a.layer0 = layer0;
  a.block_size = block_size;
  a.block_shift = (block_size & (block_size - 1)) == 0 ? __builtin_ctz((unsigned)block_size) : -1;
  a.least_row = INT64_MIN;
  RotArgs ra{};
  ra.u.layer0 = layer0;
  ra.cos_sin = reinterpret_cast<const float2*>(cos_sin);
  ra.rope_idx = rope_idx;
  ra.n_tables = n_tables;
  ra.layer_group = layer_group;
  ra.n_groups = layer_group ? n_groups : 1;
  ra.row_vecs = hv;
  ra.rot_half = rot_dim / 2;
  ra.rot_vecs = rot_dim * esize / 16;
  ra.half_vecs = rope_style == DSR_ROPE_NEOX ? rot_dim / 2 * esize / 16 : 0;
  ra.k_scale = k_scale;
  const SlotShape h = slot_shape(&a);
  if (h.units * n_layers > 0x7fffffffLL) return DSR_ERR_ARG;
  const bool large = slots_large(a);
  const hipStream_t s = (hipStream_t)stream;
  const int64_t t = tune(DSR_TUNE_SLOTS_WG_PER_CU);
  const int col = (esize == 1 ? 16 : 8) / (rope_style == DSR_ROPE_NEOX ? 1 : 2);  // pairs
  const size_t tabs = sizeof(float2) * (ra.rot_half + ra.rot_half / col * 2) * (kThreads / kWave);
  const size_t lds = occupancy_lds(t ? (int)t : kRotFlatWgPerCu, 0);
  const size_t dyn = lds > tabs ? lds : tabs;
  return launch_flat(h.units * n_layers, h.pieces, h.units, large ? kChunk : 0,
                     [&](const FlatMap& m, unsigned grid) {
    const bool neox = rope_style == DSR_ROPE_NEOX;
#define DSR_SLOT_ROT_P(DT, WIDE, POLICY)                                                     \
  (neox ? kv_slots_flat_rerotate_kernel<DT, DSR_ROPE_NEOX, WIDE, POLICY>                     \
          <<<grid, kThreads, dyn, s>>>(a, ra, m)                                             \
        : kv_slots_flat_rerotate_kernel<DT, DSR_ROPE_GPTJ, WIDE, POLICY>                     \
          <<<grid, kThreads, dyn, s>>>(a, ra, m))
#define DSR_SLOT_ROT(DT)                                     \
  (!h.wide ? DSR_SLOT_ROT_P(DT, false, kStoreNt)             \
   : large ? DSR_SLOT_ROT_P(DT, true, kStoreNtSc)            \
           : DSR_SLOT_ROT_P(DT, true, kStoreNt))
    switch (dtype) {
      case DSR_DTYPE_BF16: DSR_SLOT_ROT(DSR_DTYPE_BF16); break;
      case DSR_DTYPE_FP16: DSR_SLOT_ROT(DSR_DTYPE_FP16); break;
      case DSR_DTYPE_FP8_E4M3: DSR_SLOT_ROT(DSR_DTYPE_FP8_E4M3); break;
      default: DSR_SLOT_ROT(DSR_DTYPE_FP8_E5M2); break;
    }
#undef DSR_SLOT_ROT
#undef DSR_SLOT_ROT_P
  });
}

}  // namespace

extern "C" {

int dsr_gather_slots(const uint64_t* layer_base, int n_layers, int64_t kv_stride,
                     int64_t page_stride, int64_t page_bytes, int64_t num_blocks,
                     int block_size, int64_t row_bytes, const int64_t* slot_mapping,
                     const int64_t* row_offsets, int n_tokens, void* staging,
                     int64_t staging_bytes, int64_t layer_bytes, int layer0,
                     dsr_stream_t stream) {
  return slots_launch(true, layer_base, n_layers, kv_stride, page_stride, page_bytes,
                      num_blocks, block_size, row_bytes, slot_mapping, row_offsets, n_tokens,
                      staging, staging_bytes, layer_bytes, layer0, stream);
}

int dsr_scatter_slots(const uint64_t* layer_base, int n_layers, int64_t kv_stride,
                      int64_t page_stride, int64_t page_bytes, int64_t num_blocks,
                      int block_size, int64_t row_bytes, const int64_t* slot_mapping,
                      const int64_t* row_offsets, int n_tokens, const void* staging,
                      int64_t staging_bytes, int64_t layer_bytes, int layer0,
                      dsr_stream_t stream) {
  return slots_launch(false, layer_base, n_layers, kv_stride, page_stride, page_bytes,
                      num_blocks, block_size, row_bytes, slot_mapping, row_offsets, n_tokens,
                      staging, staging_bytes, layer_bytes, layer0, stream);
}

int dsr_scatter_slots_rerotate(const uint64_t* layer_base, int n_layers, int64_t kv_stride,
                               int64_t page_stride, int64_t page_bytes, int64_t num_blocks,
                               int block_size, int64_t row_bytes, const int64_t* slot_mapping,
                               const int64_t* row_offsets, int n_tokens, const void* staging,
                               int64_t staging_bytes, int64_t layer_bytes, int layer0,
                               const float* cos_sin, const int32_t* rope_idx, int n_tables,
                               const int32_t* layer_group, int n_groups, int head_dim,
                               int rot_dim, int rope_style, int dtype, const float* k_scale,
                               dsr_stream_t stream) {
  return slots_rerotate_launch(layer_base, n_layers, kv_stride, page_stride, page_bytes,
                               num_blocks, block_size, row_bytes, slot_mapping, row_offsets,
                               n_tokens, staging, staging_bytes, layer_bytes, layer0, cos_sin,
                               rope_idx, n_tables, layer_group, n_groups, head_dim, rot_dim,
                               rope_style, dtype, k_scale, stream);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Allocation-free load with re-rotation (dsr_scatter_rerotate_static).
//
// dsr_scatter_rerotate reads its tables (layer addresses, page ids, record
// offsets, table indices, angle tables, layer groups, scales) from device
// memory that the caller allocates per call. This variant takes them in host
// memory and stages them in `scratch`, a fixed device array of the library,
// then runs the same kernels on the staged copies. Each GPU holds its own
// copy of the array; its device address comes from hipGetSymbolAddress on
// the first call on that device (the array's name is a host-side stand-in
// and is never passed to a kernel or a copy).

namespace {

static __device__ __align__(256) uint8_t scratch[DSR_STATIC_TABLE_BYTES];

std::mutex g_scratch_mu;
uint8_t* g_scratch_ptr[kMaxDevices];  // per device, set once

// Device address of `scratch` on the current device (nullptr and *rc set
// on failure).
uint8_t* scratch_on_current_device(int* rc) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    *rc = (int)e;
    return nullptr;
  }
  if (dev < 0 || dev >= kMaxDevices) {
    *rc = DSR_ERR_ARG;
    return nullptr;
  }
  std::lock_guard<std::mutex> g(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      *rc = e != hipSuccess ? (int)e : DSR_ERR_ARG;
      return nullptr;
    }
    g_scratch_ptr[dev] = static_cast<uint8_t*>(p);
  }
  return g_scratch_ptr[dev];
}

int64_t round256(int64_t v) { return (v + 255) & ~(int64_t)255; }

}  // namespace

extern "C" {

int dsr_scatter_rerotate_static(const uint64_t* layer_base, int n_layers,
                                int64_t kv_stride, int64_t page_stride,
                                int64_t page_bytes, int64_t num_blocks,
                                const int32_t* page_ids, const int64_t* slot_offsets,
                                int n_pages, const void* staging,
                                int64_t staging_bytes, int64_t layer_bytes,
                                int layer0, const float* cos_sin,
                                const int32_t* rope_idx, int n_tables,
                                const int32_t* layer_group, int n_groups, int head_dim,
                                int rot_dim, int rope_style, int dtype,
                                const float* k_scale, unsigned flags, dsr_stream_t stream) {
  if (n_pages < 0 || n_layers < 0 || layer0 < 0 || n_tables < 0 ||
      (layer_group && n_groups < 1))
    return DSR_ERR_ARG;
  if (n_pages == 0 || n_layers == 0) return DSR_OK;
  if (!layer_base || !page_ids || !slot_offsets || !rope_idx || (n_tables > 0 && !cos_sin))
    return DSR_ERR_ARG;
  if (rot_dim <= 0 || (rot_dim & 1) || rot_dim / 2 > kMaxRotHalf) return DSR_ERR_SHAPE;
  const int64_t rec_layers = (int64_t)layer0 + n_layers;  // entries of per-layer tables
  const int64_t groups = layer_group ? n_groups : 1;
  // packed sections of the staged tables, each 256-byte aligned
  const int64_t sz_base = (int64_t)n_layers * 8;
  const int64_t sz_ids = (int64_t)n_pages * 4;
  const int64_t sz_off = (int64_t)n_pages * 8;
  const int64_t sz_idx = (int64_t)n_pages * 4;
  const int64_t sz_cs = groups * n_tables * (rot_dim / 2) * 8;
  const int64_t sz_grp = layer_group ? rec_layers * 4 : 0;
  const int64_t sz_scl = k_scale ? rec_layers * 4 : 0;
  const int64_t o_base = 0, o_ids = o_base + round256(sz_base), o_off = o_ids + round256(sz_ids),
                o_idx = o_off + round256(sz_off), o_cs = o_idx + round256(sz_idx),
                o_grp = o_cs + round256(sz_cs), o_scl = o_grp + round256(sz_grp),
                total = o_scl + round256(sz_scl);
  if (total > DSR_STATIC_TABLE_BYTES) return DSR_ERR_TOO_LARGE;

  hipStream_t s = (hipStream_t)stream;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  hipError_t e = hipStreamIsCapturing(s, &cap);
  if (e != hipSuccess) return (int)e;
  if (cap != hipStreamCaptureStatusNone) return DSR_ERR_ARG;  // host-to-device copies

  int rc = DSR_OK;
  uint8_t* base = scratch_on_current_device(&rc);
  if (!base) return rc;
  struct Piece {
    int64_t off, bytes;
    const void* src;
  } pieces[] = {{o_base, sz_base, layer_base}, {o_ids, sz_ids, page_ids},
                {o_off, sz_off, slot_offsets}, {o_idx, sz_idx, rope_idx},
                {o_cs, sz_cs, cos_sin},       {o_grp, sz_grp, layer_group},
                {o_scl, sz_scl, k_scale}};
  for (const Piece& p : pieces) {
    if (p.bytes == 0) continue;
    e = hipMemcpyAsync(base + p.off, p.src, (size_t)p.bytes, hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return (int)e;
  }
  return scatter_rerotate_any(
      reinterpret_cast<const uint64_t*>(base + o_base), n_layers, kv_stride, page_stride,
      page_bytes, num_blocks, reinterpret_cast<const int32_t*>(base + o_ids),
      reinterpret_cast<const int64_t*>(base + o_off), n_pages, staging, staging_bytes,
      layer_bytes, layer0, sz_cs ? reinterpret_cast<const float*>(base + o_cs) : nullptr,
      reinterpret_cast<const int32_t*>(base + o_idx), n_tables,
      layer_group ? reinterpret_cast<const int32_t*>(base + o_grp) : nullptr, n_groups,
      head_dim, rot_dim, rope_style, dtype,
      k_scale ? reinterpret_cast<const float*>(base + o_scl) : nullptr, 0, 0, flags, stream);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Loads of shared records (dsr_scatter_fanout): each piece of a source record
// read once and written to all of that record's destination pages.

namespace {

// Unit order, stores and workgroups per CU of the fan-out, whose destinations lie
// anywhere. All figures in us, in one process in turn: the kernel of one workgroup
// per unit that this one replaced / this choice / the other one.
//   From kFanManySources records up source-major (a record's layers follow each
//   other), else layer-major, workgroups dealt one by one. Layer-major writes one
//   layer's pages at a time, which is ahead by 1-6% while they are few (8B bf16, 1,024
//   pages of 128 records 484 / 446 / 474; 0.5B, 4,096 of 256 165 / 165 / 169) and behind
//   where they are many (8B, 5,120 of 640 2,005 / 1,915 / 2,185; 70B, 32,768 of 2,048
//   27,968 / 28,041 / 32,728; its TP8 share 3,955 / 3,926 / 4,258); from 384 to 2,048
//   records of 8B and TP8 in pools without a power of two of blocks the two are within
//   3%, either way. Chunks of 128 workgroups (the page copies') cost source-major plain
//   loads 1-3%: 70B 28,041 -> 28,805.
//   Stores sc0 sc1 from 1 GiB read and written up: 1-5% ahead of nt sc0 sc1 (8B, 4,096 of
//   256 1,655 against 1,697; 70B TP8 rotated 3,489 against 3,633), which a smaller load
//   takes (1,024 TP8 pages of 256 165 against 169; on buffers in turn that the
//   memory-side cache does not hold, up to 10% ahead at 128 pages).
//   Rotated loads of fewer waves than 4 workgroups per CU hold deal each record's
//   destinations to as many as fill them, at least 4 to a wave: 0.5B, 64 pages of one
//   record 1,212 / 322 / 1,675 (40 sets of buffers), 1,000 of one 3,012 / 324 / 4,314 (7),
//   256 of 4 710 / 301 / 978 (23); pages from 16 KiB also where a record has 64 or more,
//   16 to a wave: 8B, 1,024 of 16 843 / 816 / 892 (2 sets), e4m3 521 / 438 / 490; 4 KiB
//   pages of more waves lose 3-10% by it. Up to twice those waves, 8 per CU in place of
//   4: TP8, 1,024 of 16 279 / 276 / 301 (2), 0.5B, 512 of 64 257 / 243 / 259 (11).
//   4 workgroups per CU, for few destinations 6, on such buffers: 0.5B rotated, 512 of
//   64 1.01 times the old kernel's rate at 4, 0.94 at 6; 8B rotated, 128 of 64 1.33 and
//   1.38, TP8 plain, 64 of 32 1.10 and 1.16.
// DSR_TUNE_FANOUT_WG_PER_CU overrides the workgroups.
constexpr int64_t kFanManySources = 512;
constexpr int64_t kFanLargeBytes = 1 << 30;
constexpr int kFanFewPages = 256;
constexpr int64_t kFanFillWaves = 4096;  // 4 workgroups on each of 256 CUs
constexpr int64_t kFanMaxSplit = 64;

template <int DT, int STYLE, int LAYOUT, bool ROT>
int launch_fanout_s(const FanArgs& fa, hipStream_t s) {
  const RotArgs& ra = fa.ra;
  const int col = (is_fp8<DT>() ? 16 : 8) / (STYLE == DSR_ROPE_NEOX ? 1 : 2);  // pairs
  const size_t tabs =
      ROT ? sizeof(float2) * (ra.rot_half + ra.rot_half / col * 2) * (kThreads / kWave) : 0;
  const bool many = fa.n_src >= kFanManySources;
  const bool large =
      2 * ra.u.page_bytes * ra.u.n_layers * ((int64_t)fa.n_src + fa.n_dst) > kFanLargeBytes;
  const int64_t pieces = (ra.u.page_bytes + kPiece - 1) / kPiece;
  const int64_t waves = (int64_t)fa.n_src * ra.u.n_layers * pieces;
  int wg = fa.n_dst > kFanFewPages ? 4 : 6;
  int64_t split = 1;
  if (ROT) {
    const int64_t dests = fa.n_dst / fa.n_src;
    split = kFanFillWaves / waves;
    if (ra.u.page_bytes >= 16 << 10 && dests >= 64 && split < dests / 16) split = dests / 16;
    if (split > dests / 4) split = dests / 4;
    if (split > kFanMaxSplit) split = kFanMaxSplit;
    if (split < 1) split = 1;
    if (split == 1 && waves > kFanFillWaves && waves <= 2 * kFanFillWaves) wg = 8;
  }
  if (const int64_t t = tune(DSR_TUNE_FANOUT_WG_PER_CU)) wg = (int)t;
  const size_t lds = occupancy_lds(wg, 0);
  const size_t dyn = lds > tabs ? lds : tabs;
  const FastDiv row = fast_div((uint32_t)(ROT ? ra.row_vecs : 1));
  const FastDiv share = fast_div((uint32_t)pieces);
  return launch_flat((int64_t)fa.n_src * ra.u.n_layers, pieces * split,
                     many ? ra.u.n_layers : fa.n_src, 0,
                     [&](const FlatMap& m, unsigned grid) {
    if (large)
      kv_fanout_kernel<DT, STYLE, LAYOUT, ROT, kStorePolicy>
          <<<grid, kThreads, dyn, s>>>(fa, m, row, share, (int)split, !many);
    else
      kv_fanout_kernel<DT, STYLE, LAYOUT, ROT, kStoreNtSc>
          <<<grid, kThreads, dyn, s>>>(fa, m, row, share, (int)split, !many);
  });
}

template <int DT, int LAYOUT>
int launch_fanout_l(const FanArgs& fa, int style, hipStream_t s) {
  if (!fa.dst_rope) return launch_fanout_s<DSR_DTYPE_BF16, DSR_ROPE_NEOX, LAYOUT, false>(fa, s);
  return style == DSR_ROPE_GPTJ ? launch_fanout_s<DT, DSR_ROPE_GPTJ, LAYOUT, true>(fa, s)
                                : launch_fanout_s<DT, DSR_ROPE_NEOX, LAYOUT, true>(fa, s);
}

template <int DT>
int launch_fanout(const FanArgs& fa, int style, int layout, hipStream_t s) {
  switch (layout) {
    case kRotKx: return launch_fanout_l<DT, kRotKx>(fa, style, s);
    case kRotHnd: return launch_fanout_l<DT, kRotHnd>(fa, style, s);
    default: return launch_fanout_l<DT, kRotNhd>(fa, style, s);
  }
}

}  // namespace

extern "C" {

int dsr_scatter_fanout(const uint64_t* layer_base, int n_layers, int64_t kv_stride,
                       int64_t page_stride, int64_t page_bytes, int64_t num_blocks,
                       const int64_t* src_offsets, int n_src, const int32_t* dst_start,
                       const int32_t* dst_page_ids, const int32_t* dst_rope_idx, int n_dst,
                       const void* staging, int64_t staging_bytes, int64_t layer_bytes,
                       int layer0, const float* cos_sin, int n_tables,
                       const int32_t* layer_group, int n_groups, int head_dim, int rot_dim,
                       int rope_style, int dtype, const float* k_scale, int k_layout,
                       int block_size, int num_heads, dsr_stream_t stream) {
  if (n_src < 0 || n_dst < 0) return DSR_ERR_ARG;
  if (k_layout != DSR_K_NHD && k_layout != DSR_K_KX && k_layout != DSR_K_HND) return DSR_ERR_ARG;
  if (k_layout != DSR_K_NHD && block_size <= 0) return DSR_ERR_ARG;
  // the page-table checks of the copies, with the destination ids and the
  // source offsets in the tables' places
  int rc = check_common(layer_base, n_layers, kv_stride, page_stride, page_bytes, num_blocks,
                        dst_page_ids, src_offsets, n_dst, staging, staging_bytes, layer_bytes,
                        layer0);
  if (rc != DSR_OK) return rc;
  // the geometry is checked before the empty-work return below, so that a
  // call with n_dst = 0 tells whether the fan-out takes a geometry
  // pages of at most 32 KiB (larger ones are refused, unmeasured)
  if (page_bytes > (32 << 10)) return DSR_ERR_SHAPE;
  RotArgs ra{};
  ra.u = make_unit(layer_base, n_layers, kv_stride, page_stride, page_bytes, num_blocks,
                   nullptr, nullptr, 0, staging, staging_bytes, layer_bytes, layer0);
  ra.n_groups = 1;
  ra.rot_half = 1;
  int dt = DSR_DTYPE_BF16, style = DSR_ROPE_NEOX;
  if (dst_rope_idx) {
    if (rope_style != DSR_ROPE_NEOX && rope_style != DSR_ROPE_GPTJ) return DSR_ERR_ARG;
    int esize, ve;
    switch (dtype) {
      case DSR_DTYPE_BF16:
      case DSR_DTYPE_FP16:
        esize = 2;
        ve = 8;
        break;
      case DSR_DTYPE_FP8_E4M3:
      case DSR_DTYPE_FP8_E5M2:
        esize = 1;
        ve = 16;
        break;
      default:
        return DSR_ERR_ARG;
    }
    if (n_tables < 0 || (layer_group && n_groups < 1)) return DSR_ERR_ARG;
    if (n_tables > 0 && !cos_sin) return DSR_ERR_ARG;
    if (esize == 1 && !k_scale) return DSR_ERR_ARG;
    if (head_dim <= 0 || rot_dim <= 0 || rot_dim > head_dim || (rot_dim & 1) ||
        rot_dim / 2 > kMaxRotHalf)
      return DSR_ERR_SHAPE;
    const int64_t row_bytes = (int64_t)head_dim * esize;
    if (row_bytes % 16 || page_bytes % row_bytes) return DSR_ERR_SHAPE;
    // the vector map's geometry: whole-vector rotary widths, neox
    // partners a power of two <= 32 vectors apart inside a row
    const bool vec_ok = ((int64_t)(head_dim - rot_dim) * esize) % 16 == 0 &&
                        (rope_style == DSR_ROPE_NEOX ? (rot_dim / 2) % ve == 0 : rot_dim % ve == 0);
    const int row_vecs = (int)(row_bytes / 16);
    const int h = rope_style == DSR_ROPE_NEOX && vec_ok ? rot_dim / 2 * esize / 16 : 0;
    const bool contig = vec_ok && (rope_style == DSR_ROPE_GPTJ ||
                                   (h > 0 && h <= 32 && (h & (h - 1)) == 0 &&
                                    row_vecs % (2 * h) == 0));
    if (!contig) return DSR_ERR_SHAPE;
    ra.cos_sin = reinterpret_cast<const float2*>(cos_sin);
    ra.n_tables = n_tables;
    ra.layer_group = layer_group;
    ra.n_groups = layer_group ? n_groups : 1;
    ra.row_vecs = row_vecs;
    ra.rot_half = rot_dim / 2;
    ra.rot_vecs = rot_dim * esize / 16;
    ra.half_vecs = h;
    ra.k_scale = k_scale;
    dt = dtype;
    style = rope_style;
    if (k_layout == DSR_K_KX) {
      // the vector map's split-x conditions: head blocks of a power-of-two
      // number (>= 64) of vectors, power-of-two block size, neox partners a
      // multiple of 32 vectors apart
      const int64_t hv = row_bytes / 16 * block_size;
      const int dist = rope_style == DSR_ROPE_NEOX ? rot_dim / 2 / ve * block_size : 0;
      if ((hv & (hv - 1)) || hv < kWave || (block_size & (block_size - 1)) || dist % 32 ||
          page_bytes % (row_bytes * block_size) || page_bytes % 1024)
        return DSR_ERR_SHAPE;
      ra.kx_row_shift = __builtin_ctzll((unsigned long long)hv);
      ra.kx_bs_shift = __builtin_ctz((unsigned)block_size);
      ra.kx_dist = dist;
      ra.row_vecs = (int)hv;
    } else if (k_layout == DSR_K_HND) {
      const int64_t rows = page_bytes / row_bytes;
      if (rows % block_size) return DSR_ERR_SHAPE;
      ra.u.hnd_heads = (int)(rows / block_size);
      ra.u.hnd_block = block_size;
      ra.u.hnd_row_vecs = row_vecs;
    }
  } else if (k_layout == DSR_K_HND) {
    // plain copy of head-major pages: rows of page_bytes / (block_size *
    // num_heads) bytes, whole vectors
    if (num_heads <= 0 || page_bytes % ((int64_t)block_size * num_heads * 16)) return DSR_ERR_SHAPE;
    ra.u.hnd_heads = num_heads;
    ra.u.hnd_block = block_size;
    ra.u.hnd_row_vecs = (int)(page_bytes / ((int64_t)block_size * num_heads) / 16);
  }
  // a plain copy of split-x pages moves raw bytes: the token-major kernel
  const int layout = k_layout == DSR_K_HND ? kRotHnd
                     : k_layout == DSR_K_KX && dst_rope_idx ? kRotKx : kRotNhd;
  if ((int64_t)n_src * n_layers > 0x7fffffffLL) return DSR_ERR_ARG;
  if (n_src == 0 || n_dst == 0 || n_layers == 0) return DSR_OK;
  if (!dst_start) return DSR_ERR_ARG;
  FanArgs fa{};
  fa.ra = ra;
  fa.src_offsets = src_offsets;
  fa.dst_start = dst_start;
  fa.dst_pages = dst_page_ids;
  fa.dst_rope = dst_rope_idx;
  fa.n_src = n_src;
  fa.n_dst = n_dst;
  hipStream_t s = (hipStream_t)stream;
  switch (dt) {
    case DSR_DTYPE_BF16: return launch_fanout<DSR_DTYPE_BF16>(fa, style, layout, s);
    case DSR_DTYPE_FP16: return launch_fanout<DSR_DTYPE_FP16>(fa, style, layout, s);
    case DSR_DTYPE_FP8_E4M3: return launch_fanout<DSR_DTYPE_FP8_E4M3>(fa, style, layout, s);
    default: return launch_fanout<DSR_DTYPE_FP8_E5M2>(fa, style, layout, s);
  }
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Small tables and rotation tables.

namespace {

struct PutArgs {
  uint32_t w[DSR_PUT_BYTES / 4];
};

__global__ __launch_bounds__(kThreads) void kv_put_kernel(uint32_t* dst, int n, PutArgs a) {
  for (int i = threadIdx.x; i < n; i += kThreads) dst[i] = a.w[i];
}

// One (delta, frequency) per lane. In numpy the same cost 2.6 ms of host time for
// 1,024 deltas of 64 frequencies, more than half of a load's launch.
__global__ __launch_bounds__(kThreads) void kv_delta_tables_kernel(const double* x, int n,
                                                                   int half, float2* out) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= (int64_t)n * half) return;
  const int64_t d = i / half;
  double s, c;
  sincos(x[d] * x[n + (i - d * half)], &s, &c);
  out[i] = make_float2((float)c, (float)s);
}

}  // namespace

extern "C" {

int dsr_put(void* dst, const void* src, int64_t bytes, dsr_stream_t stream) {
  if (bytes < 0 || bytes > DSR_PUT_BYTES || bytes % 4) return DSR_ERR_ARG;
  if (bytes == 0) return DSR_OK;
  if (!dst || !src) return DSR_ERR_ARG;
  if (reinterpret_cast<uintptr_t>(dst) & 3) return DSR_ERR_ALIGN;
  PutArgs a;
  memcpy(a.w, src, (size_t)bytes);
  kv_put_kernel<<<1, kThreads, 0, (hipStream_t)stream>>>(static_cast<uint32_t*>(dst),
                                                         (int)(bytes / 4), a);
  return (int)hipGetLastError();
}

int dsr_delta_tables(const double* x, int n, int half, float* out, dsr_stream_t stream) {
  if (n < 0 || half < 0) return DSR_ERR_ARG;
  if (n == 0 || half == 0) return DSR_OK;
  if (!x || !out) return DSR_ERR_ARG;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) & 7)
    return DSR_ERR_ALIGN;
  const int64_t grid = ((int64_t)n * half + kThreads - 1) / kThreads;
  if (grid > max_wg_per_launch()) return DSR_ERR_ARG;
  kv_delta_tables_kernel<<<(unsigned)grid, kThreads, 0, (hipStream_t)stream>>>(
      x, n, half, reinterpret_cast<float2*>(out));
  return (int)hipGetLastError();
}

int dsr_gather_layers(const dsr_gather_args* g, int first, int count, dsr_stream_t stream) {
  if (!g || first < 0 || count < 0 || first > g->n_layers - count) return DSR_ERR_ARG;
  const uint64_t* base = g->layer_base ? g->layer_base + first : nullptr;
  if (g->num_heads)
    return dsr_gather_hnd(base, count, g->kv_stride, g->page_stride, g->page_bytes,
                          g->num_blocks, g->page_ids, g->slot_offsets, g->n_pages, g->staging,
                          g->staging_bytes, g->layer_bytes, g->layer0 + first, g->block_size,
                          g->num_heads, stream);
  return dsr_gather(base, count, g->kv_stride, g->page_stride, g->page_bytes, g->num_blocks,
                    g->page_ids, g->slot_offsets, g->n_pages, g->staging, g->staging_bytes,
                    g->layer_bytes, g->layer0 + first, stream);
}

}  // extern "C"
