"""Host-side wrappers of the HIP gather / scatter / re-rotate kernels.

The functions take torch tensors (device memory and streams only) and call
the C ABI of libdaser_kv.so on torch's current stream. Index tables given as
host data (lists, numpy arrays, CPU tensors) are validated on the host and
uploaded; tables given as device tensors are used as they are (the kernels
then skip out-of-range entries instead of faulting).

Reference semantics restated here:
  * LAYER_SIZE = kv.nbytes // kv.shape[1], SLOT_SIZE = LAYER_SIZE * L
    (daser/connector/daser_connector.py:404-408);
  * record of (slot i, layer l) at i * SLOT_SIZE + l * LAYER_SIZE, holding
    bytes(kv_l[:, block_id]) = K page then V page (:625-632, :536-551).
"""

from __future__ import annotations

import ctypes
import math
from dataclasses import dataclass
from typing import Optional, Sequence

import numpy as np
import torch

from daser_amd import _lib

_DTYPE_CODES = {
    torch.bfloat16: _lib.DSR_DTYPE_BF16,
    torch.float16: _lib.DSR_DTYPE_FP16,
    torch.float8_e4m3fn: _lib.DSR_DTYPE_FP8_E4M3,
    torch.float8_e5m2: _lib.DSR_DTYPE_FP8_E5M2,
}
FP8_DTYPES = (torch.float8_e4m3fn, torch.float8_e5m2)

ROPE_STYLES = {"neox": _lib.DSR_ROPE_NEOX, "gptj": _lib.DSR_ROPE_GPTJ}


@dataclass(frozen=True)
class PagedKVLayout:
    """Geometry of vLLM's per-layer paged caches ``kv_l[2, NB, ...]``.

    Built from the registered caches (reference ``register_kv_caches``,
    daser/connector/daser_connector.py:383-413): layer order is the dict's
    insertion order, every layer must share shape, dtype and strides, and a
    page (``kv_l[0, b]``) must be contiguous. The reference moves
    ``kv_l[:, b]`` of any cache shape as bytes (:545-550, :625-632), and so
    do the page copies here. Re-rotation also needs the element layout of a
    K page (``k_layout``):

    * ``"nhd"``: ``[block_size][H][D]``, the 5-D caches
      ``(2, NB, block_size, H, D)`` of vLLM's FlashAttention-style backends;
    * ``"kx"``: ``[H][D / X][block_size][X]`` with X = 16 / element bytes,
      the 3-D caches ``(2, NB, block_size * H * D)`` of vLLM's
      PagedAttention kernels (its ROCm paged-attention backend);
    * ``"hnd"``: 5-D caches whose pages are stored head-major,
      ``[H][block_size][D]`` (vLLM's HND layout). Their records still hold
      the page in index order ``[block_size][H][D]``, as the reference's
      ``reshape(-1)`` of ``kv[:, b]`` does, so the copies permute rows.

    A cache that is not 5-D carries no head geometry in its shape: pass
    ``block_size`` and ``head_dim`` (``num_heads`` follows from the page
    size); without them copies work and re-rotation is refused.
    """

    num_layers: int
    num_blocks: int
    block_size: int  # 0: unknown (copies only)
    num_heads: int
    head_dim: int
    dtype: torch.dtype
    elem_bytes: int
    page_bytes: int  # one K (or V) page
    kv_stride: int  # bytes K page -> V page
    page_stride: int  # bytes block b -> b + 1
    layer_bytes: int  # LAYER_SIZE of the slot record
    device: torch.device
    k_layout: str = "nhd"

    @property
    def slot_bytes(self) -> int:
        """SLOT_SIZE: one block's record over all layers."""
        return self.layer_bytes * self.num_layers

    @property
    def has_geometry(self) -> bool:
        return self.head_dim > 0 and self.block_size > 0

    @staticmethod
    def from_caches(kv_caches: Sequence[torch.Tensor], *, block_size: Optional[int] = None,
                    head_dim: Optional[int] = None,
                    k_layout: Optional[str] = None) -> "PagedKVLayout":
        if not kv_caches:
            raise ValueError("no KV caches registered")
        t0 = kv_caches[0]
        if t0.dim() < 3 or t0.shape[0] != 2:
            raise ValueError(
                f"expected per-layer KV cache of shape (2, num_blocks, ...) such as "
                f"(2, num_blocks, block_size, num_heads, head_dim), got {tuple(t0.shape)}"
            )
        for t in kv_caches:
            if t.shape != t0.shape or t.dtype != t0.dtype or t.stride() != t0.stride():
                raise ValueError("all layer caches must share shape, dtype and strides")
            if t.device != t0.device:
                raise ValueError("all layer caches must live on one device")
        nb = t0.shape[1]
        s = t0.stride()
        expect, c_order = 1, True
        for dim in range(t0.dim() - 1, 1, -1):  # is a page kv[0, b] C-contiguous?
            if t0.shape[dim] != 1 and s[dim] != expect:
                c_order = False
            expect *= t0.shape[dim]
        page_elems = expect
        e = t0.element_size()
        head_major = False
        if not c_order:
            # vLLM's HND layout: logical (2, NB, bs, H, D), page stored [H][bs][D]
            head_major = (t0.dim() == 5 and s[4] == 1 and s[2] == t0.shape[4] and
                          s[3] == t0.shape[2] * t0.shape[4])
            if not head_major:
                raise ValueError("a KV page kv[0, b] must be contiguous in memory, in "
                                 "(block_size, heads, head_dim) order or head-major")
        if t0.dim() == 5:
            want = "hnd" if head_major else "nhd"
            if k_layout not in (None, want):
                raise ValueError(f"this 5-D cache's pages have the {want!r} layout")
            _, _, bs, h, d = t0.shape
            if (block_size not in (None, bs)) or (head_dim not in (None, d)):
                raise ValueError(f"cache shape {tuple(t0.shape)} disagrees with "
                                 f"block_size={block_size}, head_dim={head_dim}")
            layout = want
        else:
            layout = k_layout or ("kx" if t0.dim() == 3 else "nhd")
            if layout not in ("nhd", "kx"):
                raise ValueError("k_layout must be 'nhd' or 'kx'")
            bs, d, h = int(block_size or 0), int(head_dim or 0), 0
            if bs and d:
                if page_elems % (bs * d):
                    raise ValueError(f"a page of {page_elems} elements is not block_size "
                                     f"{bs} x heads x head_dim {d}")
                h = page_elems // (bs * d)
                if layout == "kx" and (d * e) % 16:
                    raise ValueError("the 'kx' K layout needs head_dim * element size to be "
                                     "a multiple of 16 bytes")
            else:
                bs = d = 0
        page_bytes = page_elems * e
        # LAYER_SIZE as the reference derives it (kv.nbytes // num_blocks).
        layer_bytes = t0.numel() * e // nb if nb else 2 * page_bytes
        return PagedKVLayout(
            num_layers=len(kv_caches),
            num_blocks=nb,
            block_size=bs,
            num_heads=h,
            head_dim=d,
            dtype=t0.dtype,
            elem_bytes=e,
            page_bytes=page_bytes,
            kv_stride=s[0] * e,
            page_stride=s[1] * e,
            layer_bytes=layer_bytes,
            device=t0.device,
            k_layout=layout,
        )


class LayerTable:
    """Device array of per-layer cache base addresses (uint64)."""

    def __init__(self, kv_caches: Sequence[torch.Tensor], **geometry) -> None:
        """``geometry``: ``block_size``, ``head_dim``, ``k_layout`` for caches
        that are not 5-D (see PagedKVLayout)."""
        self.layout = PagedKVLayout.from_caches(kv_caches, **geometry)
        self._caches = list(kv_caches)  # keep the borrowed tensors alive
        ptrs = np.array([t.data_ptr() for t in kv_caches], dtype=np.uint64)
        self.table = torch.from_numpy(ptrs.view(np.int64)).to(self.layout.device)

    def ptr(self, first: int = 0) -> int:
        return self.table.data_ptr() + 8 * first


def _stream_handle(device: torch.device) -> int:
    return torch.cuda.current_stream(device).cuda_stream


def _on_device(x) -> bool:
    return isinstance(x, torch.Tensor) and not x.is_cpu


def _as_device_table(
    x, dtype: torch.dtype, device: torch.device, name: str
) -> torch.Tensor:
    if _on_device(x):
        if x.dtype != dtype or not x.is_contiguous():
            raise ValueError(f"{name} must be a contiguous {dtype} tensor")
        return x
    arr = torch.as_tensor(np.asarray(x), dtype=dtype)
    return _upload(arr, device)


def _upload(arr: torch.Tensor, device: torch.device) -> torch.Tensor:
    """Host table -> device, stream-ordered on the current stream without
    blocking the host: copied into pinned memory (torch's caching host
    allocator keeps it until the copy has run), then an asynchronous copy.
    A pageable copy would wait for the stream's earlier work, e.g. the
    store reads that the load's scatter follows."""
    if device.type != "cuda":
        return arr.to(device)
    if torch.cuda.is_current_stream_capturing():
        # a captured copy would replay from a pinned buffer torch reuses
        raise ValueError("host index tables cannot be used under graph capture: pass "
                         "device tensors")
    return arr.pin_memory().to(device, non_blocking=True)


def _host_array(x, np_dtype) -> Optional[np.ndarray]:
    if isinstance(x, torch.Tensor):
        if not x.is_cpu:
            return None
        return x.numpy().astype(np_dtype, copy=False)
    return np.asarray(x, dtype=np_dtype)


def _validate(layout: PagedKVLayout, page_ids, slot_offsets, staging, layer0, n_layers,
              records_written: bool):
    ids = _host_array(page_ids, np.int64)
    offs = _host_array(slot_offsets, np.int64)
    if ids is not None and offs is not None and ids.shape != offs.shape:
        raise ValueError("page_ids and slot_offsets differ in length")
    if ids is not None and ids.size and (ids.min() < 0 or ids.max() >= layout.num_blocks):
        raise IndexError(f"block id out of range [0, {layout.num_blocks})")
    if offs is not None and offs.size:
        end = offs.max() + (layer0 + n_layers - 1) * layout.layer_bytes + 2 * layout.page_bytes
        if offs.min() < 0 or end > staging.numel() * staging.element_size():
            raise IndexError("slot record outside the staging buffer")
        if np.any(offs % 16):
            raise ValueError("slot offsets must be multiples of 16 bytes")
        span = (n_layers - 1) * layout.layer_bytes + 2 * layout.page_bytes
        so = np.sort(offs)
        # a gather writes the records: two pages' records must not overlap
        # (a scatter may read one cached record into several pages)
        if records_written and so.size > 1 and np.any(np.diff(so) < span):
            raise ValueError("slot records of two pages overlap")


def check_tables(table: "LayerTable", page_ids, slot_offsets, staging: torch.Tensor, *,
                 layer0: int = 0, records_written: bool = False) -> None:
    """The checks the copy wrappers run on host tables, for device-resident
    ones (which the wrappers trust: the kernels skip a page whose block id or
    record range is out of bounds instead of faulting, where the reference's
    indexing would raise). Copies the tables to the host, so it synchronises
    the stream: for debugging and for callers that build tables on the
    device and want the reference's errors."""
    def host(x, dt):
        return x.detach().cpu().numpy().astype(dt) if isinstance(x, torch.Tensor) \
            else np.asarray(x, dt)

    _validate(table.layout, host(page_ids, np.int64), host(slot_offsets, np.int64), staging,
              layer0, table.layout.num_layers, records_written)


def dest_order(page_ids, slot_offsets, extra=None):
    """Host tables of a scatter, reordered by destination block (stable).

    Processing order does not change the result (each destination block is
    written once) but near-sequential page writes run faster. A destination
    block listed several times keeps only its last entry: the reference's
    sequential copies (daser_connector.py:536-551) leave the last one's
    bytes, while copies inside one launch would race. Device tables are
    returned unchanged (there, duplicates race)."""
    ids = _host_array(page_ids, np.int64)
    offs = _host_array(slot_offsets, np.int64)
    if ids is None or offs is None or ids.size == 0:
        return page_ids, slot_offsets, extra
    order = np.argsort(ids, kind="stable")
    sids = ids[order]
    if sids.size > 1 and np.any(sids[1:] == sids[:-1]):
        # within a run of equal ids the stable order keeps list order: the
        # run's last element is the list's last entry for that block
        last = np.append(sids[1:] != sids[:-1], True)
        order, sids = order[last], sids[last]
    ex = None
    if extra is not None:
        e = _host_array(extra, np.int64)
        ex = extra if e is None else e[order]
    return sids, offs[order], ex


_PLAN_ERRORS = {
    _lib.DSR_PLAN_ERR_RECORD: (IndexError, "slot record outside the staging buffer"),
    _lib.DSR_PLAN_ERR_ALIGN: (ValueError, "slot offsets must be multiples of 16 bytes"),
    _lib.DSR_PLAN_ERR_ROPE: (IndexError, "rope_idx outside [-1, n_tables)"),
    _lib.DSR_PLAN_ERR_OVERLAP: (ValueError, "slot records of two pages overlap"),
    _lib.DSR_PLAN_ERR_SLOT: (IndexError, "slot outside the block pool"),
    _lib.DSR_PLAN_ERR_ROW: (IndexError, "token row outside the staging buffer"),
    _lib.DSR_PLAN_ERR_ROWALIGN: (ValueError, "row offsets must be multiples of 16 bytes"),
}


def _plan_check(name: str, rc: int, num_blocks: int) -> None:
    if rc == _lib.DSR_PLAN_ERR_BLOCK:
        raise IndexError(f"block id out of range [0, {num_blocks})")
    if rc in _PLAN_ERRORS:
        kind, text = _PLAN_ERRORS[rc]
        raise kind(text)
    _lib.check(name, rc)


def _host_list(x) -> Optional[np.ndarray]:
    """A host table as a contiguous int64 vector; None for device tensors and
    for anything that is no vector."""
    a = _host_array(x, np.int64)
    return np.ascontiguousarray(a) if a is not None and a.ndim == 1 else None


def _addr(a: Optional[np.ndarray]) -> Optional[int]:
    return None if a is None else a.__array_interface__["data"][0]


_BLIT_BYTES = 16 << 10


def _plan_room(size: int) -> torch.Tensor:
    """Host memory for a plan: pinned where its upload is a copy."""
    return torch.empty(size, dtype=torch.uint8, pin_memory=size > _lib.DSR_PUT_BYTES)


def _upload_plan(host: torch.Tensor, at: int, nbytes: int, device: torch.device,
                 stream: int) -> torch.Tensor:
    """``nbytes`` of the plan at ``at``, in stream order. Copies of up to 16 KiB
    run as a kernel on the stream; larger ones go to a copy engine, which holds
    the stream up by some 10 us (a load of 2,000 pages 139 against 152 us), so two
    of the former are taken before one of the latter."""
    if host.numel() > _lib.DSR_PUT_BYTES and nbytes > 2 * _BLIT_BYTES:
        return host[at:at + nbytes].to(device, non_blocking=True)
    buf = torch.empty(nbytes, dtype=torch.uint8, device=device)
    if host.numel() > _lib.DSR_PUT_BYTES:
        for i in range(0, nbytes, _BLIT_BYTES):
            k = min(_BLIT_BYTES, nbytes - i)
            buf[i:i + k].copy_(host[at + i:at + i + k], non_blocking=True)
        return buf
    _lib.check("dsr_put", _lib.lib().dsr_put(buf.data_ptr(), host.data_ptr() + at, nbytes, stream))
    return buf


class _HostPlan:
    """Host tables of one call, planned by the library (dsr_plan_load,
    dsr_plan_gather) into one buffer and uploaded with one kernel (up to
    DSR_PUT_BYTES) or one asynchronous copy from pinned memory. ``offsets``,
    ``start``, ``ids`` and ``rope`` are the addresses of its sections."""

    def __init__(self, n: int, device: torch.device, fill) -> None:
        """``fill(address, size, plan)`` has the library write the tables."""
        cuda = device.type == "cuda"
        if cuda and torch.cuda.is_current_stream_capturing():
            raise ValueError("host index tables cannot be used under graph capture: pass "
                             "device tensors")
        size = _lib.plan_bytes(n)
        host = _plan_room(size) if cuda else torch.empty(size, dtype=torch.uint8)
        self.plan = plan = _lib.Plan()
        fill(host.data_ptr(), size, ctypes.addressof(plan))
        if cuda:
            self.stream = _stream_handle(device)
            self.buf = _upload_plan(host, 0, plan.bytes, device, self.stream)
        else:  # caches in host memory: the tables stay there
            self.stream, self.buf = None, host[:plan.bytes]
        base = self.buf.data_ptr()
        self.offsets, self.start = base, base + plan.off_start
        self.ids, self.rope = base + plan.off_ids, base + plan.off_rope

    def table(self, at: int, count: int, dtype: torch.dtype) -> torch.Tensor:
        """A section as a tensor (a view that keeps the buffer)."""
        width = torch.empty(0, dtype=dtype).element_size()
        return self.buf[at:at + count * width].view(dtype)


def _layer_range(lay: PagedKVLayout, layers) -> tuple[int, int]:
    first, count = (0, lay.num_layers) if layers is None else layers
    if first < 0 or count < 0 or first + count > lay.num_layers:
        raise IndexError("layer range outside the registered caches")
    return first, count


def _check_staging(lay: PagedKVLayout, staging: torch.Tensor) -> int:
    if staging.device != lay.device:
        raise ValueError("staging must live on the KV caches' device")
    if not staging.is_contiguous():
        raise ValueError("staging must be contiguous")
    return staging.numel() * staging.element_size()


def _load_plan(lay: PagedKVLayout, ids, offs, ridx, n_tables: int, staging_bytes: int,
               rec_layers: int, fanout: bool) -> _HostPlan:
    """The tables of a load (host vectors), in destination order or grouped by
    record."""
    rec_end = (rec_layers - 1) * lay.layer_bytes + 2 * lay.page_bytes
    lib = _lib.lib()

    def fill(out: int, size: int, plan: int) -> None:
        _plan_check("dsr_plan_load", lib.dsr_plan_load(
            _addr(ids), _addr(offs), _addr(ridx), ids.size, lay.num_blocks, max(rec_end, 0),
            staging_bytes, n_tables, int(fanout), out, size, plan), lay.num_blocks)

    return _HostPlan(ids.size, lay.device, fill)


def _copy_args(table: LayerTable, page_ids, slot_offsets, staging, layer0, layers,
               records_written: bool = False):
    lay = table.layout
    first, count = (0, lay.num_layers) if layers is None else layers
    if first < 0 or count < 0 or first + count > lay.num_layers:
        raise IndexError("layer range outside the registered caches")
    if staging.device != lay.device:
        raise ValueError("staging must live on the KV caches' device")
    if not staging.is_contiguous():
        raise ValueError("staging must be contiguous")
    _validate(lay, page_ids, slot_offsets, staging, layer0 + first, count, records_written)
    ids = _as_device_table(page_ids, torch.int32, lay.device, "page_ids")
    offs = _as_device_table(slot_offsets, torch.int64, lay.device, "slot_offsets")
    if ids.numel() != offs.numel():
        raise ValueError("page_ids and slot_offsets differ in length")
    args = (
        table.ptr(first),
        count,
        lay.kv_stride,
        lay.page_stride,
        lay.page_bytes,
        lay.num_blocks,
        ids.data_ptr(),
        offs.data_ptr(),
        ids.numel(),
        staging.data_ptr(),
        staging.numel() * staging.element_size(),
        lay.layer_bytes,
        layer0 + first,
    )
    return args, (ids, offs)


def gather(
    table: LayerTable,
    page_ids,
    slot_offsets,
    staging: torch.Tensor,
    *,
    layer0: int = 0,
    layers: Optional[tuple[int, int]] = None,
) -> None:
    """Packs pages into slot records (reference save loop, :610-632).

    ``layers=(first, count)`` restricts the launch to a layer range; the
    record index of table layer ``first + i`` is ``layer0 + first + i``.
    """
    lay = table.layout
    fn, name, extra = _copy_entry(lay, "dsr_gather")
    if _on_device(page_ids):
        args, _tables = _copy_args(table, page_ids, slot_offsets, staging, layer0, layers,
                                   records_written=True)
        _lib.check(name, fn(*args, *extra, _stream_handle(lay.device)))
        return
    (ids, offs), _plan = _gather_tables(table, page_ids, slot_offsets, staging, layer0, layers)
    first, count = _layer_range(lay, layers)
    rc = fn(table.ptr(first), count, lay.kv_stride, lay.page_stride, lay.page_bytes,
            lay.num_blocks, ids.data_ptr(), offs.data_ptr(), ids.numel(), staging.data_ptr(),
            staging.numel() * staging.element_size(), lay.layer_bytes, layer0 + first, *extra,
            _stream_handle(lay.device))
    _lib.check(name, rc)


def _copy_entry(lay: PagedKVLayout, base: str):
    """The copy entry point for the layout's pages and its extra arguments:
    head-major pages go through the row-permuting ``*_hnd`` variant."""
    if lay.k_layout == "hnd":
        return getattr(_lib.lib(), base + "_hnd"), base + "_hnd", (lay.block_size,
                                                                   lay.num_heads)
    return getattr(_lib.lib(), base), base, ()


class PreparedGather:
    """A gather of fixed page tables into a fixed staging buffer, checked and
    converted once; each call launches it for a layer range. For callers
    that launch the same gather once per layer (the connector's
    save_kv_layer runs 32-80 times a step), so that a call costs one ctypes
    launch and no table checks or conversions."""

    def __init__(self, table: LayerTable, page_ids, slot_offsets, staging: torch.Tensor,
                 *, layer0: int = 0) -> None:
        lay = table.layout
        self.tables, plan = _gather_tables(table, page_ids, slot_offsets, staging, layer0, None)
        ids, offs = self.tables  # (page_ids, slot_offsets) as device tensors
        self._keep = (table, staging, plan)
        hnd = lay.k_layout == "hnd"
        self._args = _lib.GatherArgs(
            table.ptr(), lay.kv_stride, lay.page_stride, lay.page_bytes, lay.num_blocks,
            ids.data_ptr(), offs.data_ptr(), staging.data_ptr(),
            staging.numel() * staging.element_size(), lay.layer_bytes, lay.num_layers, layer0,
            ids.numel(), lay.block_size if hnd else 0, lay.num_heads if hnd else 0, 0)
        self._args_ptr = ctypes.addressof(self._args)
        self._n_layers = lay.num_layers
        self._fn = _lib.lib().dsr_gather_layers

    def __call__(self, first: int, count: int, stream: int) -> None:
        """Gathers table layers [first, first + count) on ``stream`` (a HIP
        stream handle, e.g. ``torch.cuda.current_stream().cuda_stream``)."""
        if first < 0 or count < 0 or first + count > self._n_layers:
            raise IndexError("layer range outside the registered caches")
        rc = self._fn(self._args_ptr, first, count, stream)
        if rc:
            _lib.check("dsr_gather_layers", rc)


def _gather_tables(table: LayerTable, page_ids, slot_offsets, staging, layer0, layers):
    """Checked device tables (page_ids, slot_offsets) of a gather and, of host
    tables, the plan that holds them."""
    lay = table.layout
    ids = offs = None
    if not _on_device(page_ids):
        ids, offs = _host_list(page_ids), _host_list(slot_offsets)
    if ids is None or offs is None or not ids.size or lay.device.type != "cuda":
        return _copy_args(table, page_ids, slot_offsets, staging, layer0, layers,
                          records_written=True)[1], None
    first, count = _layer_range(lay, layers)
    nbytes = _check_staging(lay, staging)
    if ids.shape != offs.shape:
        raise ValueError("page_ids and slot_offsets differ in length")
    span = (count - 1) * lay.layer_bytes + 2 * lay.page_bytes
    end = span + (layer0 + first) * lay.layer_bytes
    lib = _lib.lib()

    def fill(out: int, size: int, plan: int) -> None:
        _plan_check("dsr_plan_gather", lib.dsr_plan_gather(
            _addr(ids), _addr(offs), ids.size, lay.num_blocks, max(end, 0), max(span, 0),
            nbytes, out, size, plan), lay.num_blocks)

    h = _HostPlan(ids.size, lay.device, fill)
    return (h.table(h.plan.off_ids, ids.size, torch.int32),
            h.table(0, ids.size, torch.int64)), h


def scatter(
    table: LayerTable,
    page_ids,
    slot_offsets,
    staging: torch.Tensor,
    *,
    layer0: int = 0,
    layers: Optional[tuple[int, int]] = None,
    shared_records: Optional[bool] = None,
) -> None:
    """Unpacks slot records into pages (reference load loop, :536-551).

    ``shared_records``: several pages read the same records. Host tables
    then take the fan-out load (:class:`PreparedFanout`: each record read
    once and written to all of its pages) where the pages allow it, device
    tables a launch shaped for cache-served reads. None: inferred from host
    ``slot_offsets`` (at most half of them distinct), False for device
    tables. Results do not depend on it. Host tables are planned by the library
    (dsr_plan_load) and uploaded once."""
    host = _host_tables(table, page_ids, slot_offsets)
    if host is not None:
        _load_host(table, *host, staging, layer0, layers, shared_records)
        return
    if shared_records is None:
        shared_records = _shared_offsets(slot_offsets)
    page_ids, slot_offsets, _ = dest_order(page_ids, slot_offsets)
    args, _tables = _copy_args(table, page_ids, slot_offsets, staging, layer0, layers)
    stream = _stream_handle(table.layout.device)
    _scatter(table.layout, args, shared_records, stream)


def _scatter(lay: PagedKVLayout, args, shared: bool, stream: int) -> None:
    """The layout's copy entry point on device tables."""
    if shared and lay.k_layout != "hnd":
        _lib.check("dsr_scatter_ex",
                   _lib.lib().dsr_scatter_ex(*args, _lib.DSR_SHARED_RECORDS, stream))
        return
    fn, name, extra = _copy_entry(lay, "dsr_scatter")
    _lib.check(name, fn(*args, *extra, stream))


def _host_tables(table: LayerTable, page_ids, slot_offsets):
    """(page_ids, slot_offsets) as host vectors if the library can plan them:
    both on the host, not empty, of one length."""
    if _on_device(page_ids):
        return None
    ids, offs = _host_list(page_ids), _host_list(slot_offsets)
    if ids is None or offs is None or not ids.size or ids.size != offs.size or \
            table.layout.device.type != "cuda":
        return None
    return ids, offs


def _load_host(table: LayerTable, ids: np.ndarray, offs: np.ndarray, staging: torch.Tensor,
               layer0: int, layers, shared: Optional[bool], rope=None) -> None:
    """A load of host tables: planned, uploaded once, launched. ``rope``: None,
    or (rope_idx, cos_sin, rot_dim, style, n_tables, n_groups, layer_group on the
    device or None, k_scale pointer)."""
    lay = table.layout
    lib = _lib.lib()
    if shared is None:
        shared = lib.dsr_plan_shared(_addr(offs), ids.size) == 1
    fan = shared and (fanout_supported(lay, rope[2], rope[3]) if rope else fanout_supported(lay))
    first, count = _layer_range(lay, layers)
    nbytes = _check_staging(lay, staging)
    ridx, n_tables = (rope[0], rope[4]) if rope else (None, 0)
    p = _load_plan(lay, ids, offs, ridx, n_tables, nbytes, layer0 + first + count, fan)
    plan = p.plan
    if fan:
        tail = (None, 0, None, 0, 0, 0, 0, 0, None) if rope is None else _fan_tail(lay, rope)
        _lib.check("dsr_scatter_fanout", lib.dsr_scatter_fanout(
            table.ptr(first), count, lay.kv_stride, lay.page_stride, lay.page_bytes,
            lay.num_blocks, p.offsets, plan.n_src, p.start, p.ids, p.rope if rope else None,
            plan.n_pages, staging.data_ptr(), nbytes, lay.layer_bytes, layer0 + first, *tail,
            _K_LAYOUTS[lay.k_layout], lay.block_size, lay.num_heads, p.stream))
        return
    args = (table.ptr(first), count, lay.kv_stride, lay.page_stride, lay.page_bytes,
            lay.num_blocks, p.ids, p.offsets, plan.n_pages, staging.data_ptr(), nbytes,
            lay.layer_bytes, layer0 + first)
    if rope is None:
        _scatter(lay, args, shared, p.stream)
        return
    _, cos_sin, rot_dim, style, n_tables, n_groups, lg_d, ks_ptr = rope
    _rerotate(lay, args, cos_sin.data_ptr(), p.rope, n_tables, n_groups, lg_d, rot_dim, style,
              ks_ptr, shared, p.stream)


def _fan_tail(lay: PagedKVLayout, rope):
    _, cos_sin, rot_dim, style, n_tables, n_groups, lg_d, ks_ptr = rope
    return (cos_sin.data_ptr(), n_tables, None if lg_d is None else lg_d.data_ptr(), n_groups,
            lay.head_dim, rot_dim, ROPE_STYLES[style], _DTYPE_CODES[lay.dtype], ks_ptr)


def _rerotate(lay: PagedKVLayout, args, cos_sin: int, rope_idx: int, n_tables: int,
              n_groups: int, lg_d, rot_dim: int, style: str, ks_ptr, shared: bool,
              stream: int) -> None:
    """The layout's re-rotation entry point on device tables."""
    common = (*args, cos_sin, rope_idx, n_tables, None if lg_d is None else lg_d.data_ptr(),
              n_groups, lay.head_dim, rot_dim, ROPE_STYLES[style], _DTYPE_CODES[lay.dtype],
              ks_ptr)
    flags = _lib.DSR_REROTATE_SHARED_RECORDS if shared else 0
    if lay.k_layout in ("kx", "hnd"):
        name = "dsr_scatter_rerotate_" + lay.k_layout
        _lib.check(name, getattr(_lib.lib(), name)(*common, lay.block_size, flags, stream))
    else:
        _lib.check("dsr_scatter_rerotate",
                   _lib.lib().dsr_scatter_rerotate(*common, flags, stream))


def _shared_offsets(slot_offsets) -> bool:
    """At most half of the host record offsets are distinct."""
    offs_h = _host_array(slot_offsets, np.int64)
    return offs_h is not None and offs_h.size > 1 and 2 * np.unique(offs_h).size <= offs_h.size


def fanout_tables(page_ids: np.ndarray, slot_offsets: np.ndarray,
                  rope_idx: Optional[np.ndarray] = None):
    """Host tables of a scatter (destination order, one entry per block)
    grouped by source record: (src_offsets, dst_start, dst_pages, dst_rope),
    where the destinations of source s are entries dst_start[s] to
    dst_start[s + 1] - 1, in block order. For callers of the C ABI; the loads
    here have the library group them (dsr_plan_load)."""
    ids = np.asarray(page_ids, np.int64)
    offs = np.asarray(slot_offsets, np.int64)
    order = np.argsort(offs, kind="stable")  # keeps block order inside a source
    so = offs[order]
    first = np.ones(so.size, bool)
    first[1:] = so[1:] != so[:-1]
    starts = np.nonzero(first)[0]
    dst_start = np.append(starts, so.size).astype(np.int32)
    dst_rope = None if rope_idx is None else np.asarray(rope_idx, np.int64)[order]
    return so[starts], dst_start, ids[order], dst_rope


_K_LAYOUTS = {"nhd": _lib.DSR_K_NHD, "kx": _lib.DSR_K_KX, "hnd": _lib.DSR_K_HND}


def fanout_supported(lay: PagedKVLayout, rot_dim: Optional[int] = None,
                     style: str = "neox") -> bool:
    """Whether dsr_scatter_fanout takes these pages (``rot_dim`` None: a
    plain copy), asked of the library itself: a call with no work checks
    the geometry and launches nothing. It takes pages of at most 32 KiB in
    every cache layout; the re-rotation wants whole-vector rotary widths
    and neox partners a power of two of at most 32 vectors apart (split-x
    pages: the split-x kernels' conditions)."""
    rot = rot_dim is not None
    if rot and (not lay.has_geometry or lay.dtype not in _DTYPE_CODES):
        return False
    if lay.k_layout != "nhd" and lay.block_size <= 0:
        return False
    rc = _lib.lib().dsr_scatter_fanout(
        16, lay.num_layers, lay.kv_stride, lay.page_stride, lay.page_bytes, lay.num_blocks,
        None, 0, None, None, 16 if rot else None, 0, 16, 0, lay.layer_bytes, 0, None, 0, None, 0,
        lay.head_dim, rot_dim or 0, ROPE_STYLES[style], _DTYPE_CODES.get(lay.dtype, 0), 16,
        _K_LAYOUTS[lay.k_layout], lay.block_size, lay.num_heads, None)
    return rc == _lib.DSR_OK


class PreparedFanout:
    """A load of host tables whose pages share records (a cached chunk
    placed in several requests), through dsr_scatter_fanout: each record is
    read once and written to all of its pages. The tables are checked,
    grouped by record (dsr_plan_load, as :func:`fanout_tables`) and uploaded
    once; each call
    launches the load on the current stream. ``rope``: None for a plain
    copy, else (rope_idx, cos_sin, rot_dim, style, k_scale, layer_group) as
    for :func:`scatter_rerotate`. Pages must satisfy
    :func:`fanout_supported`; a block listed twice keeps its last entry."""

    def __init__(self, table: LayerTable, page_ids, slot_offsets, staging: torch.Tensor, *,
                 rope=None, layer0: int = 0, layers: Optional[tuple[int, int]] = None) -> None:
        lay = table.layout
        ids, offs = _host_list(page_ids), _host_list(slot_offsets)
        if ids is None or offs is None:
            raise ValueError("PreparedFanout takes host tables")
        first, count = _layer_range(lay, layers)
        if staging.device != lay.device or not staging.is_contiguous():
            raise ValueError("staging must be a contiguous tensor on the KV caches' device")
        if ids.shape != offs.shape:
            raise ValueError("page_ids and slot_offsets differ in length")
        tail = (None, 0, None, 0, 0, 0, 0, 0, None)
        ridx, n_tables, keep = None, 0, []
        if rope is not None:
            rope_idx, cos_sin, rot_dim, style, k_scale, layer_group = rope
            rot_dim, n_tables, n_groups, lg_d, ks_ptr = _rope_args(
                lay, cos_sin, rope_idx, rot_dim, k_scale, layer0, layer_group)
            ridx = _host_list(rope_idx)
            if ridx is None:
                raise ValueError("PreparedFanout takes host tables")
            if ridx.shape != ids.shape:
                raise ValueError("rope_idx and page_ids differ in length")
            if not fanout_supported(lay, rot_dim, style):
                raise ValueError("these pages need the per-page re-rotation kernels")
            tail = _fan_tail(lay, (ridx, cos_sin, rot_dim, style, n_tables, n_groups, lg_d,
                                   ks_ptr))
            keep += [cos_sin, lg_d, k_scale]
        elif not fanout_supported(lay):
            raise ValueError("these pages need the per-page scatter kernels")
        nbytes = staging.numel() * staging.element_size()
        p = _load_plan(lay, ids, offs, ridx, n_tables, nbytes, layer0 + first + count, True)
        self._keep = keep + [table, staging, p]
        self.n_src, self.n_dst = p.plan.n_src, p.plan.n_pages
        self._args = (table.ptr(first), count, lay.kv_stride, lay.page_stride, lay.page_bytes,
                      lay.num_blocks, p.offsets, self.n_src, p.start, p.ids,
                      None if ridx is None else p.rope, self.n_dst, staging.data_ptr(), nbytes,
                      lay.layer_bytes, layer0 + first, *tail, _K_LAYOUTS[lay.k_layout],
                      lay.block_size, lay.num_heads)
        self._device = lay.device

    def __call__(self) -> None:
        rc = _lib.lib().dsr_scatter_fanout(*self._args, _stream_handle(self._device))
        _lib.check("dsr_scatter_fanout", rc)


def _rope_args(lay: PagedKVLayout, cos_sin: torch.Tensor, rope_idx, rot_dim, k_scale,
               layer0: int, layer_group):
    """Checks the re-rotation inputs shared by the page and token forms
    (rope_idx None: its entries are checked elsewhere);
    returns (rot_dim, n_tables, n_groups or 0, device layer_group or None,
    k_scale pointer or None)."""
    if lay.dtype not in _DTYPE_CODES:
        raise TypeError(f"re-rotation does not support KV dtype {lay.dtype}")
    if not lay.has_geometry:
        raise ValueError("re-rotation needs the K page geometry: register caches that are "
                         "not 5-D with block_size and head_dim")
    rot_dim = lay.head_dim if rot_dim is None else rot_dim
    grouped = layer_group is not None
    if cos_sin.dtype != torch.float32 or cos_sin.dim() != (4 if grouped else 3) or \
            cos_sin.shape[-2:] != (rot_dim // 2, 2):
        shape = "[groups, n, {}, 2]" if grouped else "[n, {}, 2]"
        raise ValueError("cos_sin must be float32 " + shape.format(rot_dim // 2))
    if cos_sin.device != lay.device or not cos_sin.is_contiguous():
        raise ValueError("cos_sin must be a contiguous device tensor")
    n_groups = cos_sin.shape[0] if grouped else 1
    n_tables = cos_sin.shape[-3]
    ridx = None if rope_idx is None else _host_array(rope_idx, np.int64)
    if ridx is not None and ridx.size and (ridx.max() >= n_tables or ridx.min() < -1):
        raise IndexError("rope_idx outside [-1, n_tables)")
    lg_d = None
    if grouped:
        lg = _host_array(layer_group, np.int64)
        if lg is not None and (lg.size < layer0 + lay.num_layers or
                               (lg.size and (lg.min() < -1 or lg.max() >= n_groups))):
            raise IndexError("layer_group needs one group in [-1, n_groups) per layer")
        lg_d = _as_device_table(layer_group, torch.int32, lay.device, "layer_group")
    ks_ptr = None
    if lay.dtype in FP8_DTYPES:
        if k_scale is None:
            raise ValueError("fp8 re-rotation needs per-layer k_scale")
        if (
            k_scale.dtype != torch.float32
            or k_scale.device != lay.device
            or k_scale.numel() < layer0 + lay.num_layers
        ):
            raise ValueError("k_scale must be a float32 device tensor with one scale per layer")
        ks_ptr = k_scale.data_ptr()
    return rot_dim, n_tables, n_groups if grouped else 0, lg_d, ks_ptr


def scatter_rerotate(
    table: LayerTable,
    page_ids,
    slot_offsets,
    staging: torch.Tensor,
    cos_sin: torch.Tensor,
    rope_idx,
    *,
    rot_dim: Optional[int] = None,
    style: str = "neox",
    k_scale: Optional[torch.Tensor] = None,
    layer0: int = 0,
    layers: Optional[tuple[int, int]] = None,
    layer_group=None,
    shared_records: Optional[bool] = None,
) -> None:
    """Scatter with K re-rotated by ``cos_sin[rope_idx[p]]`` (-1 = copy).

    ``cos_sin`` is a float32 tensor ``[n_tables, rot_dim/2, 2]`` from
    :func:`daser_amd.position.delta_tables`; ``k_scale`` holds per-layer
    fp32 scales (fp8 caches only). For models whose layers differ in RoPE
    (other frequencies, or none), ``cos_sin`` is ``[n_groups, n_tables,
    rot_dim/2, 2]`` and ``layer_group[layer0 + l]`` picks layer l's group
    (-1: no RoPE, K copied).

    ``shared_records``: several pages read the same records (a cached chunk
    placed in several requests). Host tables then take the fan-out load
    (:class:`PreparedFanout`) where the pages allow it, device tables a
    launch shaped for cache-served reads. None: inferred from host
    ``slot_offsets`` (at most half of them distinct), False for device
    tables. Results do not depend on it.
    """
    lay = table.layout
    host, ridx = _host_tables(table, page_ids, slot_offsets), _host_list(rope_idx)
    planned = host is not None and ridx is not None and ridx.size == host[0].size
    rot_dim, n_tables, n_groups, lg_d, ks_ptr = _rope_args(
        lay, cos_sin, None if planned else rope_idx, rot_dim, k_scale, layer0, layer_group)
    if planned:
        _load_host(table, *host, staging, layer0, layers, shared_records,
                   (ridx, cos_sin, rot_dim, style, n_tables, n_groups, lg_d, ks_ptr))
        return
    if shared_records is None:
        shared_records = _shared_offsets(slot_offsets)
    page_ids, slot_offsets, rope_idx = dest_order(page_ids, slot_offsets, rope_idx)
    args, _tables = _copy_args(table, page_ids, slot_offsets, staging, layer0, layers)
    ridx_d = _as_device_table(rope_idx, torch.int32, lay.device, "rope_idx")
    if ridx_d.numel() != _tables[0].numel():
        raise ValueError("rope_idx and page_ids differ in length")
    _rerotate(lay, args, cos_sin.data_ptr(), ridx_d.data_ptr(), n_tables, n_groups, lg_d, rot_dim,
              style, ks_ptr, shared_records, _stream_handle(lay.device))


def _slots_args(table: LayerTable, slot_mapping, row_offsets, staging, layer0, layers,
                records_written: bool):
    lay = table.layout
    if lay.k_layout != "nhd" or not lay.has_geometry:
        raise ValueError("the token form needs token-major pages ([block_size][H][D]) of "
                         "known geometry")
    first, count = (0, lay.num_layers) if layers is None else layers
    if first < 0 or count < 0 or first + count > lay.num_layers:
        raise IndexError("layer range outside the registered caches")
    if staging.device != lay.device or not staging.is_contiguous():
        raise ValueError("staging must be a contiguous tensor on the caches' device")
    row_bytes = lay.num_heads * lay.head_dim * lay.elem_bytes
    sm = _host_array(slot_mapping, np.int64)
    ro = _host_array(row_offsets, np.int64)
    if sm is not None and ro is not None:
        if sm.shape != ro.shape:
            raise ValueError("slot_mapping and row_offsets differ in length")
        valid = sm >= 0
        if valid.any():
            if sm[valid].max() >= lay.num_blocks * lay.block_size:
                raise IndexError("slot outside the block pool")
            r = ro[valid]
            end = r.max() + (layer0 + first + count - 1) * lay.layer_bytes + lay.page_bytes \
                + row_bytes
            if r.min() < 0 or end > staging.numel() * staging.element_size():
                raise IndexError("token row outside the staging buffer")
            if np.any(r % 16):
                raise ValueError("row offsets must be multiples of 16 bytes")
            # Two tokens writing the same record row (gather) or the same
            # slot (scatter) would race inside the launch; as the reference's
            # sequential copies leave the last one's bytes, the earlier ones
            # become padding (slot -1) in a copy of the host table.
            if records_written:
                if np.unique(r).size != r.size:
                    idx = np.nonzero(valid)[0]
                    _, last_rev = np.unique(r[::-1], return_index=True)
                    keep = np.zeros(idx.size, bool)
                    keep[idx.size - 1 - last_rev] = True
                    sm = sm.copy()
                    sm[idx[~keep]] = -1
                    slot_mapping = sm
            else:
                slot_mapping = _last_per_slot(sm)
    sm_d = _as_device_table(slot_mapping, torch.int64, lay.device, "slot_mapping")
    ro_d = _as_device_table(row_offsets, torch.int64, lay.device, "row_offsets")
    if sm_d.numel() != ro_d.numel():
        raise ValueError("slot_mapping and row_offsets differ in length")
    return (table.ptr(first), count, lay.kv_stride, lay.page_stride, lay.page_bytes,
            lay.num_blocks, lay.block_size, row_bytes, sm_d.data_ptr(), ro_d.data_ptr(),
            sm_d.numel(), staging.data_ptr(), staging.numel() * staging.element_size(),
            lay.layer_bytes, layer0 + first), (sm_d, ro_d)


def _slots_host(table: LayerTable, slot_mapping, row_offsets, staging: torch.Tensor, layer0: int,
                layers, mode: int, rope=None) -> bool:
    """A token-form call with host tables: planned by the library, its whole
    pages (loads) through the page form, the other tokens through the token
    kernels. ``rope`` as for :func:`_load_host`. False, having done nothing, for
    tables that the library cannot plan (device tables, empty or odd ones) and
    for padding alone."""
    if _on_device(slot_mapping):
        return False
    lay = table.layout
    sm, ro = _host_list(slot_mapping), _host_list(row_offsets)
    if sm is None or ro is None or not sm.size or sm.size != ro.size or \
            lay.device.type != "cuda" or not lay.has_geometry or lay.k_layout != "nhd":
        return False
    ridx, n_tables = (rope[0], rope[4]) if rope else (None, 0)
    if rope and (ridx is None or ridx.size != sm.size):
        return False
    first, count = _layer_range(lay, layers)
    if staging.device != lay.device or not staging.is_contiguous():
        raise ValueError("staging must be a contiguous tensor on the caches' device")
    if torch.cuda.is_current_stream_capturing():
        raise ValueError("host index tables cannot be used under graph capture: pass "
                         "device tensors")
    nbytes = staging.numel() * staging.element_size()
    row = lay.num_heads * lay.head_dim * lay.elem_bytes
    end = (layer0 + first + count - 1) * lay.layer_bytes + lay.page_bytes + row
    size = _lib.slot_plan_bytes(sm.size)
    host = _plan_room(size)
    plan = _lib.SlotPlan()
    lib = _lib.lib()
    _plan_check("dsr_plan_slots", lib.dsr_plan_slots(
        _addr(sm), _addr(ro), _addr(ridx), sm.size, lay.num_blocks, lay.block_size, row,
        max(end, 0), nbytes, n_tables, mode, host.data_ptr(), size, ctypes.addressof(plan)),
        lay.num_blocks)
    if not plan.n_pages and not plan.n_tokens:  # padding alone: the launch's checks remain
        return False
    if plan.n_pages:
        at = host.numpy()
        ids, offs, prope = (at[o:o + 8 * plan.n_pages].view(np.int64) for o in
                            (plan.off_ids, plan.off_offsets,
                             plan.off_page_rope if rope else plan.off_ids))
        _load_host(table, ids, offs, staging, layer0, layers, None,
                   (prope, *rope[1:]) if rope else None)
    if not plan.n_tokens:
        return True
    stream = _stream_handle(lay.device)
    buf = _upload_plan(host, plan.off_slots, plan.bytes, lay.device, stream)
    base = buf.data_ptr() - plan.off_slots
    args = (table.ptr(first), count, lay.kv_stride, lay.page_stride, lay.page_bytes,
            lay.num_blocks, lay.block_size, row, base + plan.off_slots, base + plan.off_rows,
            plan.n_tokens, staging.data_ptr(), nbytes, lay.layer_bytes, layer0 + first)
    if rope:
        _, cos_sin, rot_dim, style, n_tables, n_groups, lg_d, ks_ptr = rope
        _lib.check("dsr_scatter_slots_rerotate", lib.dsr_scatter_slots_rerotate(
            *args, cos_sin.data_ptr(), base + plan.off_rope, n_tables,
            None if lg_d is None else lg_d.data_ptr(), n_groups, lay.head_dim, rot_dim,
            ROPE_STYLES[style], _DTYPE_CODES[lay.dtype], ks_ptr, stream))
    else:
        name = "dsr_gather_slots" if mode else "dsr_scatter_slots"
        _lib.check(name, getattr(lib, name)(*args, stream))
    return True


def gather_slots(table: LayerTable, slot_mapping, row_offsets, staging: torch.Tensor, *,
                 layer0: int = 0, layers: Optional[tuple[int, int]] = None) -> None:
    """Token-granular gather driven by vLLM's slot_mapping (-1 = padding):
    each valid token's K and V rows of every layer go to its record rows at
    ``row_offsets[t]`` (see :func:`token_row_offsets`)."""
    if _slots_host(table, slot_mapping, row_offsets, staging, layer0, layers, 1):
        return
    args, _tables = _slots_args(table, slot_mapping, row_offsets, staging, layer0, layers, True)
    rc = _lib.lib().dsr_gather_slots(*args, _stream_handle(table.layout.device))
    _lib.check("dsr_gather_slots", rc)


def _last_per_slot(sm: np.ndarray) -> np.ndarray:
    """slot_mapping with every entry but the last of a repeated slot turned
    into padding (-1): the reference's sequential copies leave the last
    one's bytes, while copies inside one launch would race."""
    valid = np.nonzero(sm >= 0)[0]
    dest = sm[valid]
    if np.unique(dest).size == dest.size:
        return sm
    _, last_rev = np.unique(dest[::-1], return_index=True)
    keep = np.zeros(valid.size, bool)
    keep[valid.size - 1 - last_rev] = True
    sm = sm.copy()
    sm[valid[~keep]] = -1
    return sm


def whole_pages(slot_mapping: np.ndarray, row_offsets: np.ndarray, block_size: int,
                row_bytes: int, rope_idx: Optional[np.ndarray] = None):
    """Splits the host tables of a token-form scatter into whole pages and
    the rest. The entries must be in slot order with no slot listed twice
    (padding, -1, anywhere). :func:`scatter_slots` has the library make the same
    split (dsr_plan_slots); this one is for callers whose tables stay resident.
    A block is whole when its block_size slots sit
    in consecutive entries, in order, with consecutive record rows
    (row_offsets stepping by row_bytes: the block's K rows form one record
    page, its V rows the page after) and, with rope_idx, one table index.

    Returns (page_ids, page_offsets, page_rope or None, rest): the whole
    blocks, the record offset of each one's first row (its slot record
    offset in the page form), their table indices, and a mask of the entries
    left for the token kernels."""
    sm = np.asarray(slot_mapping, np.int64)
    ro = np.asarray(row_offsets, np.int64)
    n, bs = sm.size, int(block_size)
    rest = np.ones(n, bool)
    empty = np.zeros(0, np.int64)
    if n < bs:
        return empty, empty, None if rope_idx is None else empty, rest
    step = np.zeros(n, bool)  # entry i continues entry i - 1 inside one record page
    step[1:] = (sm[1:] == sm[:-1] + 1) & (ro[1:] == ro[:-1] + row_bytes) & (sm[:-1] >= 0)
    ri = None
    if rope_idx is not None:
        ri = np.asarray(rope_idx, np.int64)
        step[1:] &= ri[1:] == ri[:-1]
    breaks = np.cumsum(~step)
    i = np.arange(n - bs + 1)
    start = (sm[i] >= 0) & (sm[i] % bs == 0) & (breaks[i + bs - 1] == breaks[i])
    starts = i[start]
    rest[(starts[:, None] + np.arange(bs)).ravel()] = False
    return (sm[starts] // bs, ro[starts], None if ri is None else ri[starts], rest)


def slot_order(slot_mapping, row_offsets, rope_idx=None):
    """Host tables in slot order, repeated slots padded but the last; None
    for device tables."""
    sm = _host_array(slot_mapping, np.int64)
    ro = _host_array(row_offsets, np.int64)
    ri = None if rope_idx is None else _host_array(rope_idx, np.int64)
    if sm is None or ro is None or (rope_idx is not None and ri is None) or not sm.size:
        return None
    if sm.shape != ro.shape or (ri is not None and ri.shape != sm.shape):
        raise ValueError("slot_mapping, row_offsets and rope_idx differ in length")
    order = np.argsort(sm, kind="stable")
    # within a run of equal slots the stable order keeps list order
    return _last_per_slot(sm[order]), ro[order], None if ri is None else ri[order]


def scatter_slots(table: LayerTable, slot_mapping, row_offsets, staging: torch.Tensor, *,
                  layer0: int = 0, layers: Optional[tuple[int, int]] = None) -> None:
    """Inverse of :func:`gather_slots`. Host tables are processed in
    destination-slot order (near-sequential writes), like :func:`scatter`,
    and blocks whose every slot is listed with consecutive record rows go
    as whole pages through the page scatter (dsr_plan_slots, as
    :func:`whole_pages`); the other
    tokens (the ragged edges of requests) go through the token kernel;
    whole pages that share records load through :class:`PreparedFanout`,
    as in :func:`scatter`. Device tables go to the token kernel as given."""
    if _slots_host(table, slot_mapping, row_offsets, staging, layer0, layers, 0):
        return
    host = slot_order(slot_mapping, row_offsets)
    if host is not None:
        slot_mapping, row_offsets, _ = host
    args, _tables = _slots_args(table, slot_mapping, row_offsets, staging, layer0, layers, False)
    rc = _lib.lib().dsr_scatter_slots(*args, _stream_handle(table.layout.device))
    _lib.check("dsr_scatter_slots", rc)


def scatter_slots_rerotate(table: LayerTable, slot_mapping, row_offsets,
                           staging: torch.Tensor, cos_sin: torch.Tensor, rope_idx, *,
                           rot_dim: Optional[int] = None, style: str = "neox",
                           k_scale: Optional[torch.Tensor] = None, layer0: int = 0,
                           layers: Optional[tuple[int, int]] = None,
                           layer_group=None) -> None:
    """:func:`scatter_slots` with each valid token's K rotated by
    ``cos_sin[rope_idx[t]]`` (-1 = copy), as :func:`scatter_rerotate` rotates
    a page row (same tables, scales and layer groups). Host tables are
    processed in destination-slot order, whole pages with one table index
    through :func:`scatter_rerotate` (the fan-out load where they share
    records)."""
    lay = table.layout
    rot_dim, n_tables, n_groups, lg_d, ks_ptr = _rope_args(
        lay, cos_sin, rope_idx, rot_dim, k_scale, layer0, layer_group)
    if _slots_host(table, slot_mapping, row_offsets, staging, layer0, layers, 0,
                   (_host_list(rope_idx), cos_sin, rot_dim, style, n_tables, n_groups, lg_d,
                    ks_ptr)):
        return
    host = slot_order(slot_mapping, row_offsets, rope_idx)
    if host is not None:
        slot_mapping, row_offsets, rope_idx = host
    args, _tables = _slots_args(table, slot_mapping, row_offsets, staging, layer0, layers, False)
    ridx_d = _as_device_table(rope_idx, torch.int32, lay.device, "rope_idx")
    if ridx_d.numel() != _tables[0].numel():
        raise ValueError("rope_idx and slot_mapping differ in length")
    rc = _lib.lib().dsr_scatter_slots_rerotate(
        *args, cos_sin.data_ptr(), ridx_d.data_ptr(), n_tables,
        None if lg_d is None else lg_d.data_ptr(), n_groups, lay.head_dim, rot_dim,
        ROPE_STYLES[style], _DTYPE_CODES[lay.dtype], ks_ptr, _stream_handle(lay.device))
    _lib.check("dsr_scatter_slots_rerotate", rc)


def token_row_offsets(req_tokens: Sequence[int], slot_bytes: int, block_size: int,
                      row_bytes: int, base: int = 0) -> np.ndarray:
    """Record offset of each token's K row for requests whose records are
    packed back to back (request r's slot i at base + (slots before r + i) *
    slot_bytes): token t of a request sits in its slot t // block_size at row
    t % block_size, the position dsr_gather puts it at."""
    out = []
    slot0 = 0
    for n in req_tokens:
        t = np.arange(int(n), dtype=np.int64)
        out.append(base + (slot0 + t // block_size) * slot_bytes + (t % block_size) * row_bytes)
        slot0 += -(-int(n) // block_size)
    return np.concatenate(out) if out else np.zeros(0, np.int64)


def slot_mapping_for(block_tables: Sequence[Sequence[int]], req_tokens: Sequence[int],
                     block_size: int) -> np.ndarray:
    """vLLM's slot_mapping of the requests' tokens:
    slot = block_ids[t // block_size] * block_size + t % block_size."""
    out = []
    for blocks, n in zip(block_tables, req_tokens):
        t = np.arange(int(n), dtype=np.int64)
        b = np.asarray(blocks, dtype=np.int64)
        out.append(b[t // block_size] * block_size + t % block_size)
    return np.concatenate(out) if out else np.zeros(0, np.int64)


def slot_offsets_for(num_pages: Sequence[int], slot_bytes: int, base: int = 0) -> np.ndarray:
    """Record offsets for requests packed back to back in one staging buffer:
    request r's slot i lives at ``base + (pages before r + i) * slot_bytes``."""
    total = int(sum(num_pages))
    return base + np.arange(total, dtype=np.int64) * slot_bytes


def pages_for_tokens(token_count: int, block_size: int) -> int:
    """ceil(tokens / block_size): pages holding token_count tokens
    (daser/connector/daser_connector.py:280, :292)."""
    return math.ceil(token_count / block_size)
