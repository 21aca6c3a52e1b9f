"""The flat page copies (1 KiB pieces of a unit, one per wave) against plain
byte indexing of the caches: page sizes around a piece and around 8 pieces,
every store policy and launch class, launches cut inside a unit, workgroups
dealt in chunks, entries out of bounds."""

import numpy as np
import pytest
import torch

from daser_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _setup(gpu, n_pages, layers, block, heads, dim, layout, seed, slack=3):
    g = torch.Generator(device=gpu).manual_seed(seed)
    nb = n_pages + slack
    inner = (heads, block, dim) if layout == "hnd" else (block, heads, dim)
    whole = torch.randint(-2**15, 2**15, (layers, 2, nb, *inner), generator=g, device=gpu,
                          dtype=torch.int16).view(torch.bfloat16)
    views = [w.transpose(2, 3) if layout == "hnd" else w for w in whole.unbind(0)]
    rng = np.random.default_rng(seed)
    ids = rng.permutation(nb)[:n_pages].astype(np.int64)
    return whole, views, ids, rng


def _records(views, ids):
    """Records in page order: (page, layer, K then V), index order."""
    sel = [v[:, torch.from_numpy(ids).to(v.device)] for v in views]
    return torch.stack(sel).transpose(0, 2).transpose(1, 2).contiguous()  # [p, l, 2, bs, H, D]


@pytest.mark.parametrize("block,heads,dim,layout", [
    (1, 1, 8, "nhd"), (3, 1, 40, "nhd"), (16, 1, 32, "nhd"), (16, 1, 40, "nhd"),
    (16, 2, 128, "nhd"), (16, 5, 96, "nhd"), (16, 16, 128, "nhd"),
    (1, 1, 8, "hnd"), (5, 3, 24, "hnd"), (16, 4, 128, "hnd")])
@pytest.mark.parametrize("policy,pieces,max_wg", [(0, 0, 0), (1, 8, 0), (1, 1, 16), (3, 0, 16),
                                                  (0, 8, 24), (3, 8, 0)])
def test_flat_copies(gpu, tuning, block, heads, dim, layout, policy, pieces, max_wg):
    print(f"case: flat bs{block} H{heads} D{dim} {layout} {policy} {pieces} {max_wg}", flush=True)
    tuning("scatter_kernel", policy)
    tuning("gather_split", pieces)
    tuning("max_wg_per_launch", max_wg)
    n, layers = 23, 3
    whole, views, ids, rng = _setup(gpu, n, layers, block, heads, dim, layout, seed=dim + block)
    table = ops.LayerTable(views)
    slot = table.layout.slot_bytes
    place = rng.permutation(n)
    offs = place.astype(np.int64) * slot
    want = torch.zeros(n * slot, dtype=torch.uint8, device=gpu)
    want.view(n, slot)[torch.from_numpy(place).to(gpu)] = \
        _records(views, ids).view(n, -1).view(torch.uint8)
    staging = torch.zeros_like(want)
    # device tables with two entries out of bounds: skipped
    d_ids = torch.from_numpy(np.append(ids, [-1, table.layout.num_blocks]).astype(np.int32))
    d_offs = torch.from_numpy(np.append(offs, [0, slot]))
    ops.gather(table, d_ids.to(gpu), d_offs.to(gpu), staging)
    torch.cuda.synchronize()
    assert torch.equal(staging, want)
    back = torch.zeros_like(whole)
    bviews = [w.transpose(2, 3) if layout == "hnd" else w for w in back.unbind(0)]
    d_offs = torch.from_numpy(np.append(offs, [-n * slot, n * slot]))
    d_ids = torch.from_numpy(np.append(ids, [5, 6]).astype(np.int32))
    ops.scatter(ops.LayerTable(bviews), d_ids.to(gpu), d_offs.to(gpu), staging)
    torch.cuda.synchronize()
    sel = torch.from_numpy(ids).to(gpu)
    ref = torch.zeros_like(whole)
    ref[:, :, sel] = whole[:, :, sel]
    assert torch.equal(back.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("n_pages,layers", [(1, 1), (20, 8), (24, 8), (32, 8), (33, 8), (257, 8),
                                            (521, 9)])
def test_flat_copy_launch_classes(gpu, n_pages, layers):
    """32 KiB pages at sizes on both sides of every class limit (20, 32
    and 200 MiB moved; from there workgroups are dealt in chunks, the last of
    them partial), single layers and the whole table."""
    print(f"case: flat classes {n_pages}x{layers}", flush=True)
    whole, views, ids, rng = _setup(gpu, n_pages, layers, 16, 8, 128, "nhd", seed=n_pages)
    table = ops.LayerTable(views)
    slot = table.layout.slot_bytes
    offs = np.arange(n_pages, dtype=np.int64) * slot
    want = _records(views, ids).view(-1).view(torch.uint8)
    staging = torch.zeros_like(want)
    ops.gather(table, ids, offs, staging)
    single = torch.zeros_like(want)
    for l in range(layers):
        ops.gather(table, ids, offs, single, layers=(l, 1))
    back = torch.zeros_like(whole)
    ops.scatter(ops.LayerTable(list(back.unbind(0))), ids, offs, staging)
    torch.cuda.synchronize()
    assert torch.equal(staging, want) and torch.equal(single, want)
    sel = torch.from_numpy(ids).to(gpu)
    assert torch.equal(back[:, :, sel].view(torch.int16), whole[:, :, sel].view(torch.int16))


@pytest.mark.parametrize("block,heads,dim,layout,rot,style", [
    (16, 8, 128, "nhd", 128, "neox"), (16, 1, 128, "nhd", 64, "gptj"), (1, 1, 64, "nhd", 64, "neox"),
    (16, 3, 96, "nhd", 96, "neox"), (5, 2, 80, "nhd", 80, "neox"), (16, 2, 192, "nhd", 192, "neox"),
    (16, 2, 256, "nhd", 256, "neox"), (2, 1, 1024, "nhd", 64, "neox"), (7, 3, 64, "hnd", 32, "neox"),
    (16, 4, 128, "kx", 128, "neox"), (16, 2, 64, "kx", 64, "gptj")])
@pytest.mark.parametrize("dt", ["bf16", "fp16", "e4m3", "e5m2"])
@pytest.mark.parametrize("stores,max_wg", [(0, 0), (3, 24)])
def test_flat_rerotate(gpu, tuning, block, heads, dim, layout, rot, style, dt, stores, max_wg):
    """Rotated K within one rounding of float64 from the stored bits (the
    8-bit formats with their layer's scale, one of them zero: NaN codes as by
    multiplication), V and un-rotated pages unchanged; launches cut inside a
    unit, both store policies."""
    print(f"case: flat rotate bs{block} H{heads} D{dim} {layout} {rot} {style} {dt} {stores}",
          flush=True)
    tuning("scatter_kernel", stores)
    tuning("max_wg_per_launch", max_wg)
    dtype = {"bf16": torch.bfloat16, "fp16": torch.float16, "e4m3": torch.float8_e4m3fn,
             "e5m2": torch.float8_e5m2}[dt]
    fp8 = dt in ("e4m3", "e5m2")
    esize = 1 if fp8 else 2
    if layout == "hnd" and rot // 2 * esize % 16:
        pytest.skip("HND pages take whole-vector rotary widths")
    x_el = 16 // esize
    if layout == "kx" and (rot // 2 % x_el if style == "neox" else rot % x_el):
        pytest.skip("split-x pages take whole-vector rotary widths")
    n, layers = 9, 3
    g = torch.Generator(device=gpu).manual_seed(dim + rot)
    rng = np.random.default_rng(dim)
    logical = torch.randn((layers, n, 2, block, heads, dim), generator=g, device=gpu)
    scales = torch.tensor([0.03, 1.7, 0.0], device=gpu)
    stored = (logical * 20).to(dtype) if fp8 else logical.to(dtype)  # record order, token-major
    recs = stored.clone()
    if layout == "kx":  # records hold K split-x; V as it is
        k = stored[:, :, 0].reshape(layers, n, block, heads, dim // x_el, x_el)
        recs[:, :, 0] = k.permute(0, 1, 3, 4, 2, 5).reshape(layers, n, block, heads, dim)
    staging = recs.transpose(0, 1).contiguous().view(-1).view(torch.uint8)
    nb = n + 4
    inner = {"nhd": (block, heads, dim), "hnd": (heads, block, dim),
             "kx": (block * heads * dim,)}[layout]
    whole = torch.zeros((layers, 2, nb, *inner), dtype=dtype, device=gpu)
    views = [w.transpose(2, 3) if layout == "hnd" else w for w in whole.unbind(0)]
    geo = dict(block_size=block, head_dim=dim) if layout == "kx" else {}
    table = ops.LayerTable(views, **geo)
    ids = rng.permutation(nb)[:n].astype(np.int64)
    ridx = (np.arange(n) % 3 - 1).astype(np.int64)  # every third page keeps its K
    ang = torch.rand((2, rot // 2), generator=g, device=gpu, dtype=torch.float64) * 6.28
    tabs = torch.stack([ang.cos(), ang.sin()], -1).float()
    ops.scatter_rerotate(table, ids, np.arange(n, dtype=np.int64) * table.layout.slot_bytes,
                         staging, tabs, ridx, rot_dim=rot, style=style,
                         k_scale=scales if fp8 else None)
    torch.cuda.synchronize()
    got = whole[:, :, torch.from_numpy(ids).to(gpu)].transpose(1, 2)  # [l, p, 2, ...]
    if layout == "hnd":
        got = got.transpose(3, 4)
    elif layout == "kx":
        kk = got[:, :, 0].reshape(layers, n, heads, dim // x_el, block, x_el)
        kk = kk.permute(0, 1, 4, 2, 3, 5).reshape(layers, n, block, heads, dim)
        got = torch.stack([kk.view(torch.uint8), got[:, :, 1].reshape(kk.shape).view(torch.uint8)],
                          2).view(dtype)
    else:
        got = got.reshape(stored.shape)
    as_bytes = lambda t: t.contiguous().view(torch.uint8)  # noqa: E731
    assert torch.equal(as_bytes(got[:, :, 1]), as_bytes(stored[:, :, 1]))
    keep = torch.from_numpy(ridx < 0).to(gpu)
    assert torch.equal(as_bytes(got[:, keep]), as_bytes(stored[:, keep]))
    moved = torch.from_numpy(np.nonzero(ridx >= 0)[0]).to(gpu)
    t = tabs.double()[torch.from_numpy(ridx[ridx >= 0]).to(gpu)][None, :, None, None]
    x = stored[:, moved, 0].double()
    ref = x.clone()
    lo, hi = (x[..., :rot // 2], x[..., rot // 2:rot]) if style == "neox" else \
        (x[..., 0:rot:2], x[..., 1:rot:2])
    a, b = lo * t[..., 0] - hi * t[..., 1], hi * t[..., 0] + lo * t[..., 1]
    if style == "neox":
        ref[..., :rot // 2], ref[..., rot // 2:rot] = a, b
    else:
        ref[..., 0:rot:2], ref[..., 1:rot:2] = a, b
    top = {"e4m3": 448.0, "e5m2": 57344.0}.get(dt, float("inf"))
    ref = ref.clamp(-top, top)
    k = got[:, moved, 0].double()
    if fp8:  # a zero scale: 0 * inf in every rotated value
        assert torch.isnan(k[2][..., :rot]).all() and torch.equal(k[2][..., rot:], x[2][..., rot:])
        k, ref, x = k[:2], ref[:2], x[:2]
    # half a unit in the last place of the result, plus fp32's share of the inputs
    mant, least = {"bf16": (8, 2.0 ** -133), "fp16": (11, 2.0 ** -24), "e4m3": (4, 2.0 ** -9),
                   "e5m2": (3, 2.0 ** -16)}[dt]
    ulp = torch.maximum(torch.exp2(torch.floor(torch.log2(ref.abs().clamp_min(1e-300))) + 1 - mant),
                        torch.full_like(ref, least))
    bound = 0.5 * ulp + x.abs().amax(-1, keepdim=True) * 2.0 ** -21
    assert ((k - ref).abs() <= bound).all()


@pytest.mark.parametrize("heads,dim,dt", [(1, 64, "e4m3"), (1, 128, "bf16"), (3, 32, "bf16"),
                                          (5, 128, "fp16"), (4, 128, "bf16"), (9, 128, "bf16"),
                                          (2, 256, "e5m2")])
@pytest.mark.parametrize("block,max_wg", [(16, 0), (6, 24)])
def test_flat_slots(gpu, tuning, heads, dim, dt, block, max_wg):
    """Token form on device tables, rows of 4 to 144 vectors: padding, slots
    and records out of range, tokens of one wave with one table, several
    and none; gathers and copies byte for byte, rotated tokens bit for bit as
    the page form rotates them."""
    print(f"case: flat slots H{heads} D{dim} {dt} bs{block} {max_wg}", flush=True)
    tuning("max_wg_per_launch", max_wg)
    dtype = {"bf16": torch.bfloat16, "fp16": torch.float16, "e4m3": torch.float8_e4m3fn,
             "e5m2": torch.float8_e5m2}[dt]
    layers, n = 2, 7
    nb = n + 2
    g = torch.Generator(device=gpu).manual_seed(dim + heads)
    rng = np.random.default_rng(heads)
    whole = torch.randn((layers, 2, nb, block, heads, dim), generator=g, device=gpu).to(dtype)
    table = ops.LayerTable(list(whole.unbind(0)))
    lay = table.layout
    row = heads * dim * lay.elem_bytes
    ids = rng.permutation(nb)[:n]
    tokens = n * block - 3
    slots = ops.slot_mapping_for([ids], [tokens], block)
    rows = ops.token_row_offsets([tokens], lay.slot_bytes, block, row)
    drop = rng.random(tokens) < 0.2
    slots[drop] = -1
    slots[1], rows[2] = nb * block, n * lay.slot_bytes  # out of range
    slots_d, rows_d = torch.from_numpy(slots).to(gpu), torch.from_numpy(rows).to(gpu)
    ok = np.nonzero(~drop)[0]
    ok = ok[(ok != 1) & (ok != 2)]
    want = torch.zeros((n, layers, 2, block, heads, dim), dtype=dtype, device=gpu)
    for t in ok:
        want[t // block, :, :, t % block] = whole[:, :, int(ids[t // block]), t % block]
    staging = torch.zeros(n * lay.slot_bytes, dtype=torch.uint8, device=gpu)
    ops.gather_slots(table, slots_d, rows_d, staging)
    torch.cuda.synchronize()
    assert torch.equal(staging, want.view(-1).view(torch.uint8))
    back = torch.zeros_like(whole)
    ops.scatter_slots(ops.LayerTable(list(back.unbind(0))), slots_d, rows_d, staging)
    ref = torch.zeros_like(whole)
    for t in ok:
        ref[:, :, int(ids[t // block]), t % block] = whole[:, :, int(ids[t // block]), t % block]
    torch.cuda.synchronize()
    assert torch.equal(back.view(torch.uint8), ref.view(torch.uint8))
    if (dim * lay.elem_bytes // 16) & (dim * lay.elem_bytes // 16 - 1) or dim // 2 % (16 // lay.elem_bytes):
        return
    # rotated: runs of tokens with one table, then a table per token
    ang = torch.rand((3, dim // 2), generator=g, device=gpu, dtype=torch.float64) * 6.28
    tabs = torch.stack([ang.cos(), ang.sin()], -1).float()
    scales = torch.tensor([0.5, 3.0], device=gpu) if lay.elem_bytes == 1 else None
    ridx = np.where(np.arange(tokens) < 3 * block, 1, np.arange(tokens) % 4 - 1)
    rot = torch.zeros_like(whole)
    ops.scatter_slots_rerotate(ops.LayerTable(list(rot.unbind(0))), slots_d, rows_d, staging, tabs,
                               torch.from_numpy(ridx.astype(np.int32)).to(gpu), k_scale=scales)
    exp = torch.zeros_like(whole)
    offs = np.arange(n, dtype=np.int64) * lay.slot_bytes
    for r in (-1, 0, 1, 2):  # the page form with one table for every page
        tmp = torch.zeros_like(whole)
        ops.scatter_rerotate(ops.LayerTable(list(tmp.unbind(0))), ids, offs, staging, tabs,
                             np.full(n, r), k_scale=scales)
        for t in ok[ridx[ok] == r]:
            exp[:, :, int(ids[t // block]), t % block] = tmp[:, :, int(ids[t // block]), t % block]
    torch.cuda.synchronize()
    assert torch.equal(rot.view(torch.uint8), exp.view(torch.uint8))


@pytest.mark.parametrize("where", ["host", "device"])
def test_padding_alone_is_checked(gpu, where):
    """A token load whose slots are all padding is refused where its geometry is
    (96-dim neox heads), and else moves nothing."""
    for dim in (96, 128):
        print(f"case: padding alone {where} D{dim}", flush=True)
        whole, views, _, _ = _setup(gpu, 2, 2, 8, 2, dim, "nhd", seed=1)
        before = whole.clone()
        table = ops.LayerTable(views)
        staging = torch.ones(table.layout.slot_bytes, dtype=torch.uint8, device=gpu)
        dev = gpu if where == "device" else "cpu"
        slots = torch.full((5,), -1, dtype=torch.int64, device=dev)
        rows = torch.arange(5, dtype=torch.int64, device=dev) * dim * 4
        ridx = torch.zeros(5, dtype=torch.int32, device=dev)
        tabs = torch.ones((1, dim // 2, 2), device=gpu)
        if dim == 96:
            with pytest.raises(_lib.DaserKVError):
                ops.scatter_slots_rerotate(table, slots, rows, staging, tabs, ridx)
        else:
            ops.scatter_slots_rerotate(table, slots, rows, staging, tabs, ridx)
        ops.scatter_slots(table, slots, rows, staging)
        ops.gather_slots(table, slots, rows, staging)
        torch.cuda.synchronize()
        assert torch.equal(whole.view(torch.int16), before.view(torch.int16))
        assert (staging == 1).all()


@pytest.mark.parametrize("heads,dim", [(5, 104), (8, 128), (16, 128)])
def test_huge_slot_gather(gpu, heads, dim):
    """The token gather's launch above 16 GiB moved, rows of 65 vectors, of 2 KiB
    (in units of 2 tokens up to there) and of 4 KiB: the records of the page form, tokens that are left
    out untouched."""
    print(f"case: huge slot gather H{heads} D{dim}", flush=True)
    layers, block, row = 64, 16, heads * dim * 2
    n = (16 << 30) // (4 * layers * block * row) + 2
    g = torch.Generator(device=gpu).manual_seed(dim)
    rng = np.random.default_rng(dim)
    whole = torch.empty((layers, 2, n, block, heads, dim), dtype=torch.bfloat16, device=gpu)
    whole.view(-1).view(torch.int64).random_(generator=g)
    table = ops.LayerTable(list(whole.unbind(0)))
    lay = table.layout
    ids = rng.permutation(n)
    tokens = n * block - 1  # short of the last page by a token
    slots = ops.slot_mapping_for([ids], [tokens], block)
    rows = ops.token_row_offsets([tokens], lay.slot_bytes, block, row)
    assert 4 * tokens * row * layers > 16 << 30
    want, got = (torch.zeros(n * lay.slot_bytes, dtype=torch.uint8, device=gpu) for _ in range(2))
    ops.gather(table, ids, np.arange(n, dtype=np.int64) * lay.slot_bytes, want)
    want.view(n, layers, 2, block, row)[-1, :, :, -1] = 0
    ops.gather_slots(table, torch.from_numpy(slots).to(gpu), torch.from_numpy(rows).to(gpu), got)
    torch.cuda.synchronize()
    assert torch.equal(got, want) and got.any()


@pytest.mark.parametrize("n_src,n_dst,heads,dim,dt,layout,rot", [
    (3, 300, 1, 64, "bf16", "nhd", 64), (511, 1100, 1, 128, "e4m3", "nhd", 128),
    (512, 1100, 1, 128, "bf16", "nhd", 64), (600, 1300, 2, 64, "e5m2", "hnd", 64),
    (5, 200, 2, 512, "fp16", "nhd", 512)])
def test_flat_fanout(gpu, n_src, n_dst, heads, dim, dt, layout, rot):
    """Both unit orders of the fan-out (few and many sources), more
    destinations of a source than a wave holds at once, tables of up to 256
    pairs: bit for bit the per-page load, K rotated or not."""
    print(f"case: flat fanout {n_src}->{n_dst} H{heads} D{dim} {dt} {layout}", flush=True)
    dtype = {"bf16": torch.bfloat16, "fp16": torch.float16, "e4m3": torch.float8_e4m3fn,
             "e5m2": torch.float8_e5m2}[dt]
    layers, block, nb = 2, 4, n_dst + 9
    g = torch.Generator(device=gpu).manual_seed(n_src)
    rng = np.random.default_rng(n_src)
    recs = torch.randn((n_src, layers, 2, block, heads, dim), generator=g, device=gpu).to(dtype)
    staging = recs.view(-1).view(torch.uint8)
    inner = (heads, block, dim) if layout == "hnd" else (block, heads, dim)
    caches = [torch.zeros((layers, 2, nb, *inner), dtype=dtype, device=gpu) for _ in range(2)]
    tables = [ops.LayerTable([w.transpose(2, 3) if layout == "hnd" else w for w in c.unbind(0)])
              for c in caches]
    slot = tables[0].layout.slot_bytes
    ids = rng.permutation(nb)[:n_dst].astype(np.int64)
    src = np.concatenate([np.arange(n_src), rng.integers(0, n_src, n_dst - n_src)])
    offs = rng.permutation(src).astype(np.int64) * slot
    ang = torch.rand((5, rot // 2), generator=g, device=gpu, dtype=torch.float64) * 6.28
    tabs = torch.stack([ang.cos(), ang.sin()], -1).float()
    ridx = rng.integers(-1, 5, n_dst)
    scales = torch.tensor([0.02, 1.5], device=gpu) if dt in ("e4m3", "e5m2") else None
    assert ops.fanout_supported(tables[0].layout, rot)
    ops.PreparedFanout(tables[0], ids, offs, staging,
                       rope=(ridx, tabs, rot, "neox", scales, None))()
    ops.scatter_rerotate(tables[1], ids, offs, staging, tabs, ridx, rot_dim=rot, k_scale=scales,
                         shared_records=False)
    torch.cuda.synchronize()
    assert torch.equal(caches[0].view(torch.uint8), caches[1].view(torch.uint8))
    assert caches[0].view(torch.uint8).any()
    for c in caches:
        c.zero_()
    ops.PreparedFanout(tables[0], ids, offs, staging)()
    ops.scatter(tables[1], ids, offs, staging, shared_records=False)
    torch.cuda.synchronize()
    assert torch.equal(caches[0].view(torch.uint8), caches[1].view(torch.uint8))


@pytest.mark.parametrize("counts,heads,dim,layout,max_wg", [
    ((1000,), 1, 64, "nhd", 0), ((700, 1, 3, 0, 96), 2, 64, "nhd", 0),
    ((700, 1, 3, 0, 96), 2, 64, "hnd", 16), ((64,), 8, 128, "kx", 0),
    ((130, 62), 8, 128, "nhd", 0), ((7, 9), 8, 128, "nhd", 24), ((65, 66, 64), 5, 128, "nhd", 0)])
def test_fanout_shares_of_destinations(gpu, tuning, counts, heads, dim, layout, max_wg):
    """Few records of many destinations: each record's are dealt to several waves,
    uneven counts (records of none among them): bit for bit the per-page load."""
    print(f"case: fanout shares {counts} H{heads} D{dim} {layout} {max_wg}", flush=True)
    tuning("max_wg_per_launch", max_wg)
    layers, block, n = 2, 16, sum(counts)
    g = torch.Generator(device=gpu).manual_seed(n)
    rng = np.random.default_rng(n)
    inner = {"nhd": (block, heads, dim), "hnd": (heads, block, dim),
             "kx": (block * heads * dim,)}[layout]
    geo = dict(block_size=block, head_dim=dim) if layout == "kx" else {}
    caches = [torch.zeros((layers, 2, n + 3, *inner), dtype=torch.bfloat16, device=gpu)
              for _ in range(2)]
    tables = [ops.LayerTable([w.transpose(2, 3) if layout == "hnd" else w for w in c.unbind(0)],
                             **geo) for c in caches]
    slot = tables[0].layout.slot_bytes
    staging = torch.randn(len(counts) * slot // 2, generator=g, device=gpu).to(torch.bfloat16) \
        .view(torch.uint8)
    ids = rng.permutation(n + 3)[:n].astype(np.int64)
    offs = np.repeat(np.arange(len(counts), dtype=np.int64), counts) * slot
    ang = torch.rand((5, dim // 2), generator=g, device=gpu, dtype=torch.float64) * 6.28
    tabs = torch.stack([ang.cos(), ang.sin()], -1).float()
    ridx = rng.integers(-1, 5, n)
    ops.PreparedFanout(tables[0], ids, offs, staging, rope=(ridx, tabs, dim, "neox", None, None))()
    ops.scatter_rerotate(tables[1], ids, offs, staging, tabs, ridx, shared_records=False)
    torch.cuda.synchronize()
    assert torch.equal(*(c.view(torch.int16) for c in caches))
    assert caches[0].view(torch.int16).any()


@pytest.mark.parametrize("n_src,n_dst", [(300, 3800), (1000, 3100)])
def test_large_fanout(gpu, n_src, n_dst):
    """The fan-out's launch above 1 GiB, both unit orders: what the per-page load
    writes, K rotated or not."""
    print(f"case: large fanout {n_src}->{n_dst}", flush=True)
    layers, nb = 4, n_dst + 9
    g = torch.Generator(device=gpu).manual_seed(n_src)
    rng = np.random.default_rng(n_src)
    staging = torch.randn((n_src, layers, 2, 16, 8, 128), generator=g, device=gpu) \
        .to(torch.bfloat16).view(-1).view(torch.uint8)
    caches = [torch.zeros((layers, 2, nb, 16, 8, 128), dtype=torch.bfloat16, device=gpu)
              for _ in range(2)]
    tables = [ops.LayerTable(list(c.unbind(0))) for c in caches]
    slot = tables[0].layout.slot_bytes
    assert (n_src + n_dst) * slot > 1 << 30
    ids = rng.permutation(nb)[:n_dst].astype(np.int64)
    src = np.concatenate([np.arange(n_src), rng.integers(0, n_src, n_dst - n_src)])
    offs = rng.permutation(src).astype(np.int64) * slot
    ang = torch.rand((5, 64), generator=g, device=gpu, dtype=torch.float64) * 6.28
    tabs = torch.stack([ang.cos(), ang.sin()], -1).float()
    ridx = rng.integers(-1, 5, n_dst)
    ops.PreparedFanout(tables[0], ids, offs, staging, rope=(ridx, tabs, 128, "neox", None, None))()
    ops.scatter_rerotate(tables[1], ids, offs, staging, tabs, ridx, shared_records=False)
    torch.cuda.synchronize()
    assert torch.equal(*(c.view(torch.int16) for c in caches))
    assert caches[0].view(torch.int16).any()
    ops.PreparedFanout(tables[0], ids, offs, staging)()
    ops.scatter(tables[1], ids, offs, staging, shared_records=False)
    torch.cuda.synchronize()
    assert torch.equal(*(c.view(torch.int16) for c in caches))


@pytest.mark.parametrize("n,rot", [(1, 128), (7, 128), (8, 128), (60, 20), (1024, 128)])
def test_delta_tables_on_the_device(gpu, n, rot):
    """The device's float64 tables (more than a kernel's arguments hold) are the
    host's within one float32 unit in the last place."""
    from daser_amd import position

    print(f"case: delta tables {n} x {rot}", flush=True)
    rng = np.random.default_rng(n)
    deltas = rng.integers(-32768, 32768, n).tolist()
    host = position.delta_tables(deltas, rot, 500000.0)
    dev = position.delta_tables(deltas, rot, 500000.0, device=gpu)
    torch.cuda.synchronize()
    assert dev.shape == host.shape and dev.dtype == torch.float32
    diff = (dev.cpu().double() - host.double()).abs()
    assert (diff <= host.double().abs() * 2.0 ** -23 + 2.0 ** -60).all()
    # float64 sine and cosine of the same product, rounded once: nearly all the same bits
    assert (diff == 0).double().mean() > 0.999


@pytest.mark.parametrize("save_stream", ["current", "side"])
def test_saves_from_another_stream_wait_for_the_tables(gpu, tmp_path, save_stream):
    """The page tables of a step are uploaded behind the stream's earlier work
    (here a delay); layers saved from another stream still read whole tables."""
    from daser_amd.connector import ReqStoreSpec
    from daser_amd.data_plane import KVDataPlane, plan_store

    print(f"case: saves on another stream, {save_stream}", flush=True)
    whole, views, ids, _ = _setup(gpu, 40, 3, 16, 2, 64, "nhd", 5)
    plane = KVDataPlane(str(tmp_path / "s"), save_stream=save_stream, io_backend="python")
    slot = plane.register({f"model.layers.{i}.self_attn.attn": v for i, v in enumerate(views)})
    plan = plan_store({"r": ReqStoreSpec("k", 0, ids.size, ids.tolist(), 0, 16 * ids.size)}, slot)
    want = _records(views, ids)
    torch.cuda.synchronize()
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(first):
        torch.cuda._sleep(20_000_000)
        arena = plane.new_store_arena(plan)
    with torch.cuda.stream(second):
        for name in plane.layer_idx:
            plane.save_layer(name, plan, arena)
    torch.cuda.synchronize()
    assert torch.equal(arena.view(torch.int16), want.view(torch.int16).flatten())
    plane.close()


@pytest.mark.parametrize("heads,dim,skipped", [(1, 8, True), (1, 16, True), (1, 32, True),
                                               (1, 64, True), (3, 8, False), (1, 128, False),
                                               (8, 128, False)])
@pytest.mark.parametrize("load", [False, True])
def test_negative_row_offsets(gpu, heads, dim, skipped, load):
    """Device tables with row offsets below the staging buffer. Power-of-two
    rows of up to 128 bytes: the token is skipped in every layer; others: in the
    layers where its row lies outside."""
    print(f"case: negative rows H{heads} D{dim} load {load}", flush=True)
    layers, block, n = 3, 4, 6
    whole, views, _, _ = _setup(gpu, n, layers, block, heads, dim, "nhd", seed=dim)
    table = ops.LayerTable(views)
    lay, row = table.layout, heads * dim * 2
    slots = np.arange(6, dtype=np.int64)
    rows = lay.slot_bytes + np.arange(6) * row
    rows[1], rows[4] = -16, -16 - 2 * row  # in layers 1 and 2: the first record's part
    rows[5] = lay.slot_bytes + row
    g = torch.Generator(device=gpu).manual_seed(3)
    staging = torch.randint(0, 256, (2 * lay.slot_bytes,), generator=g, device=gpu,
                            dtype=torch.uint8)
    cells = whole.view(torch.uint8).view(layers, 2, -1, row)  # by slot
    want_s, want_c = staging.clone(), cells.clone()
    for t, (s, r) in enumerate(zip(slots, rows)):
        for layer in range(layers):
            off = int(r) + layer * lay.layer_bytes
            if off < 0 or (r < 0 and skipped):
                continue
            for half in range(2):
                at = slice(off + half * lay.page_bytes, off + half * lay.page_bytes + row)
                if load:
                    want_c[layer, half, s] = staging[at]
                else:
                    want_s[at] = cells[layer, half, s]
    fn = ops.scatter_slots if load else ops.gather_slots
    fn(table, torch.from_numpy(slots).to(gpu), torch.from_numpy(rows).to(gpu), staging)
    torch.cuda.synchronize()
    assert torch.equal(staging, want_s)
    assert torch.equal(whole.view(torch.uint8).view(layers, 2, -1, row), want_c)


@pytest.mark.parametrize("block,heads,dim,layout", [
    (1, 1, 8, "nhd"), (16, 1, 64, "nhd"), (16, 5, 128, "nhd"), (16, 8, 64, "kx"),
    (16, 4, 128, "hnd")])
@pytest.mark.parametrize("n,max_wg", [(1, 0), (7, 0), (40, 0), (40, 24), (333, 0)])
def test_shared_records_order(gpu, tuning, block, heads, dim, layout, n, max_wg):
    """The launch for shared records (each XCD one eighth: grids of fewer than 8
    workgroups, of no multiple of 8, cut launches) writes what the plain one does."""
    print(f"case: shared order bs{block} H{heads} D{dim} {layout} {n} {max_wg}", flush=True)
    tuning("max_wg_per_launch", max_wg)
    layers = 3
    g = torch.Generator(device=gpu).manual_seed(n)
    inner = {"nhd": (block, heads, dim), "hnd": (heads, block, dim),
             "kx": (block * heads * dim,)}[layout]
    geo = dict(block_size=block, head_dim=dim) if layout == "kx" else {}
    outs = [torch.zeros((layers, 2, n + 2, *inner), dtype=torch.bfloat16, device=gpu)
            for _ in range(2)]
    views = [[w.transpose(2, 3) if layout == "hnd" else w for w in o.unbind(0)] for o in outs]
    tables = [ops.LayerTable(v, **geo) for v in views]
    slot = tables[0].layout.slot_bytes
    n_rec = max(1, n // 3)
    staging = torch.randn(n_rec * slot // 2, generator=g, device=gpu).to(torch.bfloat16) \
        .view(torch.uint8)
    rng = np.random.default_rng(n)
    ids = torch.from_numpy(np.sort(rng.permutation(n + 2)[:n]).astype(np.int32)).to(gpu)
    offs = torch.from_numpy(rng.integers(0, n_rec, n) * slot).to(gpu)
    ridx = torch.from_numpy((np.arange(n) % 3 - 1).astype(np.int32)).to(gpu)
    ang = torch.rand((2, dim // 2), generator=g, device=gpu) * 6.28
    tabs = torch.stack([ang.cos(), ang.sin()], -1)
    for rotate in (False, True):
        for table, shared in zip(tables, (False, True)):
            if rotate and dim >= 16:
                ops.scatter_rerotate(table, ids, offs, staging, tabs, ridx, shared_records=shared)
            else:
                ops.scatter(table, ids, offs, staging, shared_records=shared)
        torch.cuda.synchronize()
        assert torch.equal(*(o.view(torch.int16) for o in outs))
        assert outs[0].view(torch.int16).any()
