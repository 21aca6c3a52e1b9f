"""The flat page copies (1 KiB pieces of a unit, one per wave) against plain
byte indexing of the caches: page sizes around a piece and around 8 pieces,
every store policy and launch class, launches cut inside a unit, workgroups
dealt in chunks, entries out of bounds."""

import numpy as np
import pytest
import torch

from daser_amd import ops

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
                                                  (0, 8, 24)])
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
