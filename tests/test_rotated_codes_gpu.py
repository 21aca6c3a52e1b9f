"""Rotated K, code for code, in every kernel that rotates: x * cos + (partner *
sin), the second product rounded to fp32 and the sum fused, then one rounding to
the cache's type. 8-bit values are multiplied by their layer's scale before and
by its fp32 inverse after (which decides ties unless the scale is a power of
two); fp16 sums are rounded to fp16 at once, except in the kernel of partial
widths, which works element by element in fp32."""

import numpy as np
import pytest
import torch

from daser_amd import ops
from tests.helpers import TORCH_DT

pytestmark = pytest.mark.gpu
TOP = {"e4m3": 448.0, "e5m2": 57344.0}
SCALES = [0.0113, 0.0137, 1.7, 0.5]  # the last one is exact


def _codes(stored, tabs, rot, style, dt, whole_vectors):
    """The bytes of stored [layers, ..., D] rotated by one table, in numpy."""
    x = stored.cpu().float().numpy()
    fp8 = dt in TOP
    scale = np.asarray(SCALES if fp8 else [1.0] * len(SCALES), np.float32)
    scale = scale.reshape(-1, *[1] * (x.ndim - 1))
    c, s = tabs[:, 0].cpu().numpy(), tabs[:, 1].cpu().numpy()
    xs = x * scale
    half = rot // 2
    lo, hi = (xs[..., :half], xs[..., half:rot]) if style == "neox" else \
        (xs[..., 0:rot:2], xs[..., 1:rot:2])
    once = dt == "fp16" and whole_vectors

    def fused(a, b, t):  # a product of two fp32 values is exact in float64
        y = a.astype(np.float64) * b.astype(np.float64) + t.astype(np.float64)
        return y.astype(np.float16 if once else np.float32).astype(np.float32)

    y = xs.copy()
    a, b = fused(lo, c, -hi * s), fused(hi, c, lo * s)
    if style == "neox":
        y[..., :half], y[..., half:rot] = a, b
    else:
        y[..., 0:rot:2], y[..., 1:rot:2] = a, b
    if fp8:
        y = np.clip(y * (np.float32(1.0) / scale), -TOP[dt], TOP[dt])
    code = torch.from_numpy(y).to(TORCH_DT[dt])
    code[..., rot:] = stored.cpu()[..., rot:]
    return code.view(torch.uint8)


@pytest.mark.parametrize("dt", ["bf16", "fp16", "e4m3", "e5m2"])
@pytest.mark.parametrize("kernel,heads,dim,rot,style", [
    ("pages", 8, 128, 128, "neox"), ("pages", 2, 64, 64, "gptj"), ("pages", 4, 96, 96, "neox"),
    ("pages", 4, 96, 24, "neox"), ("pages", 2, 96, 20, "gptj"), ("pairs", 4, 96, 96, "neox"),
    ("pairs", 8, 128, 128, "neox"), ("pairs", 2, 64, 32, "gptj"),
    ("hnd", 4, 128, 128, "neox"), ("kx", 8, 128, 128, "neox"), ("fanout", 8, 128, 64, "neox"),
    ("fanout", 8, 128, 128, "gptj"), ("tokens", 1, 128, 128, "neox"),
    ("tokens", 8, 128, 128, "neox"), ("tokens", 2, 64, 64, "gptj")])
def test_rotated_codes(gpu, tuning, kernel, heads, dim, rot, style, dt):
    print(f"case: codes {kernel} H{heads} D{dim} {rot} {style} {dt}", flush=True)
    block, n, layers = 16, 48, len(SCALES)
    dtype, fp8 = TORCH_DT[dt], dt in TOP
    esize = 1 if fp8 else 2
    ve = 16 // esize
    whole_vectors = (rot // 2) % ve == 0 if style == "neox" else rot % ve == 0
    g = torch.Generator().manual_seed(dim + heads)
    shape = (layers, n, 2, block, heads, dim)
    if fp8:
        bits = torch.randint(0, 256, shape, generator=g, dtype=torch.uint8)
        bits[(bits & 0x7c) == 0x7c] = 0x31  # no NaN codes (nor infinities)
        stored = bits.view(dtype).to(gpu)
    else:
        stored = torch.randn(shape, generator=g).to(dtype).to(gpu)
    ang = torch.rand(rot // 2, generator=g, dtype=torch.float64) * 6.28
    tabs = torch.stack([ang.cos(), ang.sin()], -1).float()
    want = _codes(stored[:, :, 0], tabs, rot, style, dt, whole_vectors)
    recs = stored.clone()
    if kernel == "kx":
        k = stored[:, :, 0].reshape(layers, n, block, heads, dim // ve, ve)
        recs[:, :, 0] = k.permute(0, 1, 3, 4, 2, 5).reshape(layers, n, block, heads, dim)
    staging = recs.transpose(0, 1).contiguous().view(-1).view(torch.uint8)
    inner = {"hnd": (heads, block, dim), "kx": (block * heads * dim,)}.get(
        kernel, (block, heads, dim))
    whole = torch.zeros((layers, 2, n, *inner), dtype=dtype, device=gpu)
    views = [w.transpose(2, 3) if kernel == "hnd" else w for w in whole.unbind(0)]
    geo = dict(block_size=block, head_dim=dim) if kernel == "kx" else {}
    table = ops.LayerTable(views, **geo)
    ids = np.random.default_rng(1).permutation(n).astype(np.int64)
    offs = np.arange(n, dtype=np.int64) * table.layout.slot_bytes
    how = dict(rot_dim=rot, style=style,
               k_scale=torch.tensor(SCALES, device=gpu) if fp8 else None)
    dev_tabs = tabs[None].to(gpu)
    if kernel == "pairs":
        tuning("rot_kernel", "pairs")
    if kernel == "tokens":
        slots = (ids[:, None] * block + np.arange(block)).reshape(-1)
        rows = (offs[:, None] + np.arange(block) * heads * dim * esize).reshape(-1)
        ops.scatter_slots_rerotate(
            table, torch.from_numpy(slots).to(gpu), torch.from_numpy(rows).to(gpu), staging,
            dev_tabs, torch.zeros(n * block, dtype=torch.int32, device=gpu), **how)
    elif kernel == "fanout":
        ops.PreparedFanout(table, ids, offs, staging, rope=(
            np.zeros(n, np.int64), dev_tabs, rot, style, how["k_scale"], None))()
    else:
        ops.scatter_rerotate(table, ids, offs, staging, dev_tabs, np.zeros(n, np.int64),
                             shared_records=False, **how)
    torch.cuda.synchronize()
    got = whole[:, 0, torch.from_numpy(ids).to(gpu)].cpu()
    if kernel == "hnd":
        got = got.transpose(2, 3).contiguous()
    elif kernel == "kx":
        got = got.reshape(layers, n, heads, dim // ve, block, ve).permute(0, 1, 4, 2, 3, 5) \
            .reshape(layers, n, block, heads, dim).contiguous()
    off = got.view(torch.uint8).reshape(want.shape) != want
    assert not off.any(), f"{int(off.sum())} of {off.numel()} bytes"
