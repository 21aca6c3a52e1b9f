"""Timed cases of the KV data-movement path.

What a serving process asks of this framework, through ``daser_amd.ops`` and
``daser_amd.position`` as the connector's data plane calls them: records of
new chunks gathered from the paged caches (save), cached chunks scattered
into a request's pages (load), with K re-rotated where a chunk moves to
another position (RAG prompts), for page tables and for vLLM's slot_mapping.
A case is one step of that kind: its model shape (the shapes of this
repository's workloads and benchmark), cache layout and type, and its requests.
The store file's transfers are not part of a pass.
"""

from __future__ import annotations

import math
import random

import numpy as np
import torch

from daser_amd import ops, position

THETA = 500000.0
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "e4m3": torch.float8_e4m3fn,
          "e5m2": torch.float8_e5m2}
# layers, KV heads, head_dim, block_size
SHAPES = {
    "qwen2-0.5b": (24, 2, 64, 16),
    "llama-3.2-1b": (16, 8, 64, 16),
    "qwen2.5-7b": (28, 4, 128, 16),
    "llama-3-8b": (32, 8, 128, 16),
    "llama-3-8b-block32": (32, 8, 128, 32),
    "gemma-2-9b": (42, 8, 256, 16),
    "phi-3-mini": (32, 32, 96, 16),
    "llama-3-70b": (80, 8, 128, 16),
    "llama-3-70b-tp8": (80, 1, 128, 16),
}
CHUNK = 256  # tokens of a cached chunk (the service's chunk length)


def _case(op, shape, dtype="bf16", layout="nhd", requests=1, low=CHUNK, high=CHUNK, chunks=0,
          chunk_tokens=0, cached=0, rot_dim=0, style="neox", tables="host"):
    """op: save_step (one gather a layer, as save_kv_layer does), gather,
    scatter, rerotate, gather_slots, scatter_slots, rerotate_slots.
    Requests of ``low`` to ``high`` tokens; or, with ``chunks``, of that many
    cached chunks of ``chunk_tokens`` each, out of ``cached`` different ones
    (0: every chunk is used once). ``tables``: where the slot_mapping is."""
    return dict(op=op, shape=shape, dtype=dtype, layout=layout, requests=requests, low=low,
                high=high, chunks=chunks, chunk_tokens=chunk_tokens, cached=cached,
                rot_dim=rot_dim, style=style, tables=tables)


def listed():
    named = {
        # smallest load: one cached chunk at its stored position, small model
        "load-chunk": _case("scatter", "qwen2-0.5b"),
        # one chunk that moves: the prefix differs from the one it was stored behind
        "load-chunk-moved": _case("rerotate", "llama-3-8b"),
        # a decode/prefill step's save: 8 requests commit a chunk each, layer by layer
        "save-step": _case("save_step", "llama-3-8b", requests=8),
        # a step's loads into the 3-D caches of vLLM's ROCm paged attention
        "load-step-splitx": _case("rerotate", "llama-3-8b", layout="kx", requests=8),
        # prefill of ragged prompts saved at once, and loaded back
        "gather-prompts": _case("gather", "llama-3-8b", requests=32, low=512, high=8192),
        "scatter-prompts": _case("scatter", "llama-3-8b", requests=32, low=512, high=8192),
        # RAG: prompts assembled from documents' chunks, each at a new position
        "rag-moved": _case("rerotate", "llama-3-8b", requests=16, chunks=10, chunk_tokens=512),
        # fp8 KV with per-layer scales, moved prefixes
        "fp8-moved": _case("rerotate", "llama-3-8b", dtype="e4m3", requests=16, low=256,
                           high=16384),
        # RAG over a few hot documents: each record goes to many requests
        "rag-shared": _case("rerotate", "llama-3-70b", requests=16, chunks=8, chunk_tokens=512,
                            cached=16),
        # the same kind of step on one rank of 8-way tensor parallelism (4 KiB pages)
        "rag-shared-tp8": _case("rerotate", "llama-3-70b-tp8", requests=16, chunks=64,
                                chunk_tokens=512, cached=64),
        # save driven by vLLM's slot_mapping, ragged ends included
        "save-slots": _case("gather_slots", "qwen2-0.5b", requests=64, low=100, high=8000,
                            tables="device"),
        # head-major (HND) caches, 16 KiB pages
        "load-hnd": _case("scatter", "qwen2.5-7b", layout="hnd", requests=8, low=100, high=4000),
    }
    return [dict(case, name=name) for name, case in named.items()]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng: random.Random):
    """A step of the same kinds at another shape, type, layout and size, from
    16 pages up to 8 GB of page data."""
    op = rng.choice(["save_step", "gather", "scatter", "scatter", "rerotate", "rerotate",
                     "rerotate", "gather_slots", "scatter_slots", "rerotate_slots"])
    shape = rng.choice(sorted(SHAPES))
    layers, heads, dim, block = SHAPES[shape]
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "e4m3", "e4m3", "e5m2"])
    layout = rng.choice(["nhd", "nhd", "kx", "hnd"])
    if "slots" in op or (layout == "hnd" and op == "rerotate" and dim & (dim - 1)):
        layout = "nhd"  # the token form is token-major; HND moves need power-of-two heads
    if op == "rerotate_slots" and dim & (dim - 1):
        op = "rerotate"
    style = rng.choice(["neox", "neox", "neox", "gptj"]) if op.startswith("rerotate") else "neox"
    rot_dim = dim // 2 if op.startswith("rerotate") and dim == 128 and rng.random() < 0.2 else 0
    if op == "rerotate" and dim == 96 and layout == "nhd" and rng.random() < 0.3:
        rot_dim = 24  # partial rotary in odd widths
    token = 2 * layers * heads * dim * (1 if dtype in ("e4m3", "e5m2") else 2)
    total = _log_uniform(rng, 256, max(1024, min(1 << 20, (8 << 30) // token)))
    case = _case(op, shape, dtype, layout, rot_dim=rot_dim, style=style,
                 tables=rng.choice(["host", "device"]) if "slots" in op else "host")
    if op in ("scatter", "rerotate") and rng.random() < 0.4:
        chunk_tokens = rng.choice([128, 256, 512])
        n = max(1, total // chunk_tokens)
        case["chunks"] = min(n, rng.randint(1, 16))
        case["requests"] = max(1, n // case["chunks"])
        case["chunk_tokens"] = chunk_tokens
        n = case["chunks"] * case["requests"]
        if n >= 4 and rng.random() < 0.5:
            case["cached"] = rng.randint(max(1, n // 16), max(1, n // 2))
        return case
    case["requests"] = requests = min(rng.randint(1, 64), max(1, total // 64))
    mean = total // requests
    case["low"], case["high"] = max(1, mean // rng.choice([1, 2, 8])), mean + mean // 3 + 1
    return case


class _Step:
    """The step of a case: sizes from the case alone, placement, positions
    and values from the seed."""

    def __init__(self, case, seed=0):
        self.case = case
        self.layers, self.heads, self.dim, self.block = SHAPES[case["shape"]]
        self.dtype = DTYPES[case["dtype"]]
        self.fp8 = case["dtype"] in ("e4m3", "e5m2")
        self.page_elems = self.block * self.heads * self.dim
        self.page_bytes = self.page_elems * (1 if self.fp8 else 2)
        self.slot_bytes = 2 * self.page_bytes * self.layers
        self.rot_dim = case["rot_dim"] or self.dim
        sizes = np.random.default_rng([case["requests"], case["low"], case["high"]])
        if case["chunks"]:
            tokens = [case["chunk_tokens"]] * (case["requests"] * case["chunks"])
        else:
            tokens = sizes.integers(case["low"], case["high"] + 1, case["requests"]).tolist()
        self.tokens = tokens  # of each run of pages that moves as one
        self.pages = [-(-t // self.block) for t in tokens]
        self.total = sum(self.pages)
        # the records in the staging buffer: one per page, or those of the cached chunks
        self.cached = min(case["cached"] or len(tokens), len(tokens)) if case["chunks"] else 0
        self.records = self.cached * self.pages[0] if self.cached else self.total
        self.num_blocks = self.total + self.total // 20 + 1
        rng = np.random.default_rng(seed)
        self.page_ids = rng.permutation(self.num_blocks)[:self.total].astype(np.int32)
        if self.cached:
            source = np.concatenate([rng.permutation(self.cached)
                                     for _ in range(-(-len(tokens) // self.cached))])
            source = source[:len(tokens)]
            record = source[:, None] * self.pages[0] + np.arange(self.pages[0])
            self.offsets = record.reshape(-1).astype(np.int64) * self.slot_bytes
        else:
            self.offsets = np.arange(self.total, dtype=np.int64) * self.slot_bytes
        # every run moves by its own distance, backwards too
        self.deltas = [int(d) or 1 for d in rng.integers(-8192, 32768, len(tokens))]

    @property
    def per_page(self):
        """The table index of each page: its run's."""
        return np.repeat(np.arange(len(self.pages), dtype=np.int32), self.pages)

    def page_shape(self, layout):
        b, h, d = self.block, self.heads, self.dim
        return {"nhd": (b, h, d), "hnd": (h, b, d), "kx": (b * h * d,)}[layout]


def _fill(out, scales, gen):
    """N(0, 1) values of the caches' type; 8-bit ones quantised by the
    scales, which run along dimension 1 of out[:, l]."""
    step = max(1, (1 << 28) // max(1, out[0].numel()))
    for i in range(0, out.shape[0], step):
        part = out[i:i + step]
        if scales is None:
            part.normal_(generator=gen)
        else:
            x = torch.empty(part.shape, dtype=torch.bfloat16, device=part.device)
            x.normal_(generator=gen)
            part.copy_(x.float() / scales.view(1, -1, 1))


def _inputs(step, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(dev).manual_seed(seed)
    scales = None
    if step.fp8:
        scales = 0.010 + 0.004 * torch.rand(step.layers, generator=gen, device=dev)
    if step.case["op"] in ("save_step", "gather", "gather_slots"):
        whole = torch.empty((step.layers, 2, step.num_blocks, step.page_elems),
                            dtype=step.dtype, device=dev)
        _fill(whole.view(step.layers, 1, -1), None if scales is None else scales[:1], gen)
        # a short last slot leaves rows of its record unwritten
        records = torch.zeros(step.records * step.slot_bytes, dtype=torch.uint8, device=dev)
    else:
        whole = torch.zeros((step.layers, 2, step.num_blocks, step.page_elems),
                            dtype=step.dtype, device=dev)
        values = torch.empty((step.records, step.layers, 2 * step.page_elems), dtype=step.dtype,
                             device=dev)
        _fill(values, scales, gen)
        records = values.view(-1).view(torch.uint8)
    return whole, records, scales


def prepare(case, seed):
    step = _Step(case, seed)
    whole, records, scales = _inputs(step, seed)
    layout = case["layout"]
    pages = whole.view(step.layers, 2, step.num_blocks, *step.page_shape(layout))
    if layout == "hnd":
        pages = pages.transpose(3, 4)
    geometry = dict(block_size=step.block, head_dim=step.dim) if layout == "kx" else {}
    table = ops.LayerTable(list(pages.unbind(0)), **geometry)
    state = dict(case=case, table=table, whole=whole, records=records, scales=scales,
                 layers=step.layers, page_ids=step.page_ids, offsets=step.offsets,
                 deltas=step.deltas, rope=step.per_page, rot_dim=step.rot_dim)
    if "slots" in case["op"]:
        first = np.concatenate([[0], np.cumsum(step.pages)])
        blocks = [step.page_ids[a:b] for a, b in zip(first[:-1], first[1:])]
        slots = ops.slot_mapping_for(blocks, step.tokens, step.block)
        rows = ops.token_row_offsets(step.tokens, step.slot_bytes, step.block,
                                     step.page_bytes // step.block)
        rope = np.repeat(np.arange(len(step.tokens), dtype=np.int32), step.tokens)
        if case["tables"] == "device":
            slots, rows, rope = (torch.from_numpy(x).to(whole.device)
                                 for x in (slots, rows, rope))
        state.update(slots=slots, rows=rows, rope=rope)
    return state


def run(state):
    s, case = state, state["case"]
    op, table, records = case["op"], s["table"], s["records"]
    tables = None
    if op.startswith("rerotate"):
        tables = position.delta_tables(s["deltas"], s["rot_dim"], THETA,
                                       device=table.layout.device)
    how = dict(rot_dim=s["rot_dim"], style=case["style"], k_scale=s["scales"])
    if op == "save_step":
        gather = ops.PreparedGather(table, s["page_ids"], s["offsets"], records)
        stream = torch.cuda.current_stream().cuda_stream
        for layer in range(s["layers"]):
            gather(layer, 1, stream)
    elif op == "gather":
        ops.gather(table, s["page_ids"], s["offsets"], records)
    elif op == "gather_slots":
        ops.gather_slots(table, s["slots"], s["rows"], records)
    elif op == "scatter":
        ops.scatter(table, s["page_ids"], s["offsets"], records)
    elif op == "scatter_slots":
        ops.scatter_slots(table, s["slots"], s["rows"], records)
    elif op == "rerotate_slots":
        ops.scatter_slots_rerotate(table, s["slots"], s["rows"], records, tables, s["rope"],
                                   **how)
    else:
        ops.scatter_rerotate(table, s["page_ids"], s["offsets"], records, tables, s["rope"],
                             **how)
    return _outputs(case, s["whole"], records)


def _outputs(case, whole, records):
    """Whole buffers: moved bytes as whole numbers, re-rotated caches as
    values (a few layers to an output)."""
    if case["op"] in ("save_step", "gather", "gather_slots"):
        return records.view(torch.int64)
    if not case["op"].startswith("rerotate"):
        return whole.view(-1).view(torch.int64)
    return list(whole.split(-(-whole.shape[0] // 8)))


def work(case):
    """Every page (token) that moves, read once from its record (a shared
    record once) or its cache and written once; 3 operations for each
    rotated value."""
    step = _Step(case)
    moved = step.total * step.slot_bytes
    read = step.records * step.slot_bytes
    if "slots" in case["op"]:  # rows of the tokens alone
        moved = read = sum(step.tokens) * (step.slot_bytes // step.block)
    flops = 0
    if case["op"].startswith("rerotate"):
        elems = moved // (2 if not step.fp8 else 1) // 2  # K's share
        flops = 3 * elems * step.rot_dim // step.dim
    return {"bytes": moved + read, "flops": flops}


def tolerance(case):
    """Copies are bytes. A rotated value is one fp32 sum of two products,
    rounded once to the caches' type: correct implementations differ where
    that sum's last bits decide a tie, one unit in the last place. Four times
    what fused against separate products and a float64 sum differ by (bf16
    1.7e-5, fp16 4.7e-6, 8-bit 2.7e-5 over 4 M values, where a single tie in
    the smallest cases weighs more)."""
    if not case["op"].startswith("rerotate"):
        return "exact"
    return {"bf16": {"rel": 1e-4, "max": 0.016}, "fp16": {"rel": 2e-5, "max": 0.002},
            "e4m3": {"rel": 2e-3, "max": 0.26}, "e5m2": {"rel": 2e-3, "max": 0.52}}[case["dtype"]]


def exact(case, seed):
    """The re-rotated caches in float64, from the inputs alone."""
    if not case["op"].startswith("rerotate"):
        return None
    step = _Step(case, seed)
    b, h, d, rot = step.block, step.heads, step.dim, step.rot_dim
    if 2 * step.num_blocks * step.layers * step.page_elems > 10e9:
        return None  # over 80 GB of float64
    whole, records, scales = _inputs(step, seed)
    records = records.view(step.dtype).view(step.records, step.layers, 2, step.page_elems)
    dev = whole.device
    out = torch.zeros(whole.shape, dtype=torch.float64, device=dev)
    inv = THETA ** (-torch.arange(0, rot, 2, dtype=torch.float64, device=dev) / rot)
    runs = torch.tensor(step.deltas, dtype=torch.float64, device=dev)
    angle = (runs[:, None] * inv)[torch.from_numpy(step.per_page).to(dev).long()]
    cos, sin = angle.cos()[:, None, None, :], angle.sin()[:, None, None, :]
    ids = torch.from_numpy(step.page_ids).to(dev).long()
    source = torch.from_numpy(step.offsets // step.slot_bytes).to(dev).long()
    # the token form moves the tokens of a short last page and no more
    keep = torch.ones(step.total, b, dtype=torch.bool, device=dev)
    if "slots" in case["op"]:
        last = np.cumsum(step.pages) - 1
        for page, tokens in zip(last.tolist(), step.tokens):
            keep[page, (tokens - 1) % b + 1:] = False
    layout = case["layout"]
    x = 16 if step.fp8 else 8  # elements of a 16-byte vector
    part = max(1, (1 << 27) // step.page_elems)
    for layer in range(step.layers):
        scale = 1.0 if scales is None else float(scales[layer])
        for i in range(0, step.total, part):
            sl = slice(i, i + part)
            n = ids[sl].numel()
            rec = records[:, layer].view(torch.uint8).view(step.records, 2, -1)[source[sl]]
            k, v = (rec[:, j].contiguous().view(step.dtype).double() for j in (0, 1))
            if layout == "kx":  # [H][D / X][block][X]; V moves as it is
                k = k.view(n, h, d // x, b, x).permute(0, 3, 1, 2, 4).reshape(n, b, h, d)
            k = (k.view(n, b, h, d) * scale).clone()
            c, s = cos[sl], sin[sl]
            if case["style"] == "neox":
                lo, hi = k[..., :rot // 2].clone(), k[..., rot // 2:rot].clone()
                k[..., :rot // 2] = lo * c - hi * s
                k[..., rot // 2:rot] = hi * c + lo * s
            else:
                lo, hi = k[..., 0:rot:2].clone(), k[..., 1:rot:2].clone()
                k[..., 0:rot:2] = lo * c - hi * s
                k[..., 1:rot:2] = hi * c + lo * s
            k /= scale
            if layout == "kx":
                k = k.view(n, b, h, d // x, x).permute(0, 2, 3, 1, 4)
            else:
                k = k * keep[sl].view(n, b, 1, 1)
                v = v.view(n, b, h, d) * keep[sl].view(n, b, 1, 1)
                if layout == "hnd":
                    k, v = k.transpose(1, 2), v.transpose(1, 2)
            out[layer, 0, ids[sl]] = k.reshape(n, -1)
            out[layer, 1, ids[sl]] = v.reshape(n, -1)
    return _outputs(case, out, records)
