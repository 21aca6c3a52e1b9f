"""dsr_plan_load / dsr_plan_gather / dsr_plan_shared against the numpy forms of
the same steps (ops.dest_order, ops.fanout_tables, ops._validate), and
their refusals."""

import ctypes

import numpy as np
import pytest
import torch

from daser_amd import _lib, ops


def _addr(a):
    return None if a is None else a.ctypes.data


def _load(ids, offs, rope, num_blocks, rec_end, staging, n_tables=4, fanout=0, room=None):
    n = len(ids)
    out = np.zeros(_lib.plan_bytes(n) if room is None else room, np.uint8)
    plan = _lib.Plan()
    rc = _lib.lib().dsr_plan_load(_addr(ids), _addr(offs), _addr(rope), n, num_blocks, rec_end,
                                  staging, n_tables, fanout, _addr(out), out.size,
                                  ctypes.addressof(plan))
    return rc, plan, out


def _section(out, at, count, dtype):
    return np.frombuffer(out[at:at + count * np.dtype(dtype).itemsize].tobytes(), dtype)


@pytest.mark.parametrize("n,num_blocks,n_records,dup", [
    (1, 1, 1, 0), (2, 4096, 1, 0), (16, 100000, 16, 0), (17, 40, 5, 0.5), (300, 310, 300, 0),
    (300, 9000, 150, 0.3), (5000, 5200, 40, 0.1), (5000, 70000, 2500, 0.02)])
@pytest.mark.parametrize("with_rope", [False, True])
def test_plan_load_matches_numpy(n, num_blocks, n_records, dup, with_rope):
    rng = np.random.default_rng(n + num_blocks)
    ids = rng.permutation(num_blocks)[:n].astype(np.int64)
    again = rng.random(n) < dup
    ids[again] = ids[rng.integers(0, n, again.sum())]
    size = 4096
    offs = rng.integers(0, n_records, n).astype(np.int64) * size
    rope = rng.integers(-1, 4, n).astype(np.int64) if with_rope else None
    rc, plan, out = _load(ids, offs, rope, num_blocks, size, n_records * size)
    assert rc == 0
    want_ids, want_offs, want_rope = ops.dest_order(ids, offs, rope)
    m = want_ids.size
    assert plan.n_pages == m and plan.bytes <= _lib.plan_bytes(n)
    assert np.array_equal(_section(out, 0, m, np.int64), want_offs)
    assert np.array_equal(_section(out, plan.off_ids, m, np.int32), want_ids)
    if with_rope:
        assert np.array_equal(_section(out, plan.off_rope, m, np.int32), want_rope)
    rc, plan, out = _load(ids, offs, rope, num_blocks, size, n_records * size, fanout=1)
    assert rc == 0
    src, start, pages, drope = ops.fanout_tables(want_ids, want_offs, want_rope)
    assert plan.n_src == src.size and plan.n_pages == m and plan.bytes <= _lib.plan_bytes(n)
    assert np.array_equal(_section(out, 0, src.size, np.int64), src)
    assert np.array_equal(_section(out, plan.off_start, src.size + 1, np.int32), start)
    assert np.array_equal(_section(out, plan.off_ids, m, np.int32), pages)
    if with_rope:
        assert np.array_equal(_section(out, plan.off_rope, m, np.int32), drope)
    assert _lib.lib().dsr_plan_shared(_addr(offs), n) == int(ops._shared_offsets(offs))


def test_plan_load_refusals():
    ids, offs = np.array([3, 1, 3], np.int64), np.array([0, 64, 128], np.int64)
    rope = np.array([0, -1, 3], np.int64)
    assert _load(ids, offs, rope, 4, 64, 192)[0] == 0
    assert _load(ids, offs, rope, 3, 64, 192)[0] == _lib.DSR_PLAN_ERR_BLOCK
    assert _load(-ids, offs, rope, 4, 64, 192)[0] == _lib.DSR_PLAN_ERR_BLOCK
    assert _load(ids, offs, rope, 4, 64, 191)[0] == _lib.DSR_PLAN_ERR_RECORD
    assert _load(ids, offs, rope, 4, 200, 192)[0] == _lib.DSR_PLAN_ERR_RECORD
    assert _load(ids, offs - 64, rope, 4, 64, 192)[0] == 0  # the bad one is superseded
    assert _load(ids, offs - 128, rope, 4, 64, 192)[0] == _lib.DSR_PLAN_ERR_RECORD
    assert _load(ids, offs + 8, rope, 4, 64, 300)[0] == _lib.DSR_PLAN_ERR_ALIGN
    assert _load(ids, offs, rope, 4, 64, 192, n_tables=3)[0] == _lib.DSR_PLAN_ERR_ROPE
    assert _load(ids, offs, rope - 1, 4, 64, 192)[0] == _lib.DSR_PLAN_ERR_ROPE
    assert _load(ids, offs, rope, 4, 64, 192, room=64)[0] == _lib.DSR_ERR_TOO_LARGE
    rc, plan, _ = _load(np.zeros(0, np.int64), np.zeros(0, np.int64), None, 4, 64, 192)
    assert rc == 0 and plan.n_pages == 0
    assert _lib.lib().dsr_plan_shared(None, 3) == _lib.DSR_ERR_ARG


@pytest.mark.parametrize("order", ["rising", "any"])
def test_plan_gather(order):
    rng = np.random.default_rng(1)
    n, span = 40, 256
    ids = rng.permutation(64)[:n].astype(np.int64)
    offs = np.arange(n, dtype=np.int64) * span
    if order == "any":
        offs = rng.permutation(offs)
    out = np.zeros(_lib.plan_bytes(n), np.uint8)
    plan = _lib.Plan()

    def call(i, o, end=span, gap=span, total=n * span):
        return _lib.lib().dsr_plan_gather(_addr(i), _addr(o), n, 64, end, gap, total, _addr(out),
                                          out.size, ctypes.addressof(plan))

    assert call(ids, offs) == 0 and plan.n_pages == n
    assert np.array_equal(_section(out, 0, n, np.int64), offs)
    assert np.array_equal(_section(out, plan.off_ids, n, np.int32), ids)
    assert call(ids, offs, gap=span + 16) == _lib.DSR_PLAN_ERR_OVERLAP
    assert call(ids, offs, total=n * span - 16) == _lib.DSR_PLAN_ERR_RECORD
    assert call(ids, offs + 4, total=n * span + 16) == _lib.DSR_PLAN_ERR_ALIGN
    assert call(ids + 64, offs) == _lib.DSR_PLAN_ERR_BLOCK


def _slots(slots, rows, rope, num_blocks, block, row, end, staging, n_tables=4, mode=0):
    n = len(slots)
    out = np.zeros(_lib.slot_plan_bytes(n), np.uint8)
    plan = _lib.SlotPlan()
    rc = _lib.lib().dsr_plan_slots(_addr(slots), _addr(rows), _addr(rope), n, num_blocks, block,
                                   row, end, staging, n_tables, mode, _addr(out), out.size,
                                   ctypes.addressof(plan))
    return rc, plan, out


@pytest.mark.parametrize("seed", range(12))
def test_plan_slots_matches_numpy(seed):
    """Ragged requests with padding, repeated slots, breaks in the record rows
    and table changes inside blocks, few and many slots for the pool."""
    rng = np.random.default_rng(seed)
    block = int(rng.choice([1, 4, 6, 16]))
    row, slot_bytes = 64, 64 * block * 2
    blocks = int(rng.integers(1, 40))
    num_blocks = blocks + int(rng.choice([0, 3, 100000]))
    ids = rng.permutation(num_blocks)[:blocks]
    tokens = blocks * block - int(rng.integers(0, block))
    slots = ops.slot_mapping_for([ids], [tokens], block)
    rows = ops.token_row_offsets([tokens], slot_bytes, block, row)
    rope = np.repeat(rng.integers(-1, 4, blocks), block)[:tokens].astype(np.int64)
    for i in rng.integers(0, tokens, 3):
        rope[i] = (rope[i] + 2) % 4 - 1
        rows[int(rng.integers(0, tokens))] = int(rng.integers(0, blocks)) * slot_bytes
    slots[rng.random(tokens) < 0.05] = -1
    again = rng.random(tokens) < 0.05
    slots[again] = slots[rng.integers(0, tokens, again.sum())]
    mix = rng.permutation(tokens) if seed % 2 else np.arange(tokens)
    slots, rows, rope = slots[mix], rows[mix], rope[mix]
    total = blocks * slot_bytes
    for r in (rope, None):
        rc, plan, out = _slots(slots, rows, r, num_blocks, block, row, row * (block + 1), total)
        assert rc == 0
        sm, ro, ri = ops.slot_order(slots, rows, r)
        sm, ro, ri = sm[sm >= 0], ro[sm >= 0], None if ri is None else ri[sm >= 0]
        pages, offs, pri, rest = ops.whole_pages(sm, ro, block, row, ri)
        rest &= sm >= 0
        n_p, n_t = pages.size, int(rest.sum())
        assert (plan.n_pages, plan.n_tokens) == (n_p, n_t)
        assert np.array_equal(_section(out, plan.off_ids, n_p, np.int64), pages)
        assert np.array_equal(_section(out, plan.off_offsets, n_p, np.int64), offs)
        assert np.array_equal(_section(out, plan.off_slots, n_t, np.int64), sm[rest])
        assert np.array_equal(_section(out, plan.off_rows, n_t, np.int64), ro[rest])
        if r is not None:
            assert np.array_equal(_section(out, plan.off_page_rope, n_p, np.int64), pri)
            assert np.array_equal(_section(out, plan.off_rope, n_t, np.int32), ri[rest])
    # a save: of a record row listed twice the last token
    rc, plan, out = _slots(slots, rows, None, num_blocks, block, row, row * (block + 1), total,
                           mode=1)
    keep = [i for i in range(tokens) if slots[i] >= 0 and
            not any(rows[j] == rows[i] and slots[j] >= 0 for j in range(i + 1, tokens))]
    assert rc == 0 and (plan.n_pages, plan.n_tokens) == (0, len(keep))
    assert np.array_equal(_section(out, plan.off_slots, len(keep), np.int64), slots[keep])
    assert np.array_equal(_section(out, plan.off_rows, len(keep), np.int64), rows[keep])


def test_plan_slots_refusals():
    slots, rows = np.array([0, -1, 7], np.int64), np.array([0, 3, 64], np.int64)
    rope = np.array([0, 1, -1], np.int64)
    call = lambda s, r, x, blocks=2, end=192, total=256, tables=2: _slots(  # noqa: E731
        s, r, x, blocks, 4, 64, end, total, tables)[0]
    assert call(slots, rows, rope) == 0
    assert call(slots + 1, rows, rope) == _lib.DSR_PLAN_ERR_SLOT
    assert call(slots, rows, rope, total=255) == _lib.DSR_PLAN_ERR_ROW
    assert call(slots, rows - 16, rope) == _lib.DSR_PLAN_ERR_ROW
    assert call(slots, rows + 8, rope, total=512) == _lib.DSR_PLAN_ERR_ROWALIGN
    assert call(slots, rows, rope, tables=1) == _lib.DSR_PLAN_ERR_ROPE


@pytest.mark.parametrize("bad,code", [(-16, _lib.DSR_PLAN_ERR_ROW), (256, _lib.DSR_PLAN_ERR_ROW),
                                      (8, _lib.DSR_PLAN_ERR_ROWALIGN)])
@pytest.mark.parametrize("num_blocks", [2, 1 << 40])
def test_plan_slots_rows_of_entries_left_out(bad, code, num_blocks):
    """A load reads the last entry of a repeated slot: the rows of the ones before
    are not looked at. A save refuses every bad row."""
    slots, rows = np.array([5, 5, 2], np.int64), np.array([bad, 64, 0], np.int64)
    rc, plan, out = _slots(slots, rows, None, num_blocks, 4, 64, 192, 256)
    assert rc == 0 and plan.n_tokens == 2
    assert np.array_equal(_section(out, plan.off_slots, 2, np.int64), [2, 5])
    assert np.array_equal(_section(out, plan.off_rows, 2, np.int64), [0, 64])
    assert _slots(slots, rows[[1, 0, 2]], None, num_blocks, 4, 64, 192, 256)[0] == code
    assert _slots(slots, rows, None, num_blocks, 4, 64, 192, 256, mode=1)[0] == code


def test_fanout_tables_of_caches_in_host_memory():
    """A fan-out load is prepared (checked, grouped) without a GPU."""
    caches = [torch.zeros(2, 8, 16, 2, 64, dtype=torch.bfloat16) for _ in range(2)]
    table = ops.LayerTable(caches)
    slot = table.layout.slot_bytes
    staging = torch.zeros(2 * slot, dtype=torch.uint8)
    load = ops.PreparedFanout(table, [6, 1, 3, 6], [0, slot, 0, slot], staging)
    assert (load.n_src, load.n_dst) == (2, 3)
    with pytest.raises(IndexError):
        ops.PreparedFanout(table, [6, 8], [0, slot], staging)
