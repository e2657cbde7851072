"""Host planner invariants (pure host code in libaspire_hip.so; no GPU needed)."""

import ctypes
from pathlib import Path

import numpy as np
import pytest
import torch

from aspire_amd import _lib

LIB = Path(_lib.LIB_PATH)
pytestmark = pytest.mark.skipif(not LIB.exists(), reason="libaspire_hip.so not built")

HEADER_INTS = 32


def layout(num_cus=256, waves_per_cu=8, float_ws=384 << 20):
    lay = _lib.PlanLayout()
    rc = _lib.lib().aspire_plan_layout_init(num_cus, waves_per_cu, 8 << 20, float_ws, 128, ctypes.byref(lay))
    _lib.check(rc, "layout")
    return lay


def offsets(lay):
    W = lay.num_waves
    cur = HEADER_INTS
    indptr = []
    for _ in range(3):
        indptr.append(cur)
        cur += W + 1
    cur = (cur + 7) & ~7
    items = []
    for _ in range(3):
        items.append(cur)
        cur += lay.max_items * 8
    return indptr, items, cur


def plan(lay, qo, kvp, kvl, hq, hkv, per_head=False, causal=True):
    buf = np.zeros(8 << 18, dtype=np.int32)
    info = _lib.PlanInfo()
    qo = np.ascontiguousarray(qo, dtype=np.int32)
    kvp = np.ascontiguousarray(kvp, dtype=np.int32)
    kvl = np.ascontiguousarray(kvl, dtype=np.int32)
    batch = len(kvl) // hkv if per_head else len(kvl)
    rc = _lib.lib().aspire_plan_build(
        ctypes.byref(lay), qo.ctypes.data_as(ctypes.c_void_p), kvp.ctypes.data_as(ctypes.c_void_p),
        kvl.ctypes.data_as(ctypes.c_void_p), batch, int(per_head), hq, hkv, 16, int(causal),
        buf.ctypes.data_as(ctypes.c_void_p), buf.nbytes, ctypes.byref(info))
    _lib.check(rc, "plan")
    return buf, info


def decode(lay, buf, info):
    indptr_off, items_off, merge_off = offsets(lay)
    W = lay.num_waves
    classes = []
    for c in range(3):
        ip = buf[indptr_off[c] : indptr_off[c] + W + 1]
        it = buf[items_off[c] : items_off[c] + info.num_items[c] * 8].reshape(-1, 8)
        classes.append((ip, it))
    merges = buf[merge_off : merge_off + info.num_merge * 8].reshape(-1, 8)
    return classes, merges


def expected_tiles(q_len, kv_len, group, causal=True):
    """Query tiles of a row, (t0, tq, keys): rows longer than 48 query rows are cut into
    tiles of 48 // group tokens whose keys end at their last token (causal)."""
    tile = max(1, 48 // group)
    if q_len * group <= 48:
        return [(0, q_len, kv_len)]
    return [(t0, min(tile, q_len - t0), max(kv_len - q_len + t0 + min(tile, q_len - t0), 0) if causal else kv_len)
            for t0 in range(0, q_len, tile)]


DIRECT = 1 << 16  # item flag: heads of a head-aligned row read different lists


def check_cover(lay, buf, info, qo, kvp, kvl, hq, hkv, per_head=False, causal=True, seg_start=None):
    classes, merges = decode(lay, buf, info)
    group = hq // hkv
    hpu = int(buf[4])
    starts = np.asarray(seg_start) if seg_start is not None else np.asarray(kvp)[: len(kvl)]
    seen = {}
    partial_rows = set()
    for c, (ip, it) in enumerate(classes):
        assert ip[0] == 0 and ip[-1] == len(it) and np.all(np.diff(ip) >= 0)
        for w in range(lay.num_waves):
            for row in it[ip[w] : ip[w + 1]]:
                q_start, q_len, kv_len, base, pb, pe, bg, prow = row.tolist()
                flag, q_len = q_len & DIRECT, q_len & (DIRECT - 1)
                b, g = bg >> 8, bg & 255
                shared = not per_head or len(set(starts[b * hkv : (b + 1) * hkv].tolist())) == 1
                assert bool(flag) == (hpu > 1 and not shared), (b, g, flag, hpu)
                assert (q_len * group - 1) // 16 == c
                seg = b * hkv + g if per_head else b
                tiles = {t0: (tq, keys) for t0, tq, keys in
                         expected_tiles(qo[b + 1] - qo[b], kvl[seg], group, causal)}
                t0 = q_start - qo[b]
                assert t0 in tiles and (q_len, kv_len) == tiles[t0], (b, t0, q_len, kv_len)
                assert base == starts[seg] and pe <= (kv_len + 15) // 16
                for p in range(pb, pe):
                    key = (b, g, t0, p)
                    assert key not in seen, f"page {key} planned twice"
                    seen[key] = prow
                if prow >= 0:
                    for r in range(q_len * group):
                        assert prow + r not in partial_rows
                        partial_rows.add(prow + r)
    # every page of every query tile of every segment with queries is covered exactly once
    nrows = len(kvl) // hkv if per_head else len(kvl)
    for b in range(min(len(qo) - 1, nrows)):
        if qo[b + 1] - qo[b] <= 0:
            continue
        for g in range(hkv):
            seg = b * hkv + g if per_head else b
            for t0, tq, keys in expected_tiles(qo[b + 1] - qo[b], kvl[seg], group, causal):
                for p in range((keys + 15) // 16):
                    assert (b, g, t0, p) in seen
    # merge items reference the split pieces; their row ranges cover each split segment's rows
    # once, in ranges the merge kernel's piece groups fit (48 rows, or 24 / 12 rows for items of
    # more than 8 / 16 pieces)
    covered = {}
    for m in merges:
        q_start, q_len, bg, first, pieces, rows, row_begin, row_count = m.tolist()
        assert pieces >= 2 and rows == q_len * group
        assert 0 <= row_begin and 0 < row_count and row_begin + row_count <= rows
        assert row_count <= (12 if pieces > 16 else 24 if pieces > 8 else 48)
        for k in range(pieces):
            assert first + k * rows in partial_rows
        got = covered.setdefault((q_start, bg, first), set())
        assert got.isdisjoint(range(row_begin, row_begin + row_count))
        got.update(range(row_begin, row_begin + row_count))
    for (q_start, bg, first), got in covered.items():
        q_len = next(int(m[1]) for m in merges if (m[0], m[2], m[3]) == (q_start, bg, first))
        assert got == set(range(q_len * group))
    return seen


def test_cover_and_balance_config1_shape():
    B, hq, hkv = 32, 32, 8
    q_len = np.array([1] * 16 + [4] * 16)
    kvl = np.array([128 * 16] * 16 + [32768] * 16 + [0])
    pages = (kvl + 15) // 16
    qo = np.concatenate([[0], np.cumsum(q_len), [80]])
    kvp = np.concatenate([[0], np.cumsum(pages[:B]), [pages[:B].sum()]])
    lay = layout()
    buf, info = plan(lay, qo, kvp, kvl, hq, hkv)
    check_cover(lay, buf, info, qo, kvp, kvl, hq, hkv)
    assert info.total_pages == int(pages[:B].sum()) * hkv
    # stream-K balance: every wave streams floor or ceil of the mean page count
    classes, _ = decode(lay, buf, info)
    ip, it = classes[0]
    per_wave = np.array([int((it[ip[w]:ip[w + 1], 5] - it[ip[w]:ip[w + 1], 4]).sum()) for w in range(lay.num_waves)])
    mean = info.total_pages / lay.num_waves
    assert per_wave.max() <= np.ceil(mean) and per_wave.min() >= np.floor(mean)


def test_mixed_classes_ragged_and_empty_rows():
    hq, hkv = 32, 8
    q_len = np.array([1, 2, 5, 9, 0, 3, 12 // 4 * 4 // 4, 1])
    kvl = np.array([37, 0, 4096 + 5, 100000, 50, 17, 16, 1, 0])
    pages = (kvl + 15) // 16
    B = len(q_len)
    qo = np.concatenate([[0], np.cumsum(q_len), [q_len.sum() + 3]])
    kvp = np.concatenate([[0], np.cumsum(pages[:B]), [pages[:B].sum()]])
    kvl_full = np.concatenate([kvl[:B], [0]])
    lay = layout(num_cus=16, waves_per_cu=4)
    buf, info = plan(lay, qo, kvp, kvl_full, hq, hkv)
    check_cover(lay, buf, info, qo, kvp, kvl_full, hq, hkv)
    assert info.num_items[2] > 0 and info.num_merge > 0


def test_per_head_lists():
    hq, hkv, B = 32, 8, 3
    rng = np.random.default_rng(0)
    kvl = rng.integers(1, 3000, size=B * hkv)
    pages = (kvl + 15) // 16
    kvp = np.concatenate([[0], np.cumsum(pages)])
    qo = np.array([0, 1, 2, 3])
    lay = layout(num_cus=8, waves_per_cu=4)
    buf, info = plan(lay, qo, kvp, kvl, hq, hkv, per_head=True)
    assert int(buf[4]) == 1  # heads of a row differ in length: one wave per (row, head)
    check_cover(lay, buf, info, qo, kvp, kvl, hq, hkv, per_head=True)
    # one length per row: head-aligned slots, every row's heads on their own lists (flagged)
    kvl_u = np.repeat(kvl[::hkv], hkv)
    kvp_u = np.concatenate([[0], np.cumsum((kvl_u + 15) // 16)])
    buf, info = plan(lay, qo, kvp_u, kvl_u, hq, hkv, per_head=True)
    assert int(buf[4]) == hkv
    check_cover(lay, buf, info, qo, kvp_u, kvl_u, hq, hkv, per_head=True)


def test_rejects_bad_inputs():
    lay = layout(num_cus=4, waves_per_cu=4)
    with pytest.raises(ValueError, match="pages"):
        plan(lay, np.array([0, 1]), np.array([0, 1]), np.array([40]), 32, 8)  # list shorter than kv_len
    with pytest.raises(ValueError, match="multiple"):
        plan(lay, np.array([0, 1]), np.array([0, 1]), np.array([16]), 30, 8)


def test_partial_capacity_shrinks_split():
    hq, hkv = 32, 8
    kvl = np.array([32768] * 4 + [0])
    qo = np.array([0, 4, 8, 12, 16, 16])
    pages = (kvl + 15) // 16
    kvp = np.concatenate([[0], np.cumsum(pages[:4]), [pages[:4].sum()]])
    small = layout(num_cus=64, waves_per_cu=8, float_ws=40 * 129 * 4 * 16)
    buf, info = plan(small, qo, kvp, kvl, hq, hkv)
    assert info.partial_rows <= small.partial_rows_cap
    check_cover(small, buf, info, qo, kvp, kvl, hq, hkv)


@pytest.mark.parametrize("causal", [True, False])
def test_prefill_rows_split_into_query_tiles(causal):
    """Chunked prefill: rows of 300 and 1000 new tokens over prefixes of 700 and 0 tokens (GQA 4:
    tiles of 12 tokens), beside a decode row."""
    hq, hkv = 32, 8
    qo = np.array([0, 300, 1300, 1301])
    kvl = np.array([1000, 1000, 5000])
    pages = (kvl + 15) // 16
    kvp = np.concatenate([[0], np.cumsum(pages)])
    lay = layout(num_cus=16, waves_per_cu=4)
    buf, info = plan(lay, qo, kvp, kvl, hq, hkv, causal=causal)
    assert info.split_rows == 2 and info.max_rows == 48
    check_cover(lay, buf, info, qo, kvp, kvl, hq, hkv, causal=causal)
    # the first tile of the second row only needs the keys up to its 12th token
    if causal:
        assert expected_tiles(1000, 1000, 4)[0] == (0, 12, 12)


def plan_segments(lay, qo, start, pages, kvl, hq, hkv, causal=True):
    buf = np.zeros(8 << 18, dtype=np.int32)
    info = _lib.PlanInfo()
    arr = lambda a: np.ascontiguousarray(a, dtype=np.int32)
    qo, start, pages, kvl = arr(qo), arr(start), arr(pages), arr(kvl)
    rc = _lib.lib().aspire_plan_build_segments(
        ctypes.byref(lay), qo.ctypes.data_as(ctypes.c_void_p), start.ctypes.data_as(ctypes.c_void_p),
        pages.ctypes.data_as(ctypes.c_void_p), kvl.ctypes.data_as(ctypes.c_void_p), len(kvl) // hkv, hq, hkv, 16,
        int(causal), buf.ctypes.data_as(ctypes.c_void_p), buf.nbytes, ctypes.byref(info))
    _lib.check(rc, "plan_segments")
    return buf, info


def test_segments_shared_and_per_head_rows():
    """Verify rows share one list across heads (staged), draft rows hold one per head (flagged
    direct); all heads of a row have one length, so the plan is head-aligned."""
    hq, hkv = 32, 8
    rng = np.random.default_rng(2)
    ctx = np.array([5000, 700, 3000, 123, 64, 2000])
    ql = np.array([1, 4, 1, 9, 1, 2])
    draft = ql == 1
    cnt = np.where(draft, np.minimum(40, (ctx + 15) // 16), (ctx + 15) // 16)
    start = np.zeros((len(ctx), hkv), dtype=np.int64)
    pos = 0
    for b in range(len(ctx)):
        if draft[b]:
            start[b] = pos + cnt[b] * np.arange(hkv)
            pos += cnt[b] * hkv
        else:
            start[b] = pos
            pos += cnt[b]
    start = start.reshape(-1)
    pages = np.repeat(cnt, hkv)
    kvl = np.repeat((cnt - 1) * 16 + (ctx - 1) % 16 + 1, hkv)
    qo = np.concatenate([[0], np.cumsum(ql)])
    lay = layout(num_cus=16, waves_per_cu=4)
    buf, info = plan_segments(lay, qo, start, pages, kvl, hq, hkv)
    assert int(buf[4]) == hkv
    check_cover(lay, buf, info, qo, None, kvl, hq, hkv, per_head=True, seg_start=start)
    # one head of one row longer than its siblings: per-(row, head) slots, no flags
    kvl2 = kvl.copy()
    kvl2[3] -= 16
    buf2, info2 = plan_segments(lay, qo, start, pages, kvl2, hq, hkv)
    assert int(buf2[4]) == 1
    check_cover(lay, buf2, info2, qo, None, kvl2, hq, hkv, per_head=True, seg_start=start)
    # a list shorter than its length is rejected
    with pytest.raises(ValueError, match="pages"):
        bad = pages.copy()
        bad[5] -= 1
        plan_segments(lay, qo, start, bad, kvl, hq, hkv)


def test_rejects_gqa_group_wider_than_three_tiles():
    """A query token's GQA group must fit one 3-tile item (48 rows): 64 q heads over one
    kv head is refused with ASPIRE_ERR_INVALID instead of planned past the last class."""
    lay = layout(num_cus=16, waves_per_cu=4)
    qo = np.array([0, 1], dtype=np.int32)
    kvp = np.array([0, 4], dtype=np.int32)
    kvl = np.array([64], dtype=np.int32)
    buf = np.zeros(8 << 18, dtype=np.int32)
    info = _lib.PlanInfo()
    rc = _lib.lib().aspire_plan_build(
        ctypes.byref(lay), qo.ctypes.data_as(ctypes.c_void_p), kvp.ctypes.data_as(ctypes.c_void_p),
        kvl.ctypes.data_as(ctypes.c_void_p), 1, 0, 64, 1, 16, 1, buf.ctypes.data_as(ctypes.c_void_p), buf.nbytes,
        ctypes.byref(info))
    assert rc == _lib.ASPIRE_ERR_INVALID
    assert "at most 48" in _lib.lib().aspire_last_error().decode()
    # the widest accepted group (48 q heads per kv head) still plans
    plan(lay, qo, kvp, kvl, 48, 1)


def test_config3_layer_cost_balance():
    """A config-3 mixed layer (64 rows, contexts U[8k, 32k], per-head top-128 draft lists, verify
    q_len U{2..9}) on 256 CUs: the three row-tile classes form one stream-K sequence in cost
    units (quarters: 33 per staged 1-tile page, 32 per staged 2-/3-tile page, 48 per per-head
    page), so every slot streams the mean cost to within one page, and no merge needs more than
    one round of loads."""
    from aspire_amd.workloads import PAGE, config3_rows

    ctx, ql, dr = config3_rows(seed=0)
    hq, hkv = 32, 8
    starts, pages, kvl = [], [], []
    pos = 0
    for b in range(len(ctx)):
        n = (int(ctx[b]) + PAGE - 1) // PAGE
        for g in range(hkv):
            starts.append(pos + g * 128 if dr[b] else pos)
            pages.append(128 if dr[b] else n)
            kvl.append(127 * PAGE + int(ctx[b]) - (n - 1) * PAGE if dr[b] else int(ctx[b]))
        pos += 128 * hkv if dr[b] else n
    qo = np.concatenate([[0], np.cumsum(ql)])
    lay = layout(num_cus=256, waves_per_cu=4)
    buf, info = plan_segments(lay, qo, starts, pages, kvl, hq, hkv)
    check_cover(lay, buf, info, qo, None, np.array(kvl), hq, hkv, per_head=True, seg_start=np.array(starts))
    classes, merges = decode(lay, buf, info)
    hpu = int(buf[4])
    assert hpu == hkv
    cost = np.zeros(lay.num_waves)
    for c, (ip, it) in enumerate(classes):
        for w in range(lay.num_waves):
            for row in it[ip[w] : ip[w + 1]]:
                direct = (int(row[1]) & DIRECT) != 0
                cost[w] += (int(row[5]) - int(row[4])) * (48 if direct else 33 if c == 0 else 32)
    slot_cost = cost[::hpu]
    assert slot_cost.max() - slot_cost.min() <= 2 * 48
    assert (merges[:, 4] <= 8).all()


def test_merge_row_ranges_lone_long_row():
    """One 131,072-token verify row with q_len 9 at GQA 4 (36 rows, 3 tiles) beside a short draft
    row: the long row streams over every slot, and its 36-row merges come as row ranges of 12 rows,
    so that four lane groups share each row's pieces."""
    hq, hkv = 32, 8
    ql = np.array([9, 1])
    kvl = np.array([131072, 300])
    pages = (kvl + 15) // 16
    qo = np.concatenate([[0], np.cumsum(ql)])
    kvp = np.concatenate([[0], np.cumsum(pages)])
    lay = layout(num_cus=256, waves_per_cu=4)
    buf, info = plan(lay, qo, kvp, kvl, hq, hkv)
    check_cover(lay, buf, info, qo, kvp, kvl, hq, hkv)
    _, merges = decode(lay, buf, info)
    long = merges[merges[:, 5] == 36]
    assert len(long) and (long[:, 4] > 16).all() and (long[:, 7] == 12).all()


@pytest.mark.parametrize("hq,hkv,q_len,kv_len,float_ws", [
    (16, 8, [1, 1, 5, 5], [1024, 1000, 4096, 4090], 384 << 20),
    (32, 8, [5, 0, 12, 1], [16, 300, 0, 513], 384 << 20),      # no queries, no keys, one page, a 3-tile row
    (16, 2, [1, 3], [5000, 77], 384 << 20),                    # 2 kv heads: not head-aligned
    (32, 4, [9] * 16, [512] * 16, 384 << 20),
    (16, 8, [1] * 128, [17] * 128, 384 << 20),                 # as many rows as slots
    (16, 8, [5] * 4, [8 * 16 * 128 // 4 - 16] * 4, 384 << 20),  # the longest short plan
    (16, 8, [5], [4096], 2 << 20),                             # little room for partials
])
@pytest.mark.parametrize("per_head", [False, True])
def test_short_plans_cut_rows_by_themselves(hq, hkv, q_len, kv_len, float_ws, per_head):
    lay = layout(waves_per_cu=4, float_ws=float_ws)
    reps = hkv if per_head else 1
    qo, kvl = np.cumsum([0] + q_len), np.repeat(kv_len, reps)
    kvp = np.cumsum(np.concatenate([[0], (kvl + 15) // 16]))
    buf, info = plan(lay, qo, kvp, kvl, hq, hkv, per_head=per_head)
    check_cover(lay, buf, info, qo, kvp, kvl, hq, hkv, per_head=per_head)
    items = [(ip, it[it[:, 5] > it[:, 4]], it) for ip, it in decode(lay, buf, info)[0]]
    held = np.zeros(lay.num_waves, dtype=int)
    for ip, _, it in items:
        for w in range(lay.num_waves):
            held[w] += int((it[ip[w] : ip[w + 1], 5] > it[ip[w] : ip[w + 1], 4]).sum())
    assert held.max() <= 1, "a wave holds pieces of two rows"
    # a row's pieces are even, and no longer than the longest piece length
    for _, it, _ in items:
        for key in {tuple(r) for r in it[:, [0, 6]].tolist()}:
            n = [r[5] - r[4] for r in it.tolist() if (r[0], r[6]) == key]
            assert max(n) - min(n) <= 1 and max(n) <= 12


@pytest.mark.parametrize("hq,hkv", [(32, 8), (8, 8), (64, 2)])
@pytest.mark.parametrize("causal", [1, 0])
@pytest.mark.parametrize("q_len,kv_len,max_slots", [
    ([64], [16064], 500), ([17, 0, 700, 300], [8000, 0, 9000, 300], 500), ([64], [16064], 20), ([8192], [8192], 500),
    ([1], [1], 500), ([0], [0], 500), ([5], [3], 500), ([300] * 40, [5000] * 40, 500)])
def test_prefill_units_cover_every_step_once(hq, hkv, causal, q_len, kv_len, max_slots):
    """Every query block's steps [0, steps) are in exactly one piece each, the last piece open-ended; the
    partial slots of a cut block are consecutive and belong to it alone; no more slots than allowed."""
    import ctypes

    import torch

    from aspire_amd import _lib

    lib = _lib.lib()
    ql, kl = torch.tensor(q_len, dtype=torch.int32), torch.tensor(kv_len, dtype=torch.int32)
    n = [ctypes.c_int32() for _ in range(3)]

    def plan(out, size):
        rc = lib.aspire_prefill_plan(_lib.ptr(ql), _lib.ptr(kl), len(q_len), hq, hkv, causal, max_slots, _lib.ptr(out), size,
                                     *(ctypes.byref(x) for x in n))
        return rc

    assert plan(None, 0) == 0
    units, merges, slots = (x.value for x in n)
    out = torch.full((units + merges + 1, 4), -7, dtype=torch.int32)
    assert plan(out, 4 * (units + merges)) == 0 and (out[-1] == -7).all()
    if units:
        assert plan(out, 4 * (units + merges) - 1) == _lib.ASPIRE_ERR_INVALID  # nothing written past a short buffer
    bt = lib.aspire_prefill_block_tokens(hq, hkv)
    steps = []
    for q, k in zip(q_len, kv_len):
        for t0 in range(0, q, bt):
            keys = min(k - q + min(t0 + bt, q), k) if causal else k
            steps.append((max(-(-keys // 16), 0) + 1) // 2)
    assert slots <= max_slots
    pieces = {}
    for blk, begin, end, slot in out[:units].tolist():
        pieces.setdefault(blk, []).append((begin, end, slot))
    assert sorted(pieces) == list(range(len(steps)))
    merge_of = {blk: (first, count) for blk, first, count, _ in out[units : units + merges].tolist()}
    used = []
    for blk, got in pieces.items():
        got.sort()
        assert got[0][0] == 0 and got[-1][1] == 0x7FFFFFFF
        assert all(a[1] == b[0] and a[0] < a[1] for a, b in zip(got, got[1:])) and got[-1][0] <= max(steps[blk] - 1, 0)
        if len(got) == 1:
            assert got[0][2] == -1 and blk not in merge_of
        else:
            first, count = merge_of[blk]
            assert count == len(got) and [p[2] for p in got] == list(range(first, first + count))
            used += [p[2] for p in got]
    assert sorted(used) == list(range(slots)) and len(merge_of) == merges


def test_prefill_run_units_of_a_batch_without_queries_needs_no_units():
    lib = _lib.lib()
    a = _lib.PrefillArgs()
    a.num_qo_heads, a.num_kv_heads, a.head_dim, a.page_size, a.sm_scale = 32, 8, 128, 16, 1.0
    a.block_tokens, a.num_rows, a.total_blocks = lib.aspire_prefill_block_tokens(32, 8), 2, 0
    a.cache_stride_t, a.cache_stride_p = 1024, 32768
    none = None, 0, None, 0, 0, None, 0, None
    assert lib.aspire_prefill_run_units(ctypes.byref(a), *none) == 0
    a.total_blocks = 1
    assert lib.aspire_prefill_run_units(ctypes.byref(a), *none) == _lib.ASPIRE_ERR_INVALID


@pytest.mark.parametrize("hq,hkv,t,p,want", [
    (32, 8, [8192], [0], (256, 0, 0)), (32, 8, [2048], [0], (64, 0, 0)), (32, 8, [512], [4096], (64, 16, 64)),
    (32, 8, [64], [16000], (64, 2, 64)), (32, 8, [17, 400, 700, 90, 333], [300, 8000, 4000, 2000, 900], (98, 35, 83)),
    (64, 2, [1000] * 8, [2000] * 8, (2000, 0, 0)), (8, 8, [300] * 32, [3000] * 32, (96, 0, 0)),
    (32, 8, [1] * 64, [9000] * 64, (128, 64, 128))])
def test_prefill_plan_skips_no_piece_length_that_is_better(hq, hkv, t, p, want):
    """Units, merges and slots that the estimate of every piece length chooses: lengths that are passed over because
    they cannot be better, and whole blocks that are not estimated, change none of it."""
    import torch

    ql = torch.tensor(t, dtype=torch.int32)
    kl = ql + torch.tensor(p, dtype=torch.int32)
    n = torch.zeros(3, dtype=torch.int32)
    at = [n.data_ptr() + 4 * i for i in range(3)]
    assert _lib.lib().aspire_prefill_plan(_lib.ptr(ql), _lib.ptr(kl), len(t), hq, hkv, 1, 508, None, 0, *at) == 0
    assert tuple(n.tolist()) == want
