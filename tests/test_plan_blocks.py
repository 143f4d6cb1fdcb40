"""Host plans over query blocks (block_batch > 0), on the CPU: the blocks partition every
request's query tokens, each with exactly the kv tokens its last token can see, every tile
of every block is scheduled once, and split blocks' partial rows are packed without
overlap.  Masks and shapes outside the rule keep a record per request, and the C entry
point without a workspace size never needs more workspace than that plan."""
import ctypes
import time

import numpy as np
import pytest

from batchspec_amd import _lib


def _plan(qo, kv, hq, hkv, d=128, ps=16, mode=_lib.MASK_CAUSAL, cus=256, ws=1 << 40):
    L = _lib.load()
    qo, kv = np.asarray(qo), np.asarray(kv)
    qoi = np.concatenate([[0], np.cumsum(qo)]).astype(np.int32)
    pages = -(-kv // ps)
    kvp = np.concatenate([[0], np.cumsum(pages)]).astype(np.int32)
    last = np.where(kv > 0, (kv - 1) % ps + 1, 0).astype(np.int32)
    bound = L.bsx_attn_plan_ints_bound(len(qo), cus)
    blob = np.zeros(bound, np.int32)
    plan = _lib.AttnPlan()
    args = (qoi.ctypes.data, kvp.ctypes.data, last.ctypes.data, len(qo), hq, hkv, d, ps, mode, 0, 0,
            0.0, cus, -1)
    tail = (blob.ctypes.data, bound, ctypes.byref(plan))
    rc = L.bsx_attn_plan(*args, *tail) if ws is None else L.bsx_attn_plan_ws(*args, ws, *tail)
    _lib.check(rc, "plan")
    return plan, blob, qoi, kvp


@pytest.mark.parametrize("hq,hkv,seed", [(32, 8, 0), (28, 4, 1), (64, 8, 2), (32, 32, 3), (12, 2, 4)])
def test_blocks_cover_every_query_token_and_visible_tile(hq, hkv, seed):
    rng = np.random.default_rng(seed)
    qo = rng.choice([0, 1, 5, 64, 65, 300, 700], size=12)
    qo[0] = 700
    kv = np.maximum(0, rng.integers(-20, 3000, size=12) + qo)
    plan, blob, qoi, kvp = _plan(qo, kv, hq, hkv)
    over, obl, _, _ = _plan(qo, kv, hq, hkv, ws=0)  # the plan over requests, if blocks split
    split_there = np.zeros(len(qo), bool)
    if over.block_batch == 0:
        osegs = obl[over.off_segments:over.off_segments + 4 * over.num_segments].reshape(-1, 4)
        split_there[osegs[osegs[:, 3] >= 0, 0]] = True
    assert (over.block_batch > 0) == (plan.num_split_requests == 0)
    g = hq // hkv
    n = plan.block_batch
    assert n > 0
    # the launched workgroups: 4 waves of 32 query rows on one kv head, one per (share, head)
    assert (plan.qrow_tile, plan.qblocks_per_cta, plan.qrow_blocks) == (32, 4, 4)
    assert plan.num_qgroups == 1 and plan.heads_per_cta == 1
    assert plan.num_ctas * hkv <= 2 * 256
    seq = blob[:4 * n].reshape(-1, 4)
    segs = blob[plan.off_segments:plan.off_segments + 4 * plan.num_segments].reshape(-1, 4)
    token_owner = np.zeros(int(qoi[-1]), int)
    for q0, ql, kl, ps0 in seq:
        assert 0 < ql * g <= 4 * 32
        token_owner[q0:q0 + ql] += 1
        r = int(np.searchsorted(qoi, q0, side="right")) - 1
        while qo[r] == 0:
            r -= 1
        assert q0 + ql <= qoi[r + 1] and ps0 == kvp[r]
        # the kv tokens the block's last token sees (bottom-right causal alignment)
        assert kl == max(0, kv[r] - (qoi[r + 1] - (q0 + ql)))
    assert np.all(token_owner == 1)
    rows_used = []
    for i, (_, ql, kl, _) in enumerate(seq):
        mine = segs[segs[:, 0] == i]
        tiles = sorted(t for s in mine for t in range(s[1], s[2]))
        assert tiles == list(range(-(-int(kl) // 32)))
        if len(mine) == 1:
            assert mine[0, 3] == -1
        else:
            r = int(np.searchsorted(qoi, seq[i, 0], side="right")) - 1
            wide = not split_there[r]  # fp32: rounded once in the plan over requests
            for s in mine:
                assert s[3] % 2 == wide
                rows_used += list(range(s[3] // 2, s[3] // 2 + ql * g * (1 + wide)))
    assert sorted(rows_used) == list(range(plan.part_rows))
    assert plan.float_ws_bytes == plan.part_rows * hkv * (128 * 2 + 4)
    rec = blob[plan.off_merge_seqs:plan.off_merge_seqs + 4 * plan.num_split_requests]
    for a, b, q0, n in rec.reshape(-1, 4):
        assert a % 2 == b % 2 and (b - a) // 2 % (n * g * (1 + a % 2)) == 0


def test_rule_and_workspace_fallback():
    qo, kv = [300, 5], [2000, 900]
    blk, _, _, _ = _plan(qo, kv, 32, 8)
    assert blk.block_batch > 0 and blk.shared_kv_tiles == 1
    for mode in (_lib.MASK_NONE, _lib.MASK_CUSTOM):
        assert _plan(qo, kv, 32, 8, mode=mode)[0].block_batch == 0
    assert _plan(qo, kv, 32, 8, ps=8)[0].block_batch == 0      # pages below 16 tokens
    # 64 * 4 query rows: one 8-wave workgroup of the plan over requests holds the longest
    assert _plan([64, 5], kv, 32, 8)[0].block_batch == 0
    whole = _plan(qo, kv, 32, 8, ws=0)[0]
    assert blk.float_ws_bytes == 0 or whole.block_batch == 0
    strict = _plan(qo, kv, 32, 8, ws=None)[0]
    assert strict.block_batch == 0 or strict.float_ws_bytes <= whole.float_ws_bytes


def test_more_blocks_than_the_blob_holds():
    """About 4000 blocks fill the blob of a small batch; from there on the plan keeps a
    record per request, without the time that scheduling the blocks would take."""
    assert _plan([64000], [64000], 64, 8)[0].block_batch == 4000
    for qo in ([65536], [8192] * 8):
        assert _plan(qo, qo, 64, 8)[0].block_batch == 0

    def least(mode):
        times = []
        for _ in range(20):
            t = time.perf_counter()
            _plan([65536], [65536], 64, 8, mode=mode)
            times.append(time.perf_counter() - t)
        return min(times)

    none = least(_lib.MASK_NONE)  # never takes blocks; the same plan otherwise
    assert least(_lib.MASK_CAUSAL) < 2 * none + 1e-4


def test_random_block_plans_fit_the_blob():
    """The bound that admits blocks covers what the schedule then needs, near the limit too."""
    rng = np.random.default_rng(8)
    for _ in range(20):
        n = int(rng.integers(1, 40))
        qo = rng.integers(1, 2 * 64000 // n, size=n)
        kv = qo + rng.integers(0, 5000, size=n)
        p, blob, _, _ = _plan(qo, kv, 64, 8)
        assert p.plan_ints <= len(blob)


def _loads(plan, blob, cost):
    seg = blob[plan.off_seg_indptr:plan.off_seg_indptr + plan.num_ctas + 1]
    recs = blob[plan.off_segments:plan.off_segments + 4 * plan.num_segments].reshape(-1, 4)
    return [sum(max(1, e - t) * cost[r] + 8 for r, t, e, _ in recs[a:b])
            for a, b in zip(seg, seg[1:])]


@pytest.mark.parametrize("qo,ctx,hq,hkv,whole", [
    ([383, 300, 250, 383, 100], [0] * 5, 32, 8, True),   # short: whole blocks are even enough
    ([512] * 4, [1024] * 4, 32, 8, True),
    ([1352, 1100], [512, 0], 40, 8, True),               # several blocks a workgroup
    ([450], [4096], 16, 8, False),                       # few long blocks
    ([128] * 6 + [5] * 30, [3000] * 36, 28, 4, False),
])
def test_blocks_stay_whole_where_splitting_gains_little(qo, ctx, hq, hkv, whole):
    qo = np.array(qo)
    kv = qo + np.array(ctx)
    plan, blob, _, _ = _plan(qo, kv, hq, hkv)
    n = plan.block_batch
    assert n > 0 and (plan.num_split_requests == 0) == whole
    seq = blob[:4 * n].reshape(-1, 4)
    waves = -(-seq[:, 1] * (hq // hkv) // 32)
    cost = np.maximum(2, waves)
    tiles = -(-seq[:, 2] // 32)
    load = np.maximum(1, tiles) * cost + 8
    share = -(-int(load.sum()) // (512 // hkv))
    limit = lambda share: share + share // 4 + 64
    if whole:
        assert plan.float_ws_bytes == 0 and plan.num_segments == n
        assert max(_loads(plan, blob, cost)) <= limit(max(share, 12))
    else:
        assert load.max() > limit(share)
