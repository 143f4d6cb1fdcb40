"""Plans over query blocks (bsx_attn_plan_t.block_batch > 0: causal host plans whose longest
request has more query rows per kv head than a workgroup holds), against the fp32 oracle
and with the fused KV update against the two calls: block edges (one row past a block, a
block that does not fill its tokens, GQA groups that do not divide it), requests of one
block beside long ones, empty requests, requests with fewer kv than query tokens, both
head dims and types, pages of 16 and 64.  Tolerances are those of tests/attn_parity.py."""
import sys

import numpy as np
import pytest
import torch

import batchspec_amd as bsx
from batchspec_amd.workloads import make_verify_batch
from tests import attn_parity as AP

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# (query heads, kv heads, head dim, page size, dtype, query tokens, cached tokens)
CASES = [
    (32, 8, 128, 16, torch.bfloat16, [65, 64, 5, 1, 129], [0, 31, 700, 33, 2000]),
    (28, 4, 128, 16, torch.bfloat16, [128, 37, 36, 5, 0, 1], [300, 0, 64, 3000, 50, 5000]),
    (32, 4, 64, 64, torch.float16, [100, 1, 33, 512], [1000, 9000, 0, 17]),
    (16, 16, 64, 16, torch.float16, [257, 300, 2], [0, 100, 40]),
    (64, 8, 128, 16, torch.bfloat16, [200, 40, 8], [-150, -7, 500]),  # kv < query tokens
    (8, 1, 128, 16, torch.bfloat16, [2000], [6000]),
    # blocks of 21 tokens (126 of 128 rows): two and a rest, one more than two, exactly one
    (12, 2, 128, 32, torch.bfloat16, [86, 43, 21], [0, 5, 200]),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_query_blocks(case):
    hq, hkv, d, ps, dtype, qo, ctx = CASES[case]
    print(f"query blocks: {hq}/{hkv} D={d} pages of {ps} {dtype} qo={qo} ctx={ctx}", flush=True)
    sys.stdout.flush()
    b = make_verify_batch(len(qo), 0, 0, 0, hq, hkv, d, ps, dtype=dtype, scale=0.5,
                          seed=70 + case, qo_lens=np.array(qo), ctx=np.array(ctx), device=DEV)
    w = bsx.BatchPrefillWithPagedKVCacheWrapper(
        torch.empty(256 << 20, dtype=torch.uint8, device=DEV), "NHD")
    w.plan(b.qo_indptr, b.kv_indptr, b.kv_indices, b.kv_last_page_len, hq, hkv, d, ps,
           causal=True, q_data_type=dtype)
    assert w.plan_info.block_batch > len([q for q in qo if q])
    two, one = b.cache.clone(), b.cache.clone()
    bsx.append_kv(b.k_new, b.v_new, b.qo_indptr, two, b.kv_indptr, b.kv_indices,
                  b.kv_last_page_len)
    out, lse = w.run(b.q, two, return_lse=True)
    out1, lse1 = w.run(b.q, one, return_lse=True, append_key=b.k_new, append_value=b.v_new)
    torch.cuda.synchronize()
    assert torch.equal(one, two) and torch.equal(out, out1) and torch.equal(lse, lse1)
    b.cache = two
    ref = AP.oracle_per_request(b, "causal")[None]
    AP.check(out, ref[0], lse, ref[1])


def test_small_workspace_keeps_the_plan_over_requests():
    """A workspace too small for a block plan's partials still takes the plan it took
    without blocks."""
    b = make_verify_batch(1, 0, 0, 0, 32, 8, 128, 16, dtype=torch.bfloat16, scale=0.5, seed=5,
                          qo_lens=np.array([80]), ctx=np.array([4000]), device=DEV)
    args = (b.qo_indptr, b.kv_indptr, b.kv_indices, b.kv_last_page_len, 32, 8, 128, 16)
    big = bsx.BatchPrefillWithPagedKVCacheWrapper(
        torch.empty(256 << 20, dtype=torch.uint8, device=DEV), "NHD")
    big.plan(*args, causal=True, q_data_type=b.q.dtype)
    assert big.plan_info.block_batch > 0
    need = big._blob_bytes + int(big.plan_info.float_ws_bytes)
    small = bsx.BatchPrefillWithPagedKVCacheWrapper(
        torch.empty(need - 1, dtype=torch.uint8, device=DEV), "NHD")
    small.plan(*args, causal=True, q_data_type=b.q.dtype)
    assert small.plan_info.block_batch == 0
    out = small.run(b.q, b.cache)
    ref = AP.oracle_per_request(b, "causal")[None]
    AP.check(out, ref[0])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_exact_workspace_cache_pair_and_strided_q(dtype):
    """A block plan whose partials fill its workspace to the last byte, on separate K and V
    caches, with queries that are a slice of a wider tensor and appended rows with a token
    stride of their own, against the plain call in a large workspace."""
    hq, hkv, d = 32, 8, 128
    b = make_verify_batch(3, 0, 0, 0, hq, hkv, d, 16, dtype=dtype, scale=0.5, seed=51,
                          qo_lens=np.array([128, 80, 5]), ctx=np.array([965, 2158, 1782]),
                          device=DEV)
    args = (b.qo_indptr, b.kv_indptr, b.kv_indices, b.kv_last_page_len, hq, hkv, d, 16)
    big = bsx.BatchPrefillWithPagedKVCacheWrapper(
        torch.empty(256 << 20, dtype=torch.uint8, device=DEV), "NHD")
    big.plan(*args, causal=True, q_data_type=dtype)
    p = big.plan_info
    assert p.block_batch > 0 and p.num_split_requests > 0
    cache = b.cache.clone()
    out, lse = big.run(b.q, cache, return_lse=True, append_key=b.k_new, append_value=b.v_new)
    need = big._blob_bytes + int(p.float_ws_bytes)
    guard = 4096
    ws = torch.full((need + guard,), 0x5A, dtype=torch.uint8, device=DEV)
    exact = bsx.BatchPrefillWithPagedKVCacheWrapper(ws[:need], "NHD")
    exact.plan(*args, causal=True, q_data_type=dtype)
    assert exact.plan_info.block_batch == p.block_batch
    n = b.q.shape[0]
    wide = torch.zeros((n, hq + 2 * hkv, d), dtype=dtype, device=DEV)  # q, k and v of a layer
    wide[:, :hq], wide[:, hq:hq + hkv], wide[:, hq + hkv:] = b.q, b.k_new, b.v_new
    kv = (b.cache[:, 0].contiguous(), b.cache[:, 1].contiguous())
    out1, lse1 = exact.run(wide[:, :hq], kv, return_lse=True, append_key=wide[:, hq:hq + hkv],
                           append_value=wide[:, hq + hkv:])
    torch.cuda.synchronize()
    assert torch.equal(out1, out) and torch.equal(lse1, lse)
    assert torch.equal(kv[0], cache[:, 0]) and torch.equal(kv[1], cache[:, 1])
    assert bool((ws[need:] == 0x5A).all())
    b.cache = cache
    ref = AP.oracle_per_request(b, "causal")[None]
    AP.check(out, ref[0], lse, ref[1])


def _exact64(b, r):
    """float64 output [qo_len, heads, D] of request r (causal)."""
    q0, q1 = int(b.qo_indptr[r]), int(b.qo_indptr[r + 1])
    pages = b.kv_indices[int(b.kv_indptr[r]):int(b.kv_indptr[r + 1])].long()
    L, n, g = int(b.kv_lens[r]), q1 - q0, b.num_qo_heads // b.num_kv_heads
    kv = b.cache[pages]
    seen = torch.arange(L, device=DEV) <= torch.arange(n, device=DEV)[:, None, None] + L - n
    out = torch.empty((n, b.num_qo_heads, b.head_dim), dtype=torch.float64, device=DEV)
    for h in range(b.num_kv_heads):
        k = kv[:, 0, :, h].reshape(-1, b.head_dim)[:L].double()
        v = kv[:, 1, :, h].reshape(-1, b.head_dim)[:L].double()
        q = b.q[q0:q1, h * g:(h + 1) * g].double().reshape(n * g, b.head_dim)
        s = (q @ k.t().contiguous() / b.head_dim ** 0.5).reshape(n, g, L)
        p = torch.softmax(s.masked_fill(~seen, -torch.inf), -1).reshape(n * g, L)
        out[:, h * g:(h + 1) * g] = (p @ v).reshape(n, g, b.head_dim)
    return out


@pytest.mark.parametrize("n,qo,ctx,split_there", [(1, 2100, 0, 0), (4, 160, 3000, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_split_blocks_lose_no_precision(dtype, n, qo, ctx, split_there):
    """Query tokens of split blocks, where the plan over requests runs their request whole and
    where it splits it too: the error against 64 bits is no larger than that plan's.  fp32 parts
    add roundings of 2^-24 to an output rounded to 2^-9 or 2^-12; the bound leaves 2% for the
    softmax weights' rounding, which falls differently (a second rounding to the 16-bit
    type makes it about 1.2 times)."""
    b = make_verify_batch(n, 0, 0, 0, 32, 8, 128, 16, dtype=dtype, scale=0.5, seed=41,
                          qo_lens=np.full(n, qo), ctx=np.full(n, ctx), device=DEV)
    args = (b.qo_indptr, b.kv_indptr, b.kv_indices, b.kv_last_page_len, 32, 8, 128, 16)

    def planned(nbytes):
        w = bsx.BatchPrefillWithPagedKVCacheWrapper(
            torch.empty(nbytes, dtype=torch.uint8, device=DEV), "NHD")
        w.plan(*args, causal=True, q_data_type=dtype)
        return w

    blocks = planned(256 << 20)
    p = blocks.plan_info
    assert p.block_batch > 0 and p.num_split_requests > 0
    whole = planned(blocks._blob_bytes + int(p.float_ws_bytes) - 1)  # no room for the partials
    assert whole.plan_info.block_batch == 0
    assert whole.plan_info.num_split_requests == split_there
    rec = blocks.plan_blob[p.off_merge_seqs:p.off_merge_seqs + 4 * p.num_split_requests]
    split = torch.zeros(b.q.shape[0], dtype=torch.bool, device=DEV)
    for _, _, q0, ql in rec.reshape(-1, 4):
        split[int(q0):int(q0) + int(ql)] = True
    ref = torch.cat([_exact64(b, r) for r in range(n)])[split]
    err = [float((w.run(b.q, b.cache).double()[split] - ref).norm() / ref.norm())
           for w in (whole, blocks)]
    print(f"split query tokens {int(split.sum())} of {len(split)}: relative error whole "
          f"{err[0]:.6f}, blocks {err[1]:.6f}", flush=True)
    assert err[1] <= 1.02 * err[0]


def test_whole_blocks_equal_the_plan_over_requests():
    """Chunks that neither plan splits: the same tiles in the same order, so the outputs of the
    two plans are the same bits."""
    b = make_verify_batch(4, 0, 0, 0, 32, 8, 128, 16, dtype=torch.bfloat16, scale=0.5, seed=42,
                          qo_lens=np.full(4, 512), ctx=np.full(4, 1024), device=DEV)
    args = (b.qo_indptr, b.kv_indptr, b.kv_indices, b.kv_last_page_len, 32, 8, 128, 16)
    res = []
    for graph in (False, True):  # graph mode keeps a record per request
        kw = dict(use_cuda_graph=True, paged_kv_indices_buf=b.kv_indices.clone()) if graph else {}
        w = bsx.BatchPrefillWithPagedKVCacheWrapper(
            torch.empty(256 << 20, dtype=torch.uint8, device=DEV), "NHD", **kw)
        w.plan(*args, causal=True, q_data_type=b.q.dtype)
        assert (w.plan_info.block_batch == 0) == graph
        n_seg = int(w.plan_blob[w.plan_info.off_seg_indptr + w.plan_info.num_ctas])
        assert n_seg == (4 if graph else w.plan_info.block_batch)
        res.append(w.run(b.q, b.cache, return_lse=True))
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])
