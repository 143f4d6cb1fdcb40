"""Top-p alone over few rows, each row split over several workgroups
(csrc/filter_nucleus.h), bit for bit against the CPU oracle: sample(), the chain and
get_sampling_probs.  The edges: the row counts where the number of workgroups per row
changes (128, 256, 512), the shortest vocabulary of the path and the one below it, rows of
which a canonical thread has 7, 8 and 9 whole rounds, a last partial group (fp32, V mod 8 =
4), rows that are not 16-byte aligned, more than eight elements per draw lane; ties, rows
whose threshold lies outside the bf16 key window (around zero, or in a row of two values),
all-negative rows, -inf padding, and nearly certain rows.  Rows and temperatures outside the
statistics' domain (+inf, all -inf, scores past 2^31) give what the path with one workgroup
per row gives (more than 512 rows); rows with a NaN, which have no distribution, give an id
of the vocabulary or -1."""
import numpy as np
import pytest
import torch

from batchspec_amd import sampling as S
from oracle import accept as OAc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _rows(kind, rows, V, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn((rows, V), generator=g)
    if kind == "peaked":
        x = x * 2
        x[:, :40] += torch.rand((rows, 40), generator=g) * 14
    elif kind == "flat":
        x = x * 2
    elif kind == "zero":  # the nucleus reaches below 0: past the window of bf16 keys
        x = x * 0.3
    elif kind == "negative":
        x = -20 + x
    elif kind == "ties":
        x = torch.round(x) * 2
    elif kind == "two":
        x = torch.where(torch.rand((rows, V), generator=g) < 0.5, 1.0, 1000.0)
    elif kind == "certain":
        x = x - 30
        x[:, V // 3] = 20.0
    elif kind == "padded":
        x = x * 2
        x[:, V // 2:] = float("-inf")
    return x.to(dtype)


SAMPLE = [
    ("bf16", "peaked", 5, 16384, 0.95), ("bf16", "peaked", 5, 16383, 0.95),
    ("bf16", "flat", 3, 16383 * 2, 0.9), ("bf16", "flat", 2, 8 * 2048 * 9 + 16, 0.95),
    ("bf16", "zero", 3, 20000, 0.9), ("bf16", "negative", 3, 20000, 0.9),
    ("bf16", "ties", 3, 20000, 0.7), ("bf16", "two", 2, 16384, 0.5),
    ("bf16", "certain", 3, 20000, 0.95), ("bf16", "padded", 3, 32000, 0.95),
    ("bf16", "peaked", 2, 1100000, 0.95), ("bf16", "flat", 129, 16392, 0.95),
    ("bf16", "flat", 128, 16384, 0.5), ("bf16", "peaked", 257, 16384, 0.95),
    ("bf16", "peaked", 513, 16384, 0.95),
    ("fp16", "flat", 4, 20000, 0.95), ("fp16", "zero", 3, 20000, 0.9),
    ("fp16", "ties", 3, 20001, 0.7), ("fp16", "peaked", 130, 16384, 0.9),
    ("fp32", "flat", 4, 20004, 0.95), ("fp32", "two", 2, 16384, 0.5),
    ("fp32", "padded", 3, 20001, 0.9), ("fp32", "negative", 260, 16388, 0.99),
]


@pytest.mark.parametrize("dt,kind,rows,V,top_p", SAMPLE)
def test_sample(dt, kind, rows, V, top_p):
    print(f"nucleus sample {dt} {kind} rows={rows} V={V} top_p={top_p}", flush=True)
    x = _rows(kind, rows, V, DT[dt], rows + V)
    u = np.random.default_rng(V).random(rows, dtype=np.float32)
    u[0], u[-1] = 0.0, np.float32(1 - 2 ** -24)
    ref = OAc.sample(x.float().numpy(), 0.8, 0, top_p, u)
    got = S.sample(x.to(DEV)[:, None], top_p, 0, 0.8, uniforms=torch.from_numpy(u).to(DEV))
    assert got.dtype == torch.int64
    np.testing.assert_array_equal(got.cpu().numpy().reshape(-1), ref)


@pytest.mark.parametrize("dt,kind,B,k,V", [("bf16", "peaked", 7, 3, 20000),
                                           ("bf16", "zero", 3, 2, 20000),
                                           ("fp16", "flat", 4, 2, 16384),
                                           ("fp32", "ties", 4, 2, 16388)])
@pytest.mark.parametrize("onehot", [True, False])
def test_chain_and_probs(dt, kind, B, k, V, onehot):
    print(f"nucleus chain {dt} {kind} B={B} k={k} V={V} onehot={onehot}", flush=True)
    t = _rows(kind, B * (k + 1), V, DT[dt], 3 + V).reshape(B, k + 1, V)
    d = (t[:, :k].float() + 0.25 * torch.round(2 * torch.rand(B, k, V))).to(DT[dt])
    ids = d.float().argmax(-1)
    u = torch.rand((B, k + 1), generator=torch.Generator().manual_seed(1)) * 0.7
    ref = OAc.chain_filtered(None if onehot else d.float().numpy(), ids.numpy(),
                             t.float().numpy(), 0.7, 0, 0.9, u.numpy())
    got = S.chain_speculative_sampling_from_logits(
        None if onehot else d.to(DEV), ids.to(DEV), t.to(DEV), 0.7, uniforms=u.to(DEV), top_p=0.9)
    for g, r in zip(got, ref):
        np.testing.assert_array_equal(g.cpu().numpy(), r)
    p = S.get_sampling_probs(t.to(DEV), 0.9, 0, 0.7).cpu().numpy().reshape(-1, V)
    want = OAc.filtered_probs(t.float().numpy().reshape(-1, V), 0.7, 0, 0.9)
    np.testing.assert_array_equal(p, want.reshape(-1, V))


SPECIAL = ["one +inf", "many +inf", "one nan", "all nan", "all -inf", "+inf and nan", "-inf but one",
           "lowest", "plain"]


def _special_rows(V, dtype):
    g = torch.Generator().manual_seed(V)
    x = torch.randn((len(SPECIAL), V), generator=g) * 2
    x[0, 7] = float("inf")
    x[1, 3::1000] = float("inf")
    x[2, V - 1] = float("nan")
    x[3] = float("nan")
    x[4] = float("-inf")
    x[5, 100], x[5, 200] = float("nan"), float("inf")
    x[6] = float("-inf")
    x[6, V // 2] = 1.0
    x = x.to(dtype)
    x[7] = torch.finfo(dtype).min  # a mask of the type's lowest value
    x[7, 5:9] = 1.0
    return x


@pytest.mark.parametrize("temperature", [0.8, 1e-9, 1e-30, 1e-38])
@pytest.mark.parametrize("V", [20000, 20001])
@pytest.mark.parametrize("dt", sorted(DT))
def test_rows_outside_the_domain(dt, V, temperature):
    print(f"nucleus special rows {dt} V={V} T={temperature}", flush=True)
    x = _special_rows(V, DT[dt]).to(DEV)
    n = len(SPECIAL)
    rest = torch.zeros((513 - n, V), dtype=x.dtype, device=DEV)
    rest[:, 0] = 9.0
    more = torch.cat([x, rest])  # too many rows for the split path
    u = torch.rand(513, generator=torch.Generator().manual_seed(5)).to(DEV)
    nan = torch.tensor(["nan" in kind for kind in SPECIAL], device=DEV)
    for top_p in (0.5, 0.95):
        many = S.sample(more[:, None], top_p, 0, temperature, uniforms=u)[:n]
        few = S.sample(x[:, None], top_p, 0, temperature, uniforms=u[:n].clone())
        assert torch.equal(few[~nan], many[~nan]), (few.flatten().tolist(), many.flatten().tolist())
        assert bool(((few >= -1) & (few < V)).all())
        pm = S.get_sampling_probs(more[:, None], top_p, 0, temperature)[:n][~nan]
        pf = S.get_sampling_probs(x[:, None], top_p, 0, temperature)[~nan]
        assert torch.equal(pf.isnan(), pm.isnan())
        assert torch.equal(pf.nan_to_num(nan=-1.0), pm.nan_to_num(nan=-1.0))
