"""Sampling and acceptance calls issued at the same time from two streams, and from two host
threads on one stream, over different inputs: each result equals the one of the same call
issued alone.  (The calls pass intermediate results between their kernels through a cached
workspace.)"""
import threading

import pytest
import torch

from batchspec_amd import sampling as S
from batchspec_amd.posterior import evaluate_posterior

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
B, K, V, REPS = 24, 4, 32000, 12


def _inputs(seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = (torch.randn((B, K + 1, V), generator=g, device=DEV) * 3).to(torch.bfloat16)
    d = (x[:, :K].float() + 0.5 * torch.randn((B, K, V), generator=g, device=DEV)).to(x.dtype)
    u = torch.rand((B, K + 1), generator=g, device=DEV)
    return x, d, d.float().argmax(-1), u


CALLS = {
    "sample": lambda x, d, i, u: [S.sample(x, 0.95, 0, 0.8, uniforms=u)],
    "sampling": lambda x, d, i, u: evaluate_posterior(
        i, x, greedy=False, eos_token_id=2, temperature=0.8, top_k=20, top_p=0.95, uniforms=u),
    "greedy": lambda x, d, i, u: evaluate_posterior(i, x, greedy=True, eos_token_id=2),
    "chain": lambda x, d, i, u: S.chain_speculative_sampling_from_logits(d, i, x, 0.8, uniforms=u),
    "chain_top_p": lambda x, d, i, u: S.chain_speculative_sampling_from_logits(
        d, i, x, 0.8, uniforms=u, top_p=0.9),
    "probs": lambda x, d, i, u: [S.get_sampling_probs(x, 0.9, 0, 0.8)],
}


@pytest.mark.parametrize("how", ["streams", "threads"])
@pytest.mark.parametrize("name", sorted(CALLS))
def test_concurrent_calls(name, how):
    print(f"concurrent {name} over two {how}", flush=True)
    call = CALLS[name]
    data = [_inputs(3), _inputs(4)]
    want = [[t.clone() for t in call(*d)] for d in data]
    torch.cuda.synchronize()
    got = [[], []]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    if how == "streams":
        for _ in range(REPS):
            for n in range(2):
                with torch.cuda.stream(streams[n]):
                    got[n].append(call(*data[n]))
    else:
        start = threading.Barrier(2)

        def work(n):
            start.wait(timeout=30)
            with torch.cuda.stream(streams[0]):
                for _ in range(REPS):
                    got[n].append(call(*data[n]))

        threads = [threading.Thread(target=work, args=(n,)) for n in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join(timeout=60)
            assert not t.is_alive()
    torch.cuda.synchronize()
    for n in range(2):
        assert len(got[n]) == REPS
        for res in got[n]:
            assert all(torch.equal(a, b) for a, b in zip(res, want[n]))
