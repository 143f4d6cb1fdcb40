"""evaluate_posterior's sampling branch (batchspec/backends/mtp_engine.py:569-575): bonus,
accept counts and eos flags written by the kernel that ends a request's chain, against the
same three computed with torch from the chain's output rows, on every path a chain takes
(no filter, top-k in one launch per request, top-k over many rows or positions, top-p alone),
with eos ids that hit accepted drafts, the emitted id, the padding (-1) and nothing."""
import pytest
import torch

from batchspec_amd.posterior import evaluate_posterior
from batchspec_amd.sampling import chain_speculative_sampling_from_logits

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# (B, k, V, dtype, top_k, top_p)
CASES = [
    (9, 4, 20000, torch.bfloat16, 20, 0.95),   # split rows, one launch per request
    (9, 7, 20000, torch.bfloat16, 24, 0.0),    # its largest number of positions
    (5, 8, 20000, torch.float16, 20, 0.95),    # more positions than that
    (120, 5, 17000, torch.bfloat16, 10, 0.9),  # too many rows to split
    (6, 3, 1003, torch.float32, 20, 0.95),     # rows that are not 16-byte aligned
    (7, 3, 20000, torch.bfloat16, 0, 0.9),     # top-p alone
    (8, 3, 3000, torch.bfloat16, 0, 0.0),      # no filter
    (4, 0, 20000, torch.bfloat16, 20, 0.95),   # no draft token
    (0, 3, 3000, torch.bfloat16, 20, 0.95),    # no request
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_sampling_verdict(case):
    B, k, V, dtype, top_k, top_p = CASES[case]
    gen = torch.Generator(device=DEV).manual_seed(40 + case)
    logits = (torch.randn((B, k + 1, V), generator=gen, device=DEV) * 4).to(dtype)
    draft = logits[:, :k].float().argmax(-1) if B else torch.zeros((B, k), device=DEV)
    draft = draft.to(torch.int64)
    u = torch.rand((B, k + 1), generator=gen, device=DEV)
    u[:, 1:k:2] *= 0.1  # some drafts accepted
    out, _, emitted = chain_speculative_sampling_from_logits(
        None, draft, logits, 0.8, uniforms=u, top_k=top_k, top_p=top_p)
    last = (out != -1).long() * torch.arange(k + 1, device=DEV)
    bonus = out.gather(1, last.argmax(dim=1, keepdim=True))
    for eos in {-1, 2, V + 5} | ({int(out[0, 0]), int(out[-1].max())} if B else set()):
        got = evaluate_posterior(draft, logits, greedy=False, eos_token_id=eos, temperature=0.8,
                                 top_p=top_p, top_k=top_k, uniforms=u)
        assert got[0].dtype == torch.int32 and got[1].dtype == torch.int32
        assert torch.equal(got[0], bonus) and torch.equal(got[1], emitted + 1)
        assert torch.equal(got[2], (out == eos).any(dim=1, keepdim=True))


def test_sampling_verdict_other_eos_ids():
    """An eos id that is not a plain integer compares as torch compares it: a tensor of one
    id, a tensor of one id per request, and floats, equal to an id or not."""
    B, k, V = 6, 3, 3000
    gen = torch.Generator(device=DEV).manual_seed(9)
    logits = torch.randn((B, k + 1, V), generator=gen, device=DEV) * 4
    draft = logits[:, :k].argmax(-1)
    u = torch.rand((B, k + 1), generator=gen, device=DEV)
    out, _, emitted = chain_speculative_sampling_from_logits(None, draft, logits, 0.8, uniforms=u)
    hit = int(out[0, 0])
    for eos in (torch.tensor(hit, device=DEV), out[:, :1].clone(), float(hit), hit + 0.5, 1e30):
        got = evaluate_posterior(draft, logits, greedy=False, eos_token_id=eos, temperature=0.8,
                                 uniforms=u)
        assert torch.equal(got[2], (out == eos).any(dim=1, keepdim=True))
        assert torch.equal(got[1], emitted + 1)
        assert got[0].dtype == torch.int32 and got[1].dtype == torch.int32
