"""DeepSeek routing with expert groups of one, two and four lanes and of
parts of lanes, ties and biases of both signs, at token counts around a
block's: indices and counts exact against the oracle's rule on the device's
own scores, weights within fp32 rounding of K terms."""
import pytest
import torch

from moe_amd import ops
from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"

CASES = [
    # T, E, K, groups, kept
    (1, 128, 8, 8, 4), (63, 128, 8, 8, 4), (65, 64, 8, 8, 4), (129, 32, 4, 8, 2),
    (513, 256, 8, 8, 4),   # two lanes per group
    (200, 256, 16, 4, 4),  # four lanes per group
    (300, 128, 8, 4, 2),   # two lanes, K = 8 of G = 8
    (300, 128, 8, 2, 2),   # four lanes
    (300, 128, 8, 1, 1),   # one group of all lanes
    (300, 96, 6, 6, 3),    # groups of parts of lanes
    (8200, 128, 8, 8, 4),
]


@pytest.mark.parametrize("T,E,K,groups,kept", CASES)
def test_grouped_routing(T, E, K, groups, kept):
    print(f"grouped routing T={T} E={E} K={K} groups={groups}/{kept}", flush=True)
    g = torch.Generator().manual_seed(T + E + groups)
    logits = torch.randn(T, E, generator=g).to(DEV)
    logits[::3] = (logits[::3] * 2).round() / 2  # exact ties
    bias = ((torch.rand(E, generator=g) * 2 - 1) * 0.05).to(DEV)
    bias[: E // 2] = 0.0
    counts = torch.zeros(E, device=DEV)
    scores, w, idx = ops.router_sigmoid_topk(logits, bias, K, True, 2.5, groups, kept,
                                             torch.float32, counts)
    torch.cuda.synchronize()
    assert torch.equal(scores, torch.sigmoid(logits))
    # biased scores as the kernel forms them (an fp32 add); scores of a group
    # added best first
    biased = (scores + bias).cpu()
    by = biased.reshape(T, groups, E // groups)
    top = by.sort(dim=-1, descending=True).values[..., : K // kept]
    gs = torch.zeros(T, groups)
    for q in range(K // kept):
        gs = gs + top[..., q]
    _, gi = O.rank_topk(gs, kept)
    mask = torch.zeros(T, groups).scatter_(1, gi, 1.0).bool()
    _, want = O.rank_topk(by.masked_fill(~mask[..., None], float("-inf")).reshape(T, E), K)
    assert torch.equal(idx.cpu(), want)
    assert torch.equal(counts.cpu(), torch.bincount(want.reshape(-1), minlength=E).float())
    v = scores.cpu().double().gather(1, want)
    ref = v / v.sum(-1, keepdim=True) * 2.5
    assert float(((w.cpu().double() - ref).abs() / ref).max()) <= (K + 3) * 2.0 ** -24


@pytest.mark.parametrize("T,E,K,groups,kept", [
    (300, 128, 8, 8, 4), (300, 64, 6, 0, 0), (300, 256, 8, 0, 0),  # lanes per token, vectors
    (300, 100, 8, 0, 0), (300, 96, 6, 6, 3),                       # ... without vectors
    (300, 64, 20, 0, 0), (300, 512, 8, 8, 4),                      # a wave per token
    (300, 320, 8, 0, 0), (300, 1792, 8, 0, 0),                     # a workgroup per token
])
def test_scores_in_the_logits_buffer(T, E, K, groups, kept):
    """scores written over the logits: the same scores, weights and indices."""
    print(f"scores in place T={T} E={E} K={K} groups={groups}/{kept}", flush=True)
    g = torch.Generator().manual_seed(T + E + K)
    logits = torch.randn(T, E, generator=g).to(DEV)
    bias = ((torch.rand(E, generator=g) * 2 - 1) * 0.05).to(DEV)
    want = ops.router_sigmoid_topk(logits, bias, K, True, 2.5, groups or None, kept or None)
    buf, w = logits.clone(), torch.empty(T, K, device=DEV)
    idx = torch.empty(T, K, device=DEV, dtype=torch.int64)
    ops._call("moe_amd_router_sigmoid_topk", buf.data_ptr(), bias.data_ptr(), T, E, K, 1, 2.5, groups,
              kept, buf.data_ptr(), w.data_ptr(), 0, idx.data_ptr(), None, ops._stream(buf))
    torch.cuda.synchronize()
    for a, b in zip((buf, w, idx), want):
        assert torch.equal(a, b)
