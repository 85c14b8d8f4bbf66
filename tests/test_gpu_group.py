"""Clean-commit token grouping on the GPU (ssa_group_order) against the
float64 oracle (oracle/group.py) on identical seeded inputs: two layers x 12
heads batched in one call, the plain order, the first chunk's frame re-sort
and a non-identity page order.  Both run in float64, so the orders must agree
token for token."""
import pytest
import torch

from oracle import group as og
from streaming_sparse_amd import group, workload

pytestmark = pytest.mark.gpu


def inputs(seed, layers=2, heads=12):
    g = torch.Generator().manual_seed(workload.seed_for(4, 0, 0, 40 + seed))
    k = torch.randn(layers, 4608, heads, 128, generator=g)
    v = torch.randn(layers, 4608, heads, 128, generator=g)
    freqs = workload.rope_table(128)
    k = torch.stack([workload.apply_rope(k[l], 3, freqs) for l in range(layers)])
    return k.bfloat16(), v.bfloat16()


@pytest.mark.parametrize("first_chunk,history", [(False, 360), (True, 360), (False, 338)])
def test_group_order_matches_oracle(device, first_chunk, history):
    k, v = inputs(0)
    w = group.GroupWeights.seeded(2, 12, 5, device)
    pd = group.page_destinations(history)
    got = group.order(k.to(device), v.to(device), w, first_chunk=first_chunk, page_dst=pd).cpu()
    pages = og.page_order(history)
    for layer in range(2):
        want = og.group_order(k[layer].transpose(0, 1), v[layer].transpose(0, 1), w.bank[layer].cpu(),
                              w.group_v[layer].cpu(), w.gate[layer].cpu(), pages=pages, first_chunk=first_chunk)
        same = (got[layer] == want).all(-1)
        print(f"layer {layer} first_chunk={first_chunk} history={history}: {int(same.sum())}/12 heads identical",
              flush=True)
        assert torch.equal(got[layer].long(), want)


@pytest.mark.parametrize("scale,offset", [(1.0, 0.0), (1.0, 48.0), (12.0, 0.0)])
def test_group_order_one_row(device, scale, offset):
    """One layer and head (the smallest batch), and the statistics that are
    merged over token blocks where they could cancel: keys far from zero, and
    scores of standard deviation 12, whose softmax leaves a few tokens."""
    gen = torch.Generator().manual_seed(int(scale + offset))
    k = (scale * torch.randn(1, 4608, 1, 128, generator=gen) + offset).bfloat16()
    v = torch.randn(1, 4608, 1, 128, generator=gen).bfloat16()
    w = group.GroupWeights.seeded(1, 1, 7, torch.device("cpu"))
    g = group.GroupWeights(*(t.to(device) for t in (w.bank, w.group_v, w.gate)))
    got = group.order(k.to(device), v.to(device), g).cpu()
    want = og.group_order(k[0].transpose(0, 1), v[0].transpose(0, 1), w.bank[0], w.group_v[0], w.gate[0])
    assert torch.equal(got[0].long(), want)


@pytest.mark.parametrize("distinct", [1, 7, 512])
def test_group_order_is_stable_on_duplicates(device, distinct):
    """Equal tokens have equal projections at every level, so the stable
    sorts keep them in token order, through every merge of sorted runs; with
    one distinct token every direction is zero and the order is the
    identity."""
    gen = torch.Generator().manual_seed(distinct)
    rows = torch.randint(0, distinct, (4608,), generator=gen)
    k = torch.randn(distinct, 2, 128, generator=gen).bfloat16()[rows][None].contiguous()
    v = torch.randn(distinct, 2, 128, generator=gen).bfloat16()[rows][None].contiguous()
    w = group.GroupWeights.seeded(1, 2, 8, device)
    got = group.order(k.to(device), v.to(device), w).cpu().long()
    for h in range(2):
        assert torch.equal(got[0, h].sort().values, torch.arange(4608))
        for r in range(distinct):
            mine = got[0, h][rows[got[0, h]] == r]
            assert bool((mine[1:] > mine[:-1]).all())
    if distinct == 1:
        assert torch.equal(got[0, 0], torch.arange(4608))
