"""The work that is timed: single calls of the page-sparse attention path
through the package's public entry points, over the sizes a stream meets.

A stream of 3-frame chunks (24 pages of 64 tokens per frame) runs, per layer
and denoise step, one call of 12 heads x 72 query blocks against a window that
grows from 72 pages (the first chunk) to 432 (history + the current chunk); a
rank of a head-sharded run holds fewer heads, and a caller may hand over one
frame or any number of query blocks.  Q, K and V are N(0, 1) with Wan RoPE on
Q and K, rounded to bf16; summaries come from a 4-iteration k-means of each
page's keys, the basis from the page-centred V.

``exact`` forms the same results in float64 with plain torch.
"""
from __future__ import annotations

import math

import torch

from streaming_sparse_amd import group, pset, summary, workload
from streaming_sparse_amd.attention import Workspace
from streaming_sparse_amd.legacy_components import REP_OP_ELEMS, attention, rep_operands, rep_tiles
from streaming_sparse_amd.ops import Summary
from streaming_sparse_amd.route import route, tier_count

DEV = 'cuda'
D = 128
ANCHORS, CURRENT = 24, 72
BASE_PAGES = 168             # shortest window whose base table (15% of the pages) holds own and every anchor
PROBES = (0, 4, 8, 13, 17, 21, 25, 29, 34, 38, 42, 46, 50, 55, 59, 63)
HAAR = ((1, 1, -1, -1), (1, -1, 1, -1), (1, -1, -1, 1))
FULL_PSET = (3, 4, 9)        # the heads a 12-head layer corrects
READER = workload.reader_weights(3)


def listed():
    return [
        # the smallest call: one frame's queries, one head, the shortest window whose base table holds every anchor
        dict(name='attend_frame_p168', kind='attend', heads=1, blocks=24, pages=168, tier='base', n=0, single=False),
        # a rank holding 2 of the 12 heads, half-full window
        dict(name='attend_rank_p216', kind='attend', heads=2, blocks=72, pages=216, tier='base', n=0, single=False),
        # odd sizes: a window that is no multiple of a rep tile, an odd number of blocks and heads
        dict(name='attend_quota_p301', kind='attend', heads=5, blocks=37, pages=301, tier='intersection', n=41,
             single=False),
        # the ordinary call of the base tier at the full window
        dict(name='attend_base_p432', kind='attend', heads=12, blocks=72, pages=432, tier='base', n=0, single=False),
        # the same window with quota tables, callers that opt into one bf16 product
        dict(name='attend_single_p432', kind='attend', heads=12, blocks=72, pages=432, tier='intersection', n=41,
             single=True),
        # the first chunk's layers: every page exact, window = the chunk itself
        dict(name='dense_p72', kind='dense', heads=12, blocks=72, pages=72),
        # layer 0 and the clean step at the full window: every page exact
        dict(name='dense_p432', kind='dense', heads=12, blocks=72, pages=432),
        # the router of the base tier with the attention's operand tiles on the side
        dict(name='route_base_p432', kind='route', heads=12, blocks=72, pages=432, tier='base', n=0),
        # a Full_Pset layer's page table: current encodings, quota router, swap correction of 3 heads
        dict(name='correct_p432', kind='correct', heads=12, blocks=72, pages=432, n=41, scoped=3),
        # the current chunk's rows into the window and their summaries, at every denoise step
        dict(name='summarise_p72', kind='summarise', heads=12, pages=72),
        # a sparse layer of a denoise step, whole: window write and summaries, quota router, attention
        dict(name='layer_p432', kind='layer', heads=12, blocks=72, pages=432, n=41),
        # the commit's token grouping over a 30-layer stack
        dict(name='group_l30', kind='group', layers=30, heads=12, first=False),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(('attend', 'attend', 'attend', 'dense', 'route', 'correct', 'summarise', 'layer', 'group'))
    heads = _log(rng, 1, 12)
    if kind == 'attend':
        tier = rng.choice(('base', 'intersection'))
        pages = rng.randint(BASE_PAGES if tier == 'base' else 97, 480)
        return dict(kind=kind, heads=heads, blocks=_log(rng, 4, 72), pages=pages, tier=tier,
                    n=0 if tier == 'base' else rng.randint(4, min(56, pages - ANCHORS)), single=rng.random() < 0.3)
    if kind == 'dense':
        return dict(kind=kind, heads=heads, blocks=_log(rng, 4, 72), pages=_log(rng, 24, 432))
    if kind == 'route':
        tier = rng.choice(('base', 'intersection'))
        pages = rng.randint(BASE_PAGES if tier == 'base' else 97, 480)
        return dict(kind=kind, heads=heads, blocks=_log(rng, 4, 72), pages=pages, tier=tier,
                    n=0 if tier == 'base' else rng.randint(4, min(56, pages - ANCHORS)))
    if kind == 'correct':
        return dict(kind=kind, heads=heads, blocks=CURRENT, pages=rng.randint(100, 480), n=rng.randint(8, 56),
                    scoped=rng.randint(1, min(3, heads)))
    if kind == 'summarise':
        return dict(kind=kind, heads=heads, pages=_log(rng, 8, 432))
    if kind == 'layer':
        return dict(kind=kind, heads=heads, blocks=CURRENT, pages=rng.randint(120, 480), n=rng.randint(8, 56))
    return dict(kind=kind, layers=_log(rng, 1, 30), heads=heads, first=rng.random() < 0.3)


# ---------------------------------------------------------------- inputs ----

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


_FREQS = []


def _rope(x, first_page):
    """Wan RoPE of [L, H, D] rows that start at page `first_page`."""
    if not _FREQS:
        _FREQS.append(workload.rope_table(D).to(torch.complex64).to(DEV))
    L, H, _ = x.shape
    c = D // 2
    ch = c // 3
    ft, fh, fw = _FREQS[0].split([c - 2 * ch, ch, ch], dim=1)
    tok = torch.arange(L, device=DEV) + 64 * first_page
    i = tok % workload.TOKENS_PER_FRAME
    f = torch.cat([ft[tok // workload.TOKENS_PER_FRAME], fh[i // workload.GRID_W], fw[i % workload.GRID_W]], 1)
    z = torch.view_as_complex(x.reshape(L, H, c, 2).contiguous())
    return torch.view_as_real(z * f[:, None]).reshape(L, H, D)


def _rows(g, tokens, heads, first_page=None):
    """bf16 rows [tokens, H, D]; with first_page, rotated."""
    x = _randn(g, tokens, heads, D)
    return (x if first_page is None else _rope(x, first_page)).to(torch.bfloat16).contiguous()


def _basis(v, heads):
    """Per-head top-8 directions of page-centred V ([L, H, D]), [H, D, 8] bf16."""
    x = v.float().reshape(-1, 64, heads, D).permute(2, 0, 1, 3)
    x = (x - x.mean(2, keepdim=True)).reshape(heads, -1, D)
    cov = torch.bmm(x.transpose(1, 2).contiguous(), x).double().cpu()
    vec = torch.linalg.eigh(cov)[1][..., -8:].flip(-1)
    sign = torch.sign(vec.gather(1, vec.abs().argmax(1, keepdim=True)))
    return (vec * sign).to(torch.bfloat16).to(DEV).contiguous()


def _init(g, heads, pages):
    return torch.rand(heads * pages, 64, generator=g, device=DEV).argsort(-1)[:, :4].reshape(heads, pages, 4) \
        .to(torch.int32).contiguous()


def _summaries(k, v, basis, init, dtype, iters=4):
    """Summary fields of the pages of k, v [L, H, D] in `dtype`, unrounded
    where the stored field is an end result (the reps that later statistics
    are taken against are the stored bf16 ones)."""
    H, P = init.shape[:2]

    def bf(x):
        return x.to(torch.bfloat16).to(dtype)

    kb = k.reshape(P, 64, H, D).permute(2, 0, 1, 3).reshape(H * P, 64, D).to(dtype)
    vb = v.reshape(P, 64, H, D).permute(2, 0, 1, 3).reshape(H * P, 64, D).to(dtype)
    bas = basis.to(dtype).repeat_interleave(P, 0)
    cent = kb.gather(1, init.long().reshape(-1, 4, 1).expand(-1, -1, D))
    for _ in range(iters):
        dist = torch.stack([(kb - cent[:, r:r + 1]).square().sum(-1) for r in range(4)], -1)
        one = torch.nn.functional.one_hot(dist.argmin(-1), 4).to(dtype)
        cnt = one.sum(1)[..., None]
        sums = torch.bmm(one.transpose(1, 2).contiguous(), kb)
        cent = torch.where(cnt > 0, sums / cnt.clamp_min(1), cent)
    vmean = vb.mean(1)
    vm = torch.where(cnt > 0, torch.bmm(one.transpose(1, 2).contiguous(), vb) / cnt.clamp_min(1), vmean[:, None])
    keys = cent - cent.mean(1, keepdim=True) + kb.mean(1, keepdim=True)
    ha = torch.tensor(HAAR, dtype=dtype, device=DEV)
    detail = torch.matmul(ha, torch.bmm(vm, bas)) / 4
    pk, mu, det = bf(keys), bf(vmean), bf(detail)
    recon = mu[:, None] + torch.bmm(torch.matmul(ha.t(), det), bas.transpose(1, 2).contiguous())
    stats = torch.zeros(H * P, 4, 12, dtype=dtype, device=DEV)
    for r in range(4):
        w = one[..., r]
        n = cnt[:, r].clamp_min(1)
        var = (w[..., None] * (kb - cent[:, r:r + 1]).square()).sum(1) / n
        stats[:, r, :8] = var.reshape(-1, 8, 16).mean(-1)
        stats[:, r, 10] = ((w * (vb - vm[:, r:r + 1]).square().sum(-1)).sum(1) / n[:, 0]).sqrt()
    stats[..., 8] = (cent - pk).norm(dim=-1)
    stats[..., 9] = (vm - recon).norm(dim=-1)
    stats[:, 0, 11] = (vmean - mu).norm(dim=-1)
    stats[:, 1, 11] = vb.norm(dim=-1).amax(1)
    return (keys.reshape(H, P, 4, D), vmean.reshape(H, P, D), detail.reshape(H, P, 3, 8),
            stats.reshape(H, P, 4, 12))


def _summary(k, v, basis, init):
    return Summary(*(x.to(torch.bfloat16).contiguous() for x in _summaries(k, v, basis, init, torch.float32)))


def _window(g, heads, blocks, pages):
    q = _rows(g, 64 * blocks, heads, max(0, pages - blocks))
    return q, _rows(g, 64 * pages, heads, 0), _rows(g, 64 * pages, heads)


def _own(heads, blocks, pages):
    return (torch.arange(blocks, device=DEV) + pages - blocks).clamp_min(0).expand(heads, -1)


def _quota(g, heads, n, pages):
    """A per head: current-chunk pages of a quota n = A + B."""
    lo, hi = max(min(4, n), n - 40), min(36, n)
    return torch.randint(lo, hi + 1, (heads,), generator=g, device=DEV).to(torch.int32)


def _risk(q, keys, stats, dtype):
    """Page risk [H, T, P] of the 16 probe rows of each query block, and the
    probes' log-sum-exp [H, T, 16]."""
    n, H, _ = q.shape
    T, P = n // 64, keys.shape[1]
    pr = q.reshape(T, 64, H, D).permute(2, 0, 1, 3)[:, :, list(PROBES)].to(dtype).reshape(H, T * 16, D)
    st = stats.to(dtype)
    z = torch.bmm(pr, keys.to(dtype).reshape(H, 4 * P, D).transpose(1, 2).contiguous()) / math.sqrt(D)
    lse = z.logsumexp(-1)
    prob = (z - lse[..., None]).exp().reshape(H, T * 16, P, 4)
    q2 = pr.square().reshape(H, T * 16, 8, 16).sum(-1) / D
    qn = pr.norm(dim=-1) / math.sqrt(D)
    u = torch.bmm(q2, st[..., :8].reshape(H, 4 * P, 8).transpose(1, 2).contiguous()).clamp_min(0)
    u = u.reshape(H, T * 16, P, 4)
    beta = qn[..., None, None] * st[:, None, :, :, 8]
    bp = st[:, :, 1, 11]
    c = (bp + bp.amax(-1, keepdim=True))[:, None]
    alpha = prob.sum(-1)
    x0 = alpha * st[:, None, :, 0, 11] + ((prob - alpha[..., None] / 4).abs() * st[:, None, :, :, 9]).sum(-1)
    x1 = (prob * u.sqrt() * st[:, None, :, :, 10]).sum(-1)
    x2 = c * (prob * beta).sum(-1)
    x3 = c * (prob * (u + beta.square())).sum(-1)
    value = x0 + x1 + x2 + 0.5 * x3
    return value.reshape(H, T, 16, P).mean(2), lse.reshape(H, T, 16)


def _top(scores, slots):
    return scores.sort(dim=-1, descending=True, stable=True).indices[..., :max(0, slots)]


def _table(risk, own, tier, n, quota):
    """(ids, mask) of the base tier or of the quota tier."""
    H, T, P = risk.shape
    count = tier_count(tier, P, n)
    page = torch.arange(P, device=DEV)
    if tier == 'base':
        order = _top(risk.masked_fill((page < ANCHORS) | (page == own[..., None]), -torch.inf), count - 1 - ANCHORS)
        ids = torch.cat([own[..., None], page[:ANCHORS].expand(H, T, -1), order], -1)
        return ids.int().contiguous(), torch.zeros_like(risk, dtype=torch.bool).scatter(-1, ids, True)
    mask = torch.zeros_like(risk, dtype=torch.bool)
    mask[..., :ANCHORS] = True
    ranked = risk.scatter(-1, own[..., None], torch.inf)
    for h in range(H):
        a = int(quota[h])
        mask[h].scatter_(-1, _top(risk[h, :, ANCHORS:P - CURRENT], n - a) + ANCHORS, True)
        mask[h].scatter_(-1, _top(ranked[h, :, P - CURRENT:], a) + (P - CURRENT), True)
    score, ids = ranked.masked_fill(~mask & (page != own[..., None]), -torch.inf) \
        .sort(dim=-1, descending=True, stable=True)
    ids = ids[..., :count].int().masked_fill(score[..., :count] == -torch.inf, -1)
    return ids.contiguous(), mask


# ------------------------------------------------------------------ cases ----

def _make(case, seed):
    """The inputs of a case as a dict of tensors, from the seed alone."""
    g = _gen(seed)
    kind, H = case['kind'], case['heads']
    if kind == 'group':
        L = case['layers']
        k = torch.empty(L, 4608, H, D, device=DEV, dtype=torch.bfloat16)
        v = torch.empty_like(k)
        for i in range(L):
            k[i], v[i] = _rows(g, 4608, H, 288), _rows(g, 4608, H)
        bank = _randn(g, L, H, 32, D)
        gv = torch.nn.functional.normalize(bank, dim=-1).transpose(-1, -2).contiguous()
        return dict(k=k, v=v, bank=bank, group_v=gv, gate=0.1 + 0.05 * _randn(g, L, H, 32))
    P = case['pages']
    if kind == 'summarise':
        # 24 pages of history before the pages that are written
        k, v = _rows(g, 64 * (P + ANCHORS), H, 0), _rows(g, 64 * (P + ANCHORS), H)
        return dict(k=k, v=v, src=(_rows(g, 64 * P, H, ANCHORS), _rows(g, 64 * P, H)), basis=_basis(v, H),
                    init=_init(g, H, P))
    q, k, v = _window(g, H, case['blocks'], P)
    if kind == 'dense':
        return dict(q=q, k=k, v=v, basis=_basis(v, H))
    basis = _basis(v, H)
    x = dict(q=q, k=k, v=v, basis=basis, summary=_summary(k, v, basis, _init(g, H, P)),
             quota=_quota(g, H, case['n'], P), own=_own(H, case['blocks'], P))
    if kind == 'attend':
        risk, _ = _risk(q, x['summary'].keys, x['summary'].stats, torch.float32)
        x['ids'], _ = _table(risk, x['own'], case['tier'], case['n'], x['quota'])
    if kind == 'layer':
        x['src'] = (_rows(g, 64 * CURRENT, H, P - CURRENT), _rows(g, 64 * CURRENT, H))
        x['init'] = _init(g, H, CURRENT)
    return x


def prepare(case, seed):
    x = _make(case, seed)
    kind, H = case['kind'], case['heads']
    x['case'] = case
    x['ws'] = Workspace()
    x['theta'] = torch.tensor([1.0, 1.0, 1.0, 0.5], device=DEV).expand(H, 4).contiguous()
    for name in ('q', 'k', 'v'):
        if name in x and kind != 'group':
            x[name] = x[name][None]
    if kind == 'group':
        x['weights'] = group.GroupWeights(x['bank'], x['group_v'], x['gate'])
        return x
    P = case['pages']
    if kind == 'summarise':
        cap = P + ANCHORS
        x['slab'] = Summary(*(torch.zeros(H, cap, *inner, device=DEV, dtype=torch.bfloat16)
                              for inner in ((4, D), (D,), (3, 8), (4, 12))))
    if kind == 'dense':
        # a dense call reads neither summaries nor the table
        x['summary'] = Summary(*(torch.zeros(H, P, *inner, device=DEV, dtype=torch.bfloat16)
                                 for inner in ((4, D), (D,), (3, 8), (4, 12))))
        own = _own(H, case['blocks'], P)[0] % P
        x['ids'] = ((torch.arange(P, device=DEV) + own[:, None]) % P).int().expand(H, -1, -1).contiguous()
    if kind in ('route', 'layer', 'attend'):
        x['ops'] = torch.zeros(H, rep_tiles(P), REP_OP_ELEMS, device=DEV, dtype=torch.bfloat16)
    if kind == 'attend':
        rep_operands(x['summary'], P, x['ops'])
    if kind == 'correct':
        x['reader'] = pset.Reader(READER, DEV)
        x['encoding'] = pset.encode(x['summary'], x['basis'], x['reader'])
        x['scoped'] = FULL_PSET[:case['scoped']] if H == 12 else tuple(range(case['scoped']))
    return x


def _fields(s, first=0):
    return {f: getattr(s, f)[:, first:] for f in Summary.FIELDS}


def run(state):
    x = state
    case = x['case']
    kind = case['kind']
    if kind == 'attend':
        return attention(x['q'], x['k'], x['v'], x['summary'], x['basis'], x['ids'], x['ws'], rep_ops=x['ops'],
                         single_av=case['single'])
    if kind == 'dense':
        return attention(x['q'], x['k'], x['v'], x['summary'], x['basis'], x['ids'], x['ws'], all_pages=True,
                         single_av=True)
    if kind == 'route':
        ids, mask, risk, _ = route(x['q'], x['summary'], x['theta'], tier=case['tier'], n=case['n'],
                                   current_slots=None if case['tier'] == 'base' else x['quota'],
                                   workspace=x['ws'], rep_out=x['ops'])
        return dict(ids=ids, mask=mask, risk=risk, ops=x['ops'])
    if kind == 'correct':
        P = case['pages']
        e = pset.encode(x['summary'], x['basis'], x['reader'], out=x['encoding'], first=P - CURRENT, pages=CURRENT)
        ids, mask, risk, _ = route(x['q'], x['summary'], x['theta'], tier='intersection', n=case['n'],
                                   current_slots=x['quota'], workspace=x['ws'], full_pset=x['scoped'], encoding=e,
                                   reader=x['reader'])
        return dict(ids=ids, mask=mask, risk=risk, coef=e.coef, mean=e.mean, detail=e.detail)
    if kind == 'summarise':
        P = case['pages']
        summary.build(x['k'], x['v'], x['basis'], x['init'], x['slab'], ANCHORS, P, src=x['src'])
        return dict(_fields(x['slab'], ANCHORS), k=x['k'][:, 64 * ANCHORS:], v=x['v'][:, 64 * ANCHORS:])
    if kind == 'layer':
        P = case['pages']
        s = x['summary']
        summary.build(x['k'], x['v'], x['basis'], x['init'], s, P - CURRENT, CURRENT, src=x['src'])
        ids, _, risk, _ = route(x['q'], s, x['theta'], tier='intersection', n=case['n'], current_slots=x['quota'],
                                workspace=x['ws'], want_mask=False, rep_out=x['ops'])
        out = attention(x['q'], x['k'], x['v'], s, x['basis'], ids, x['ws'], rep_ops=x['ops'])
        return dict(_fields(s, P - CURRENT), out=out, risk=risk)
    return group.order(x['k'], x['v'], x['weights'], first_chunk=case['first'], workspace=x['ws'])


# -------------------------------------------------------------- what it is ----

def _attend_work(H, T, P, C):
    n = 64 * T
    pages = min(P, T * C)
    flops = 4.0 * n * H * D * 64 * C
    byte = 2 * n * H * D * 2 + 2 * pages * 64 * H * D * 2 + H * T * C * 4
    if C < P:
        flops += n * H * (2 * D * 4 * P + 2 * P * D + 6 * P * 8 + 16 * D)
        byte += H * P * (5 * D + 24) * 2
    return byte, flops


def _route_work(H, T, P, C):
    byte = H * T * 16 * D * 2 + H * P * (4 * D + 48 + 24) * 2 + H * T * (P * 5 + C * 4) + H * P * 64
    return byte, 2.0 * H * 16 * T * 4 * P * D + 30.0 * H * 16 * T * 4 * P


def _summary_work(H, P, write):
    byte = H * P * (2 * 64 * D * 2 * (2 if write else 1) + (5 * D + 72) * 2)
    return byte, H * P * (4 * 64 * 4 * 3 * D + 2 * 64 * 4 * D + 6 * 64 * D)


def work(case):
    kind, H = case['kind'], case['heads']
    if kind == 'group':
        B = case['layers'] * H
        return dict(bytes=B * 4608 * (2 * D * 2 + 4),
                    flops=B * 4608 * (2.0 * 64 * D + 7 * 4 * 4 * 32))
    P = case['pages']
    if kind == 'dense':
        b, f = _attend_work(H, case['blocks'], P, P)
    elif kind == 'attend':
        b, f = _attend_work(H, case['blocks'], P, tier_count(case['tier'], P, case['n']))
    elif kind == 'route':
        b, f = _route_work(H, case['blocks'], P, tier_count(case['tier'], P, case['n']))
    elif kind == 'summarise':
        b, f = _summary_work(H, P, True)
    elif kind == 'correct':
        b, f = _route_work(H, case['blocks'], P, ANCHORS + case['n'])
        rows = case['scoped'] * case['blocks']
        # encodings of the current pages; readout and candidate scores of the scoped rows
        b += H * CURRENT * (712 * 2 + 256 + 64 * 8) + case['scoped'] * P * (256 + 64 * 8)
        f += H * CURRENT * 2.0 * (712 * 512 + 256 * 117) + rows * 16 * (P * 400.0 + 512 * 100)
    else:
        b, f = 0, 0.0
        for x, y in (_summary_work(H, CURRENT, True), _route_work(H, CURRENT, P, ANCHORS + case['n']),
                     _attend_work(H, CURRENT, P, ANCHORS + case['n'])):
            b, f = b + x, f + y
    return dict(bytes=b, flops=f)


def tolerance(case):
    """bf16 outputs carry a relative rounding error of 1.7e-3 (2-norm); the
    single-product arithmetic adds 2.5e-3.  Risks are 32-bit sums whose
    near-ties order the tables."""
    kind = case['kind']
    if kind == 'attend':
        return dict(rel=1.2e-2 if case['single'] else 6.5e-3, max=0.1)
    if kind == 'dense':
        return dict(rel=1.2e-2, max=0.1)
    if kind == 'route':
        return dict(rel=1e-5, max=1e-4, differ=5e-3)
    if kind == 'correct':
        return dict(rel=6.5e-3, max=0.05, differ=5e-3)
    if kind == 'summarise':
        return dict(rel=6.5e-3, max=0.05)
    if kind == 'layer':
        return dict(rel=6.5e-3, max=0.1)
    return dict(rel=0.0, differ=1e-4)      # an order of tokens by float64 projections: only their last bits may tie


# ------------------------------------------------------------------ exact ----

def _attend_exact(q, k, v, s, basis, ids):
    """One softmax over the listed pages' tokens and the 4 reps (16 tokens
    each) of every page that is not listed; q [N, H, D], k, v [L, H, D]."""
    n, H, _ = q.shape
    T, P = n // 64, k.shape[0] // 64
    kk = k.transpose(0, 1).double().contiguous()
    vv = v.transpose(0, 1).double().contiguous()
    reps, means = s[0].double().reshape(H, 4 * P, D), s[1].double()
    ha = torch.tensor(HAAR, dtype=torch.float64, device=DEV)
    # value of rep r of page p: mean + sum_a HAAR[a, r] detail_a . basis^T
    code = torch.einsum('ar,hpak->hprk', ha, s[2].double())
    val = means[:, :, None] + torch.matmul(code, basis.double().transpose(1, 2)[:, None].contiguous())
    val = val.reshape(H, 4 * P, D)
    keys_t, reps_t = kk.transpose(1, 2).contiguous(), reps.transpose(1, 2).contiguous()
    tok = torch.arange(64, device=DEV)
    out = torch.empty(n, H, D, dtype=torch.float64, device=DEV)
    for t in range(T):
        sel = ids[:, t].long()
        ok = sel >= 0
        col = torch.where(ok, sel, P)
        used = torch.zeros(H, P + 1, dtype=torch.bool, device=DEV).scatter(1, col, True)[:, :P]
        idx = (sel.clamp_min(0)[:, :, None] * 64 + tok).flatten(1)
        qt = q[64 * t:64 * t + 64].transpose(0, 1).double().contiguous()
        ke = keys_t.gather(2, idx[:, None].expand(-1, D, -1))
        z = torch.bmm(qt, ke) / math.sqrt(D)
        z = z.masked_fill(~ok.repeat_interleave(64, 1)[:, None], -torch.inf)
        zr = torch.bmm(qt, reps_t) / math.sqrt(D) + math.log(16)
        zr = zr.masked_fill(used.repeat_interleave(4, 1)[:, None], -torch.inf)
        w = torch.cat([z, zr], -1).softmax(-1)
        ve = vv.gather(1, idx[:, :, None].expand(-1, -1, D))
        o = torch.bmm(w[..., :z.shape[-1]].contiguous(), ve) + torch.bmm(w[..., z.shape[-1]:].contiguous(), val)
        out[64 * t:64 * t + 64] = o.transpose(0, 1)
    return out[None]


def _dense_exact(q, k, v):
    n, H, _ = q.shape
    kt = k.permute(1, 2, 0).double().contiguous()
    vv = v.transpose(0, 1).double().contiguous()
    out = torch.empty(n, H, D, dtype=torch.float64, device=DEV)
    for a in range(0, n, 256):
        z = torch.bmm(q[a:a + 256].transpose(0, 1).double().contiguous(), kt) / math.sqrt(D)
        out[a:a + 256] = torch.bmm(z.softmax(-1), vv).transpose(0, 1)
    return out[None]


def _encode_exact(x):
    s = x['summary']
    w = {k: t.to(DEV).double() for k, t in READER.items()}
    parts = [s.keys.double().flatten(2), s.mean.double(), s.detail.double().flatten(2), s.stats.double().flatten(2)]
    f = torch.cat([p / (p.square().mean(-1, keepdim=True).sqrt() + 1e-4) for p in parts], -1)

    def mlp(name):
        y = torch.nn.functional.linear(f, w[name + '_w1'], w[name + '_b1'])
        return torch.nn.functional.linear(torch.nn.functional.gelu(y), w[name + '_w2'], w[name + '_b2'])

    co, a = mlp('reader'), mlp('phi')
    coef = torch.cat([co, torch.zeros_like(co[..., :11]), a], -1)
    mean = torch.matmul(s.mean.double(), w['B'])
    proj = torch.matmul(x['basis'].double().transpose(1, 2).contiguous(), w['B'])
    return dict(coef=coef, mean=mean, detail=torch.matmul(s.detail.double(), proj[:, None]))


def _group_exact(x, first):
    """The order of group.order: float64 features, then 7 levels of balanced
    splits by a power-iteration direction with stable sorts."""
    L, n, H, _ = x['k'].shape
    out = torch.empty(L, H, n, dtype=torch.int32, device=DEV)
    for i in range(L):
        k = x['k'][i].transpose(0, 1).double()
        v = x['v'][i].transpose(0, 1).double()
        kc = k - k.mean(1, keepdim=True)
        score = torch.bmm(kc.contiguous(), x['bank'][i].double().transpose(1, 2).contiguous()) / math.sqrt(D)
        key = score / score.square().mean((1, 2), keepdim=True).sqrt().clamp_min(1e-6)
        a = score.softmax(1)
        vp = torch.bmm(v.contiguous(), x['group_v'][i].double())
        resp = a * n * (vp - (a * vp).sum(1, keepdim=True))
        resp = resp / resp.square().mean((1, 2), keepdim=True).sqrt().clamp_min(1e-6)
        f = key + 0.1 * x['gate'][i].double().tanh()[:, None] * resp
        ids = torch.arange(n, device=DEV).expand(H, n)
        groups = 1
        for factor in (3, 3, 2, 2, 2, 2, 2):
            size = n // groups
            y = f.reshape(H * groups, size, 32)
            ids = ids.reshape(H * groups, size)
            yc = y - y.mean(1, keepdim=True)
            var = yc.square().mean(1)
            d = torch.zeros_like(var).scatter_(1, var.argmax(-1, keepdim=True), 1.0)
            for _ in range(4):
                d = (yc * (yc * d[:, None]).sum(-1, keepdim=True)).sum(1)
                d = d / d.norm(dim=-1, keepdim=True).clamp_min(1e-8)
            order = (yc * d[:, None]).sum(-1).argsort(dim=-1, stable=True)
            f = y.gather(1, order[:, :, None].expand_as(y))
            ids = ids.gather(1, order)
            groups *= factor
        ids = ids.reshape(H, n)
        if first:
            ids = ids.gather(1, torch.argsort(ids // 1536, dim=1, stable=True))
        out[i] = ids.int()
    return out


def exact(case, seed):
    x = _make(case, seed)
    kind = case['kind']
    if kind == 'group':
        return _group_exact(x, case['first'])
    if kind == 'dense':
        return _dense_exact(x['q'], x['k'], x['v'])
    if kind == 'summarise':
        k, v = x['src']
        s = _summaries(k, v, x['basis'], x['init'], torch.float64)
        return dict(zip(Summary.FIELDS, s), k=k.double()[None], v=v.double()[None])
    s = x['summary']
    if kind == 'attend':
        return _attend_exact(x['q'], x['k'], x['v'], (s.keys, s.mean, s.detail), x['basis'], x['ids'])
    if kind == 'layer':
        P = case['pages']
        k, v = x['src']
        new = _summaries(k, v, x['basis'], x['init'], torch.float64)
        cur = dict(zip(Summary.FIELDS, new))
        # the layer's router and attention read the stored (bf16) summaries
        full = [torch.cat([getattr(s, f)[:, :P - CURRENT], cur[f].to(torch.bfloat16)], 1) for f in Summary.FIELDS]
        risk, _ = _risk(x['q'], full[0], full[3], torch.float64)
        ids, _ = _table(risk, x['own'], 'intersection', case['n'], x['quota'])
        kw = torch.cat([x['k'][:64 * (P - CURRENT)], k])
        vw = torch.cat([x['v'][:64 * (P - CURRENT)], v])
        return dict(cur, out=_attend_exact(x['q'], kw, vw, full[:3], x['basis'], ids), risk=risk)
    risk, _ = _risk(x['q'], s.keys, s.stats, torch.float64)
    if kind == 'route':
        ids, mask = _table(risk, x['own'], case['tier'], case['n'], x['quota'])
        return dict(ids=ids, mask=mask, risk=risk, ops=None)
    # the swaps that the correction makes are whole decisions and have no 64-bit value
    return dict(_encode_exact(x), ids=None, mask=None, risk=risk)
