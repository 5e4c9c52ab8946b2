"""Decode walks at the edges of a wave's chunk of 64 tiles: a wave looks its
tiles up 64 at a time, requests each tile while the one before it is used,
and runs on from one chunk into the next.  Page counts around one tile per
wave, one and two chunks, mixed over the heads of one launch, against a
float32 restatement of the softmax over the listed tokens
(cvsa/kernels/sparse_decode.py:76-124)."""
import pytest
import torch

from cvsa import ops
from cvsa.ops import _lib
from cvsa.synthetic import jitter_query, make_paged_inputs

pytestmark = pytest.mark.gpu

# Four waves share a workgroup's pages: 4 * 64 pages are one chunk each.
COUNTS = (0, 1, 3, 4, 5, 8, 255, 256, 257, 260, 261, 511, 512, 513, 516, 520)


def _reference(q, k, v, bt, pages, ctx, b, h, G, bs):
    """(o, m, l, sum p |v|) of one KV head over the tokens of `pages`."""
    tok = (pages[:, None] * bs + torch.arange(bs, device=q.device)).reshape(-1)
    rows = bt[b, pages].long()
    K = k[rows, :, h].reshape(-1, k.shape[3])[tok < ctx].float()
    V = v[rows, :, h].reshape(-1, k.shape[3])[tok < ctx].float()
    Q = q[b, h * G:(h + 1) * G].float()
    s = (Q @ K.t().contiguous()) * k.shape[3] ** -0.5
    m = s.amax(1)
    p = torch.exp(s - m[:, None])
    return p @ V, m, p.sum(1), p @ V.abs()


@pytest.mark.parametrize("B,H,G,D,bs", [(64, 4, 4, 128, 16), (128, 2, 1, 64, 16),
                                        (64, 4, 7, 128, 32), (64, 4, 2, 256, 16),
                                        (32, 8, 8, 128, 8), (64, 4, 3, 32, 64)])
def test_walks_across_chunks(gpu, B, H, G, D, bs):
    """256 heads, so a listed head's pages all lie in one workgroup; the
    listed decode, a verified launch with every other head rejected and the
    dense decode."""
    g = torch.Generator(device=gpu)
    g.manual_seed(B + D + bs)
    tiles = max(1, bs // 16)
    W = -(-max(COUNTS) // tiles)
    nb = 96  # pages share blocks: only the walk's order matters here
    shape = (nb, bs, H, D)
    k = torch.randn(shape, generator=g, device=gpu).to(torch.bfloat16)
    v = torch.randn(shape, generator=g, device=gpu).to(torch.bfloat16)
    q = torch.randn(B, H * G, D, generator=g, device=gpu).to(torch.bfloat16)
    bt = torch.randint(nb, (B, W), generator=g, device=gpu, dtype=torch.int32)
    ctx = torch.full((B,), W * bs, dtype=torch.int32, device=gpu)
    ctx[1::3] -= bs // 2 + 1  # a partial last page
    ctx[2] = max(1, bs // 2)
    nv = (ctx + bs - 1) // bs
    n = torch.tensor([-(-c // tiles) for c in COUNTS], device=gpu).repeat(B * H // 16)
    n = torch.minimum(n[:B * H].view(B, H), nv[:, None]).to(torch.int32)
    order = torch.rand(B, H, W, generator=g, device=gpu)
    order = order.masked_fill(torch.arange(W, device=gpu) >= nv[:, None, None], 2.0)
    idx = order.argsort(-1).to(torch.int32).contiguous()
    acc = (torch.arange(B * H, device=gpu) % 2 == 0).view(B, H)
    args = (q, k, v, bt)
    listed = ops.sparse_decode_unnorm(*args, idx, n, ctx, H, G, bs)
    _, ver = ops.verified_decode(*args, ctx, idx, n, acc, H, G, bs, return_state=True)
    _, dense = ops.dense_decode(*args, ctx, H, G, bs, return_state=True)
    cl, cn = ctx.tolist(), n.tolist()
    for b in range(0, B, 3):
        for h in range(H):
            every = torch.arange(nv[b].item(), device=gpu)
            sel = idx[b, h, :cn[b][h]].long()
            full = _reference(q, k, v, bt, every, cl[b], b, h, G, bs)
            part = _reference(q, k, v, bt, sel, cl[b], b, h, G, bs) if cn[b][h] else None
            for got, want in ((listed, part), (ver, part if acc[b, h] else full),
                              (dense, full)):
                o, m, l = (t[b, h * G:(h + 1) * G] for t in got)
                if want is None:  # no page: (0, -inf, 0)
                    assert not o.any() and not l.any() and bool((m == -float("inf")).all())
                    continue
                # P is held to 16 mantissa bits and a score to ~1e-6 of |s| <= 8:
                # each product is off by at most 2^-16 + 1e-5 of itself.
                assert bool(((o - want[0]).abs() <= 4e-5 * want[3] + 1e-6).all()), (b, h)
                assert torch.allclose(m, want[1], rtol=0, atol=2e-5), (b, h)
                assert torch.allclose(l, want[2], rtol=4e-5), (b, h)


@pytest.mark.parametrize("B,H,G,D", [(64, 4, 4, 128), (32, 8, 5, 32), (64, 4, 16, 64),
                                     (64, 4, 2, 256), (128, 2, 1, 128)])
def test_walks_of_8_token_pages(gpu, B, H, G, D):
    """The 8-row tiles' engines: more tiles in flight (1 at D = 256, 8 at
    D = 32) and K and V tiles whose upper half no load writes.  A walk before
    each one leaves infinities in the LDS that they start from."""
    shape = (8, 16, H, D)
    inf = torch.full(shape, float("inf"), device=gpu, dtype=torch.bfloat16)
    q = torch.ones(B, H * G, D, device=gpu, dtype=torch.bfloat16)
    bt = torch.zeros(B, 8, device=gpu, dtype=torch.int32)
    ctx = torch.full((B,), 128, device=gpu, dtype=torch.int32)
    ops.dense_decode(q, inf, inf, bt, ctx, H, G, 16, return_state=True)
    test_walks_across_chunks(gpu, B, H, G, D, 8)


def _whole_head_batch(gpu, ctx, G, max_pages):
    """256 heads of up to 301 pages: one workgroup walks a head, 76 tiles a wave."""
    return make_paged_inputs(32, 8 * G, 8, 128, ctx, seed=5, device=gpu, max_pages=max_pages,
                             spare_blocks=64)


def test_folded_append_across_chunks(gpu):
    """The appended token's page at the edges of a wave's chunks (tiles 0, 63,
    64 and the last of waves 0 and 3), mid-page and on a page that the append
    allocates: bit for bit the append followed by the listed decode."""
    B, H, G, last = 32, 8, 4, 300
    ctx = [16 * last + (0, 5, 15)[b % 3] for b in range(B)]
    inp = _whole_head_batch(gpu, ctx, G, last + 1)
    alloc = torch.tensor([-(-c // 16) for c in ctx], dtype=torch.int32, device=gpu)
    g = torch.Generator().manual_seed(9)
    pi = torch.zeros(B, H, last + 1, dtype=torch.int32)
    nph = torch.zeros(B, H, dtype=torch.int32)
    places = (0, 3, 252, 255, 256, 259, -1, None)  # entry that lists the new page
    for b in range(B):
        for h in range(H):
            at, n = places[(b + h) % 8], last + 1 - (b + 3 * h) % 4
            pages = torch.randperm(last, generator=g)[:n - (at is not None)].tolist()
            if at is not None:
                pages.insert(len(pages) if at < 0 else at, last)
            pi[b, h, :len(pages)] = torch.tensor(pages)
            nph[b, h] = len(pages)
    pi, nph = pi.to(gpu), nph.to(gpu)
    kn, vn = (torch.randn(B, H, 128, generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    slots, fresh = [], inp.used_blocks
    for c in ctx:
        slots += [c, fresh if c % 16 == 0 else -1]
        fresh += c % 16 == 0
    state = [inp.k_cache.clone(), inp.v_cache.clone(), inp.block_tables.clone(),
             inp.context_lens.clone(), alloc.clone()]
    out = ops.sparse_decode_append(inp.q, *state[:4], pi, nph, kn, vn, state[4], slots, H, G, 16)
    ref = [inp.k_cache, inp.v_cache, inp.block_tables, inp.context_lens, alloc]
    ops.append_kv(kn, vn, *ref, 0, inp.used_blocks, 16)
    want = ops.sparse_decode(inp.q, ref[0], ref[1], ref[2], pi, nph, ref[3], H, G, 16)
    assert torch.equal(out, want)
    assert all(torch.equal(a, b) for a, b in zip(state, ref))


@pytest.mark.parametrize("predict,tau", [(1, 0.0), (2, 1.5)])
def test_walk_scores_across_chunks(gpu, predict, tau):
    """Page scores written by the walks of a fused check (the kept selection's
    and the dense one) whose waves run over several chunks: bit for bit the
    page scoring's, and the check that of a plan without speculation."""
    H, G, budget = 8, 2, 290
    ctx = [16 * 300 - (b * 7) % 40 for b in range(32)]
    inp = _whole_head_batch(gpu, ctx, G, 300)
    ctx, bt = inp.context_lens, inp.block_tables
    ps = ops.score_pages(inp.q, inp.k_cache, bt, ctx, H, G, 16)
    sel, nph = ops.select_topk(ps, budget, ctx, 16)
    q = jitter_query(inp.q, 0.5, 3)
    plans = [ops.StepPlan(inp.q, inp.k_cache, inp.v_cache, bt, ctx, H, G, 16, budget, tau,
                          sel.clone(), nph.clone(), speculate=s) for s in (True, False)]
    plans[0].spec_state[0] = predict
    got, want = (p.run(_lib.STEP_LAZY_CHECK, q) for p in plans)
    assert plans[0].spec_state.tolist() == [predict, predict]
    assert torch.equal(plans[0].page_scores, ops.score_pages(q, inp.k_cache, bt, ctx, H, G, 16))
    assert torch.equal(got, want)
    assert torch.equal(plans[0].accept, plans[1].accept)
    assert torch.equal(plans[0].page_indices, plans[1].page_indices)
