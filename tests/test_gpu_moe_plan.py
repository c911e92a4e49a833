"""Grouping of (token, choice) pairs with few and with many experts, with and without a group of all tokens in front; a mixture's weighted sum inside the
residual's launch against the launch of its own."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("n,top,E", [(1, 1, 1), (7, 2, 8), (64, 3, 31), (1000, 2, 32), (513, 4, 33), (4096, 2, 8), (300, 6, 200)])
def test_groups(dev, n, top, E, shared):
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(n + E)
    idx = torch.randint(0, E + 2, (n, top), generator=g).to(torch.int32)      # (the last two are no experts)
    wgt = torch.rand(n, top, generator=g)
    rows = n * top + (n if shared else 0)
    off, tok, row, pw = (torch.full((s,), -7, dtype=dt, device=dev) for s, dt in ((E + 1 + shared, torch.int32), (rows, torch.int32), (n * top, torch.int32), (rows, torch.float32)))
    D.moe_plan(idx.to(dev), n=n, top=top, experts=E, group_off=off, pair_token=tok, pair_row=row, wgt=wgt.to(dev), pair_wgt=pw, shared=shared)
    off, tok, row, pw = off.tolist(), tok.cpu(), row.cpu().view(n, top), pw.cpu()
    if shared:
        assert off[0] == 0 and off[1] == n and tok[:n].tolist() == list(range(n)) and bool((pw[:n] == 1).all())
        off = off[1:]
    assert off[0] == (n if shared else 0)
    seen = set()
    for e in range(E):
        where = (idx == e).nonzero()
        assert off[e + 1] - off[e] == len(where)
        for t, k in where.tolist():
            r = int(row[t, k])
            assert off[e] <= r < off[e + 1] and r not in seen and int(tok[r]) == t and pw[r] == wgt[t, k]
            seen.add(r)
    assert bool((row[idx >= E] == -1).all())


@pytest.mark.parametrize("W", [4, 1000, 2048, 4100])
@pytest.mark.parametrize("top,beside,gated,weighted", [(1, False, False, True), (2, True, True, True), (5, False, True, False), (4, True, False, False)])
def test_sum_inside_the_residual(dev, W, top, beside, gated, weighted):
    from vllm_i64_amd import ops_dense as D
    n = 9
    g = torch.Generator(device=dev).manual_seed(W + top)
    f = lambda *s: torch.randn(*s, generator=g, device=dev)
    x, y, ey, h, sh, sg, wgt, nw, ls = f(1, n, W), f(n, W), f(n * top, W), f(n, W), f(n, W), f(n), f(n, top), f(W), f(W)
    row = torch.randperm(n * top, generator=g, device=dev).to(torch.int32).view(n, top).contiguous()
    row[3, 0] = -1
    one = torch.ones(1, device=dev)
    kw = dict(h=h, shared=sh, top=top, shared_gate=sg if gated else None)
    z = torch.empty(n, W, device=dev)
    D.moe_combine(ey, row, wgt if weighted else None, h, sh, z, n=n, top=top, width=W, shared_gate=kw["shared_gate"])
    outs = []
    for inside in (False, True):
        xs, hn = x.clone(), torch.empty(n, W, device=dev)
        args = dict(out_w=one, norm_w=nw, eps=1e-6, h=hn, y_scale=ls)
        if inside:
            D.streams_step(xs, y=y if beside else None, moe=dict(y=ey, pair_row=row, wgt=wgt if weighted else None, **kw), **args)
        else:
            D.streams_step(xs, **(dict(y=y, y2=z) if beside else dict(y=z)), **args)
        outs.append((xs, hn))
    assert all(torch.equal(a, b) for a, b in zip(*outs))
