"""i64h_streams_route: the residual's norm, the choice of experts and (few rows) the plan in one launch, against the three launches."""
import pytest
import torch

from vllm_i64_amd import ops_dense as D

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# rows, width, entries, experts, gate, options
CASES = [
    (1, 4, 1, 1, False, dict()), (7, 1024, 8, 8, True, dict(chosen_softmax=True, biased=True)), (8, 2048, 8, 8, False, dict(sigmoid_scores=True, raw_weights=True)),
    (9, 1028, 16, 12, True, dict(corrected=True, scale=2.5)), (64, 2052, 9, 9, False, dict(sigmoid_scores=True, corrected=True)), (65, 4096, 17, 17, False, dict()),
    (128, 8192, 5, 5, True, dict(chosen_softmax=True)), (129, 1024, 8, 8, False, dict()), (500, 2048, 8, 8, True, dict(biased=True)), (1030, 1024, 16, 16, False, dict(chosen_softmax=True)),
]


@pytest.mark.parametrize("n,W,E,experts,gated,opt", CASES)
def test_one_launch_is_the_three(n, W, E, experts, gated, opt):
    opt = dict(opt)
    g = torch.Generator(device=DEV).manual_seed(n + W + E)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)
    top, shared, weigh = min(2, E), n % 2 == 1, E != 8
    x, y, nw, nb, one = r(1, n, W), r(n, W), r(W), r(W), torch.ones(1, device=DEV)
    w = (r(E + gated, W) * W ** -0.5).bfloat16()
    route = dict(w=w, entries=E, top=top, scale=opt.pop("scale", 1.0), groups=1, keep=1, bias=r(E) if opt.pop("biased", False) else None, correction=r(E) if opt.pop("corrected", False) else None, **opt)
    if n == 64:      # choices that tie, and a row that holds no number
        w[3], w[5] = w[1], w[1]
        y[7, 11] = float("nan")

    def buffers():
        i = lambda k: torch.full((k,), -7, dtype=torch.int32, device=DEV)
        rows = n * top + (n if shared else 0)
        return dict(idx=i(n * top), wgt=torch.full((n * top,), -7.0, device=DEV), gate_out=torch.full((n,), -7.0, device=DEV) if gated else None), \
            dict(experts=experts, group_off=i(experts + 2), pair_token=i(rows), pair_row=i(n * top), pair_wgt=torch.full((rows,), -7.0, device=DEV) if weigh else None, shared=shared)

    add = dict(y=y, out_w=one, norm_w=nw, norm_b=nb, eps=1e-6, h_center=True)
    x1, h1, h16 = x.clone(), torch.empty(n, W, device=DEV), torch.empty(n, W, dtype=torch.bfloat16, device=DEV)
    a, pa = buffers()
    D.streams_step(x1, h=h1, h16=h16, **add)
    D.route_topk(None, h=h1, n=n, **route, **a)
    D.moe_plan(a["idx"], n=n, top=top, wgt=a["wgt"], **pa)
    sync = torch.zeros(32 * 17, dtype=torch.int32, device=DEV)
    for bare in (False, True, False):      # (the counters are zeros again behind every launch)
        x2, h2, g16 = x.clone(), torch.empty(n, W, device=DEV), torch.empty(n, W, dtype=torch.bfloat16, device=DEV)
        b, pb = buffers()
        small = n <= D.PLAN_ROWS
        D.streams_step(x2, h=None if bare else h2, h16=g16, route=dict(**route, **b), **(dict(plan=pb, sync=sync) if small else {}), **add)
        if not small:
            D.moe_plan(b["idx"], n=n, top=top, wgt=b["wgt"], **pb)
        assert not sync.any()
        same = lambda u, v: torch.equal(torch.nan_to_num(u, nan=3e38), torch.nan_to_num(v, nan=3e38))
        assert same(x1, x2) and same(h16.float(), g16.float()) and (bare or same(h1, h2))
        if n <= 512:      # the sums' order of launches of few rows
            assert torch.equal(a["idx"], b["idx"]) and same(a["wgt"], b["wgt"])
            assert not gated or same(a["gate_out"], b["gate_out"])
        else:             # many rows have another order: choices may differ on a tie of some roundings of the largest score
            assert (a["idx"] != b["idx"]).float().mean() < 0.01
            assert torch.allclose(a["wgt"][a["idx"] == b["idx"]], b["wgt"][a["idx"] == b["idx"]], rtol=1e-4, atol=1e-6)
        # the plan of the choice that was made: offsets by count, every pair's row inside its expert's group and its own
        idx, base = b["idx"].long(), n if shared else 0
        count = torch.bincount(idx, minlength=E)[:experts]
        off = torch.cat([torch.tensor([0], device=DEV), count.cumsum(0)]) + base
        got = pb["group_off"].long()
        assert torch.equal(got[int(shared):experts + 1 + int(shared)], off) and (not shared or got[0] == 0)
        row, mine = pb["pair_row"].long(), idx < experts
        assert (row[~mine] == -1).all()
        r_, e_ = row[mine], idx[mine]
        assert (r_ >= off[e_]).all() and (r_ < off[e_ + 1]).all() and r_.unique().numel() == r_.numel()
        t_ = (torch.arange(n * top, device=DEV) // top)[mine]
        assert torch.equal(pb["pair_token"].long()[r_], t_)
        assert not weigh or same(pb["pair_wgt"][r_], b["wgt"][mine])
        if shared:
            assert torch.equal(pb["pair_token"].long()[:n], torch.arange(n, device=DEV)) and (not weigh or (pb["pair_wgt"][:n] == 1).all())


def test_what_does_not_fit_is_refused():
    x, h, i = torch.zeros(1, 4, 64, device=DEV), torch.zeros(4, 64, device=DEV), torch.zeros(64, dtype=torch.int32, device=DEV)
    kw = dict(norm_w=torch.ones(64, device=DEV), eps=1e-6, h=h)
    route = lambda E, **k: dict(w=torch.zeros(E, 64, dtype=torch.bfloat16, device=DEV), entries=E, top=2, scale=1.0, idx=i, wgt=h.view(-1), **k)
    D.streams_step(x, route=route(17), **kw)
    for bad in (route(18), route(16, groups=2, keep=1), dict(route(8), top=9)):
        with pytest.raises(Exception, match="route"):
            D.streams_step(x, route=bad, **kw)
    with pytest.raises(Exception, match="router on rows"):
        D.streams_step(x, route=route(8), rows=i[:2], **kw)
    with pytest.raises(Exception, match="counters"):
        D.streams_step(x, route=route(8), plan=dict(experts=8, group_off=i, pair_token=i, pair_row=i), sync=i, **kw)


# rows, width, experts and choices of the mixture that is summed, of the one that is chosen, a gate on each
SUMMED = [(1, 64, 3, 1, 4, 2, False), (7, 1024, 8, 1, 8, 2, True), (100, 2048, 4, 3, 6, 1, True), (128, 4100, 5, 2, 5, 2, False), (129, 1024, 8, 2, 8, 1, True), (700, 8192, 2, 1, 4, 3, False),
          (4100, 1024, 4, 1, 8, 2, True), (5000, 512, 8, 3, 4, 1, False), (4500, 2048, 8, 2, 8, 2, True)]


@pytest.mark.parametrize("n,W,Ea,ta,Eb,tb,gated", SUMMED)
def test_a_mixture_summed_and_the_next_one_chosen(n, W, Ea, ta, Eb, tb, gated):
    """One launch sums a mixture, norms the row and chooses the next mixture's experts, its normed rows and gates in the place of those it read: against the launches apart.  Weights and rows of
    the two mixtures lie apart, or (as many choices a row) at one place."""
    g = torch.Generator(device=DEV).manual_seed(n + W + ta)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)
    x, y, ey, h0, sh, nw, one = r(1, n, W), r(n, W), r(n * ta, W), r(n, W), r(n, W), r(W), torch.ones(1, device=DEV)
    row = torch.randperm(n * ta, generator=g, device=DEV).to(torch.int32)
    row[::5] = -1      # choices that are no expert: the mixture's input row
    wgt, gates = r(n * ta), r(n)
    w = (r(Eb + gated, W) * W ** -0.5).bfloat16()
    route = dict(w=w, entries=Eb, top=tb, scale=1.0, chosen_softmax=True)
    add = dict(y=y, out_w=one, norm_w=nw, eps=1e-6)

    def run(apart, shared_place):
        i = lambda k: torch.full((k,), -7, dtype=torch.int32, device=DEV)
        xs, h, sg, wa, pr = x.clone(), h0.clone(), gates.clone(), wgt.clone(), row.clone()
        idx, wb, pb = i(n * tb), wa if shared_place else torch.full((n * tb,), -7.0, device=DEV), pr if shared_place else i(n * tb)
        plan = dict(experts=Eb, group_off=i(Eb + 1), pair_token=i(n * tb), pair_row=pb)
        moe = dict(y=ey, pair_row=pr, wgt=wa, h=h, shared=sh, top=ta, shared_gate=sg if gated else None)
        ride = dict(route, idx=idx, wgt=wb, gate_out=sg if gated else None)
        if apart:
            D.streams_step(xs, moe=moe, h=h, **add)
            D.route_topk(None, h=h, n=n, correction=None, groups=1, keep=1, **ride)
        else:
            sync = torch.zeros(32 * 17, dtype=torch.int32, device=DEV)
            D.streams_step(xs, moe=moe, h=h, route=ride, **(dict(plan=plan, sync=sync) if n <= D.PLAN_ROWS else {}), **add)
            assert not sync.any()
        if apart or n > D.PLAN_ROWS:
            D.moe_plan(idx, n=n, top=tb, wgt=wb, **plan)
        return xs, h, sg, idx, wb[: n * tb], plan["group_off"], pb

    want = run(True, False)
    pick = torch.where(row < 0, 0, row).long()
    terms = torch.where((row < 0)[:, None], h0.repeat_interleave(ta, 0).double(), ey[pick].double()) * wgt[:, None].double()
    sums = x[0].double() + y.double() + terms.view(n, ta, W).sum(1) + (gates[:, None] if gated else 1.0) * sh.double()
    assert ((want[0][0].double() - sums).abs().max() <= 2e-6 * sums.abs().max())      # (a sum of at most seven terms)
    for shared_place in ([False, True] if ta == tb else [False]):
        got = run(False, shared_place)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
        same = got[3] == want[3]
        if n <= 512:      # the router's sums in one order: the same bits
            assert same.all() and torch.equal(got[4], want[4]) and torch.equal(got[2], want[2]) and torch.equal(got[5], want[5])
        else:
            assert same.float().mean() > 0.99 and torch.allclose(got[4][same], want[4][same], rtol=1e-4, atol=1e-6) and torch.allclose(got[2], want[2], rtol=1e-4, atol=1e-6)
        e, at = got[3].long(), got[6].long()
        off = torch.cat([torch.zeros(1, dtype=torch.long, device=DEV), torch.bincount(e, minlength=Eb).cumsum(0)])
        assert torch.equal(got[5].long(), off) and (at >= off[e]).all() and (at < off[e + 1]).all() and at.unique().numel() == n * tb


def test_a_choice_over_what_other_rows_still_read_is_refused():
    n, W = 6, 64
    f, i = lambda *s: torch.zeros(*s, device=DEV), lambda k: torch.zeros(k, dtype=torch.int32, device=DEV)
    buf, h = f(64), f(n, W)

    def run(wa, ta, wb, tb, **kw):
        moe = dict(y=f(n * ta, W), pair_row=kw.get("row", i(n * ta)), wgt=wa, h=h, shared=f(n, W), top=ta, shared_gate=kw.get("gate"))
        route = dict(w=f(4 + ("out" in kw), W).bfloat16(), entries=4, top=tb, scale=1.0, idx=kw.get("idx", i(n * tb)), wgt=wb, gate_out=kw.get("out"))
        D.streams_step(f(1, n, W), moe=moe, out_w=f(1), norm_w=f(W), eps=1e-6, h=h, route=route)

    run(buf, 2, buf, 2), run(buf[:12], 2, buf[12:], 1), run(buf[32:], 1, buf, 2, gate=buf[56:], out=buf[56:])
    words = i(64)
    for bad in (lambda: run(buf, 1, buf, 2), lambda: run(buf, 3, buf, 1), lambda: run(buf[4:], 2, buf, 2), lambda: run(buf, 2, buf[11:], 2), lambda: run(f(12), 2, f(12), 2, gate=buf, out=buf[1:]),
                lambda: run(f(12), 2, buf, 2, gate=buf[4:]), lambda: run(f(12), 2, f(6), 1, row=words, idx=words)):
        with pytest.raises(Exception, match="still read"):
            bad()
