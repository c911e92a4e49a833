"""i64h_rec_step: a decode step's recurrence in one launch against the launches it stands for (convolution, gates, decays' Linear, scan, norm and gate)."""
import pytest
import torch

from vllm_i64_amd import ops_dense as D

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# heads, dim, vdim, ranks, taps, rows
SIZES = [(8, 128, 128, (128, 128), 4, 7), (1, 4, 1, (8, 8), 2, 1), (3, 64, 64, (16, 136), 4, 33), (2, 68, 65, (264, 8), 8, 5), (5, 60, 128, (128, 40), 3, 2), (16, 128, 64, (128, 128), 4, 64)]


def _close(got, want, what):
    """Both sides round the same inputs; they differ in the order of 32-bit sums of at most a few hundred terms, through a decay, a step and a norm: 1e-5 of the largest value is
    some eighty roundings of it."""
    g, w = got.double(), want.double()
    assert torch.isfinite(g).all(), what
    assert (g - w).abs().max() <= 1e-5 * w.abs().max().clamp(min=1e-20), (what, ((g - w).abs().max() / w.abs().max()).item())


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("delta", [True, False])
@pytest.mark.parametrize("H,d,dv,ranks,taps,n", SIZES)
def test_one_launch_is_the_six(H, d, dv, ranks, taps, n, delta, exact):
    g = torch.Generator(device=DEV).manual_seed(H * d + dv + n)
    r = lambda *s, std=1.0: torch.randn(*s, generator=g, device=DEV) * std
    pad4 = lambda x: (x + 3) // 4 * 4
    nd, rv, slots = H * d, H * dv, n + 3
    C = 2 * nd + rv
    a_off = pad4(C)
    z_off = a_off + pad4(ranks[0])
    b_off = z_off + max(pad4(ranks[1]), pad4(rv))
    P = r(n, pad4(b_off + H))
    ld = P.shape[-1]
    a, bias, rate = r(nd, ranks[0], std=ranks[0] ** -0.5).bfloat16(), r(nd), torch.rand(nd, generator=g, device=DEV) + 0.1
    z, norm_w, eps = r(rv, ranks[1], std=ranks[1] ** -0.5).bfloat16(), r(dv), 1e-6
    conv_w, conv = r(C, taps, std=0.5), r(slots, taps - 1, C)
    pos = torch.randint(1, 2000, (n,), generator=g, device=DEV, dtype=torch.int32)
    pos[::3] = torch.arange(len(pos[::3]), device=DEV, dtype=torch.int32) % taps      # rows at a sequence's start: no state, fewer carried inputs
    slot = torch.randperm(slots, generator=g, device=DEV)[:n].to(torch.int32)
    state = r(slots, H, dv, d, std=0.3)
    seg = torch.arange(n + 1, dtype=torch.int32, device=DEV)
    s1, s2, c1, c2 = state.clone(), state.clone(), conv.clone(), conv.clone()

    F, R, want, got, got16 = (torch.empty(n, w, device=DEV) for w in (nd, rv, rv, rv, rv))
    got16 = got16.bfloat16()
    D.linear(P, a, F, m=n, a_off=a_off, exact=exact, bias=bias, epilogue=D.EPI_DECAY, e=rate)
    if delta:
        X, G, Z = torch.empty(n, C, device=DEV), torch.empty(n, 2 * H, device=DEV), torch.empty(n, rv, device=DEV)
        D.causal_conv(P, off=0, channels=C, w=conv_w, bias=None, positions=pos, slot_ids=slot, state=c1, out=X, n=n, single_rows=True)
        cols = dict(q_off=0, k_off=nd, v_off=2 * nd, heads=H, kv_heads=H, dim=d, vdim=dv, n=n)
        D.gdn_gates(X, G, P, b_off=b_off, a_off=-1, a_log=None, dt_bias=None, unit_eps=1e-6, q_scale=d ** -0.5, **cols)
        D.linear(P, z, Z, m=n, a_off=z_off, exact=exact)
        D.gdn_scan(X, G, f=F, seg_start=seg, nseg=n, positions=pos, slot_ids=slot, state=s1, out=R, **cols)
        D.gate_norm(R, norm_w, want, groups=H, eps=eps, z=Z, ldz=rv, n=n, gate_after=True, width=rv, sigmoid=True)
        kw = dict(q_off=0, conv_w=conv_w, conv=c2, b_off=b_off, unit_eps=1e-6, z=z, z_off=z_off, sigmoid=True)
    else:
        D.gla_scan(P, f=F, q_off=0, k_off=nd, f_off=0, v_off=2 * nd, heads=H, dim=d, vdim=dv, seg_start=seg, nseg=n, positions=pos, slot_ids=slot, state=s1, out=R, n=n, q_scale=d ** -0.5)
        D.gate_norm(R, norm_w, want, groups=H, eps=eps, z=P, z_off=z_off, ldz=ld, n=n, gate_after=True, width=rv)
        kw = dict(q_off=0, k_off=nd, v_off=2 * nd, z_off=z_off)
    D.rec_step(P, heads=H, dim=d, vdim=dv, a=a, a_off=a_off, a_bias=bias, a_rate=rate, norm_w=norm_w, eps=eps, positions=pos, slot_ids=slot, state=s2, n=n, out=got, out16=got16,
               q_scale=d ** -0.5, exact=exact, **kw)
    _close(s2, s1, "state")
    _close(got, want, "result")
    assert torch.equal(got16, got.bfloat16())
    assert torch.equal(c1, c2)
    idle = torch.ones(slots, dtype=torch.bool, device=DEV)
    idle[slot.long()] = False
    assert torch.equal(s2[idle], state[idle])      # other sequences' states are left alone


def test_what_does_not_fit_is_refused():
    t = torch.zeros(4, 64, device=DEV)
    i = torch.zeros(4, dtype=torch.int32, device=DEV)
    kw = dict(a=torch.zeros(8, 8, device=DEV).bfloat16(), a_off=16, a_bias=t[0], a_rate=t[0], z_off=24, norm_w=t[0], eps=0.0, positions=i, slot_ids=i, n=1, out=t, heads=1)
    with pytest.raises(Exception, match="rec_step"):      # the gate's columns lie outside the row
        D.rec_step(t, q_off=0, k_off=8, v_off=8, dim=8, vdim=48, state=torch.zeros(1, 1, 48, 8, device=DEV), **kw)
    with pytest.raises(Exception, match="rec_step"):      # key channels that are no four
        D.rec_step(t, q_off=0, k_off=8, v_off=8, dim=6, vdim=4, state=torch.zeros(1, 1, 4, 6, device=DEV), **{**kw, "a": kw["a"][:6]})


# heads, dim, vdim, ranks, taps, rows of the runs
RUNS = [(8, 128, 128, (128, 128), 4, (150, 1, 16, 2, 33)), (3, 64, 64, (8, 136), 3, (17, 3, 160)), (2, 68, 60, (264, 8), 2, (31, 1, 1, 48)), (1, 4, 4, (8, 40), 4, (1, 2, 3, 4, 5)),
        (5, 36, 128, (40, 128), 4, (145, 15))]


@pytest.mark.parametrize("delta", [True, False])
@pytest.mark.parametrize("H,d,dv,ranks,taps,runs", RUNS)
def test_tiles_from_the_projections(H, d, dv, ranks, taps, runs, delta):
    """The same in tiles of 16 tokens, runs that start afresh, inside the first taps, or far behind: against the separate launches, their scan in tiles too."""
    from vllm_i64_amd import _lib
    g = torch.Generator(device=DEV).manual_seed(H * d + dv + len(runs))
    r = lambda *s, std=1.0: torch.randn(*s, generator=g, device=DEV) * std
    pad4 = lambda x: (x + 3) // 4 * 4
    n, nseg, nd, rv = sum(runs), len(runs), H * d, H * dv
    slots, C = nseg + 2, 2 * nd + rv
    a_off = pad4(C)
    z_off = a_off + pad4(ranks[0])
    b_off = z_off + max(pad4(ranks[1]), pad4(rv))
    P = r(n, pad4(b_off + H))
    a, bias, rate = r(nd, ranks[0], std=ranks[0] ** -0.5).bfloat16(), r(nd), torch.rand(nd, generator=g, device=DEV) + 0.1
    z, norm_w, eps = r(rv, ranks[1], std=ranks[1] ** -0.5).bfloat16(), r(dv), 1e-6
    conv_w, conv, state = r(C, taps, std=0.5), r(slots, taps - 1, C), r(slots, H, dv, d, std=0.3)
    own = torch.randperm(slots, generator=g, device=DEV)[:nseg]
    pos = torch.cat([torch.arange(m, device=DEV) + (0, 1, 2, 3, 700)[i % 5] for i, m in enumerate(runs)]).to(torch.int32)
    slot = torch.cat([own[i].repeat(m) for i, m in enumerate(runs)]).to(torch.int32)
    seg = torch.tensor([0, *torch.tensor(runs).cumsum(0).tolist()], dtype=torch.int32, device=DEV)
    s1, s2, c1, c2 = state.clone(), state.clone(), conv.clone(), conv.clone()
    work = torch.full((D.scan_work_floats(n, nseg, H, d),), float("nan"), device=DEV)
    F, R, want, got, got16, X2, R2 = (torch.full((n, w), float("nan"), device=DEV) for w in (nd, rv, rv, rv, rv, rv, rv))
    got16 = got16.bfloat16()
    D.linear(P, a, F, m=n, a_off=a_off, bias=bias, epilogue=D.EPI_DECAY, e=rate)
    scan = dict(seg_start=seg, nseg=nseg, positions=pos, slot_ids=slot)
    try:
        _lib.call_dense("i64h_set_gdn_scan_form", 5)
        if delta:
            X, G, Z = torch.empty(n, C, device=DEV), torch.empty(n, 2 * H, device=DEV), torch.empty(n, rv, device=DEV)
            D.causal_conv(P, off=0, channels=C, w=conv_w, bias=None, positions=pos, slot_ids=slot, state=c1, out=X, n=n, seg_start=seg, nseg=nseg)
            cols = dict(q_off=0, k_off=nd, v_off=2 * nd, heads=H, kv_heads=H, dim=d, vdim=dv, n=n)
            D.gdn_gates(X, G, P, b_off=b_off, a_off=-1, a_log=None, dt_bias=None, unit_eps=1e-6, q_scale=d ** -0.5, **cols)
            D.linear(P, z, Z, m=n, a_off=z_off)
            D.gdn_scan(X, G, f=F, state=s1, out=R, work=work, **scan, **cols)
            D.gate_norm(R, norm_w, want, groups=H, eps=eps, z=Z, ldz=rv, n=n, gate_after=True, width=rv, sigmoid=True)
            kw = dict(q_off=0, conv_w=conv_w, conv=c2, b_off=b_off, unit_eps=1e-6, z=z, z_off=z_off, sigmoid=True, x=X2)
        else:
            D.gla_scan(P, f=F, q_off=0, k_off=nd, f_off=0, v_off=2 * nd, heads=H, dim=d, vdim=dv, state=s1, out=R, n=n, q_scale=d ** -0.5, work=work, **scan)
            D.gate_norm(R, norm_w, want, groups=H, eps=eps, z=P, z_off=z_off, ldz=P.shape[-1], n=n, gate_after=True, width=rv)
            kw = dict(q_off=0, k_off=nd, v_off=2 * nd, z_off=z_off)
    finally:
        _lib.call_dense("i64h_set_gdn_scan_form", 0)
    work.fill_(float("nan"))
    D.rec_tiles(P, heads=H, dim=d, vdim=dv, a=a, a_off=a_off, a_bias=bias, a_rate=rate, norm_w=norm_w, eps=eps, state=s2, n=n, out=got, out16=got16, q_scale=d ** -0.5, work=work, r=R2,
                **scan, **kw)
    _close(s2, s1, "state")
    _close(R2, R, "read-out")
    # (a head's row is divided by its root mean square: small read-outs carry the largest one's roundings, hence row by row)
    e = (got.double() - want.double()).view(n, H, dv).abs().amax(-1) / want.double().view(n, H, dv).abs().amax(-1).clamp(min=1e-20)
    big = R.view(n, H, dv).abs().amax(-1)
    assert (e * (big / big.max()).double() <= 2e-5).all()
    assert torch.equal(got16, got.bfloat16()) and torch.equal(c1, c2)
    idle = torch.ones(slots, dtype=torch.bool, device=DEV)
    idle[own] = False
    assert torch.equal(s2[idle], state[idle])


class Layer:
    """A recurrence's operands for runs of rows, and the same in 64 bits on the CPU."""
    def __init__(self, H, d, dv, ranks, taps, runs, delta):
        self.H, self.d, self.dv, self.taps, self.runs, self.delta = H, d, dv, taps, runs, delta
        g = torch.Generator().manual_seed(H * d + dv + len(runs))
        r = lambda *s, std=1.0: torch.randn(*s, generator=g) * std
        n, nd, rv = sum(runs), H * d, H * dv
        C, slots = 2 * nd + rv, len(runs) + 2
        pad4 = lambda x: (x + 3) // 4 * 4
        self.a_off = pad4(C)
        self.z_off = self.a_off + pad4(ranks[0])
        self.b_off = self.z_off + max(pad4(ranks[1]), pad4(rv))
        self.P = r(n, pad4(self.b_off + H))
        self.a, self.bias, self.rate = r(nd, ranks[0], std=ranks[0] ** -0.5).bfloat16(), r(nd), torch.rand(nd, generator=g) + 0.1
        self.z, self.norm_w = r(rv, ranks[1], std=ranks[1] ** -0.5).bfloat16(), r(dv)
        self.conv_w, self.conv, self.state = r(C, taps, std=0.5), r(slots, taps - 1, C), r(slots, H, dv, d, std=0.3)
        self.own = torch.randperm(slots, generator=g)[:len(runs)]
        self.first = [(0, 700, 1, 2, 3)[i % 5] for i in range(len(runs))]

    def launch(self, P):
        n, nseg, rv, nd = len(P), len(self.runs), self.H * self.dv, self.H * self.d
        gpu = lambda t: t.to(DEV).clone()
        pos = torch.cat([torch.arange(m) + p for m, p in zip(self.runs, self.first)]).to(torch.int32).to(DEV)
        slot = torch.cat([s.repeat(m) for m, s in zip(self.runs, self.own)]).to(torch.int32).to(DEV)
        state, conv, out = gpu(self.state), gpu(self.conv), torch.full((n, rv), float("nan"), device=DEV)
        kw = dict(heads=self.H, dim=self.d, vdim=self.dv, a=gpu(self.a), a_off=self.a_off, a_bias=gpu(self.bias), a_rate=gpu(self.rate), norm_w=gpu(self.norm_w), eps=1e-6, positions=pos,
                  slot_ids=slot, state=state, n=n, out=out, q_scale=self.d ** -0.5, q_off=0, z_off=self.z_off)
        kw.update(dict(conv_w=gpu(self.conv_w), conv=conv, b_off=self.b_off, unit_eps=1e-6, z=gpu(self.z), sigmoid=True) if self.delta else dict(k_off=nd, v_off=2 * nd))
        if max(self.runs) == 1:
            D.rec_step(gpu(P), **kw)
        else:
            seg = torch.tensor([0, *torch.tensor(self.runs).cumsum(0).tolist()], dtype=torch.int32, device=DEV)
            room = lambda: torch.full((n, rv), float("nan"), device=DEV)
            D.rec_tiles(gpu(P), seg_start=seg, nseg=nseg, work=torch.full((D.scan_work_floats(n, nseg, self.H, self.d),), float("nan"), device=DEV), r=room(), x=room(), **kw)
        return out.cpu(), state.cpu()[self.own]

    def exact(self, P):
        H, d, dv, nd = self.H, self.d, self.dv, self.H * self.d
        outs, states, at = [], [], 0
        map_ = lambda x, w: (x.bfloat16().double()[:, None, :] * w.double()[None]).sum(-1)
        for m, slot, pos in zip(self.runs, self.own, self.first):
            p = P[at:at + m].double()
            at += m
            f = torch.exp(-self.rate.double() * torch.logaddexp(torch.zeros(1).double(), map_(p[:, self.a_off:self.a_off + self.a.shape[1]].float(), self.a) + self.bias.double())).view(m, H, d)
            x = p[:, :2 * nd + H * dv]
            if self.delta:
                back = self.conv[slot].double().clone()
                back[:max(0, self.taps - 1 - pos)] = 0      # (before the sequence's first token)
                rows = torch.cat([back, x])
                x = sum(rows[k:k + m] * self.conv_w[:, k].double() for k in range(self.taps))
                x = x * torch.sigmoid(x)
            q, k, v = x[:, :nd].view(m, H, d), x[:, nd:2 * nd].view(m, H, d), x[:, 2 * nd:].view(m, H, dv)
            if self.delta:
                unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)
                q, k, beta = unit(q), unit(k), torch.sigmoid(p[:, self.b_off:self.b_off + H])
                gate = torch.sigmoid(map_(p[:, self.z_off:self.z_off + self.z.shape[1]].float(), self.z))
            else:
                zc = p[:, self.z_off:self.z_off + H * dv]
                gate = zc * torch.sigmoid(zc)
            S, o = self.state[slot].double() * (pos != 0), torch.zeros(m, H, dv).double()
            for t in range(m):
                S = S * f[t][:, None, :]
                u = beta[t][:, None] * (v[t] - (S * k[t][:, None, :]).sum(-1)) if self.delta else v[t]
                S = S + u[:, :, None] * k[t][:, None, :]
                o[t] = (S * q[t][:, None, :]).sum(-1) * d ** -0.5
            outs.append((o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-6) * self.norm_w.double()).view(m, H * dv) * gate)
            states.append(S)
        return torch.cat(outs), torch.stack(states), o


LAYERS = [(3, 64, 64, (8, 136), 3, (17, 3, 40)), (2, 68, 60, (40, 72), 2, (31, 1, 48)), (2, 128, 128, (136, 40), 4, (50, 1, 20)), (2, 64, 68, (40, 8), 8, (1,) * 5), (3, 128, 64, (136, 72), 4, (1,) * 7)]


def _near(got, want):
    """32-bit sums of some hundred terms through up to 50 steps and a division by a row's root mean square, against 64 bits: 1e-4 of the largest value."""
    ok = torch.isfinite(want)
    assert torch.equal(torch.isfinite(got), ok)
    assert (got[ok].double() - want[ok]).abs().max() <= 1e-4 * want[ok].abs().max()


@pytest.mark.parametrize("delta", [True, False])
@pytest.mark.parametrize("H,d,dv,ranks,taps,runs", LAYERS)
def test_infinite_weights_of_the_maps(H, d, dv, ranks, taps, runs, delta):
    """A decay of an infinite sum is zero or one and a gate too: ranks that are no whole steps of the products meet nothing but their own values."""
    L = Layer(H, d, dv, ranks, taps, runs, delta)
    _near(L.launch(L.P)[0], L.exact(L.P)[0])
    inf = float("inf")
    L.a[1, 0], L.a[d, ranks[0] - 1], L.a[H * d - 1, ranks[0] - 6] = inf, -inf, inf
    L.z[0, 1], L.z[dv, ranks[1] - 8] = inf, -inf
    got, want = L.launch(L.P), L.exact(L.P)
    assert torch.isfinite(want[0]).all()
    _near(got[0], want[0]), _near(got[1], want[1])


@pytest.mark.parametrize("what", ["q", "k", "v", "decay", "strength", "gate"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), 3e38])
@pytest.mark.parametrize("delta", [True, False])
@pytest.mark.parametrize("H,d,dv,ranks,taps,runs", LAYERS)
def test_a_row_that_is_no_number(H, d, dv, ranks, taps, runs, delta, what, value):
    """... reaches what 64 bits say it reaches: its own columns, its head or its sequence, from its token on, and no other run's bits."""
    L = Layer(H, d, dv, ranks, taps, runs, delta)
    P, row = L.P.clone(), sum(runs[:-1]) + runs[-1] * 2 // 3
    P[row, {"q": d + 1, "k": H * d + d + 2, "v": 2 * H * d + 3, "decay": L.a_off + ranks[0] - 2, "strength": L.b_off + 1, "gate": L.z_off + min(ranks[1], dv) - 1}[what]] = value
    (got, gs), (want, ws, _), (clean, cs) = L.launch(P), L.exact(P), L.launch(L.P)
    first = sum(runs[:-1])
    assert torch.equal(got[:first], clean[:first]) and torch.equal(gs[:-1], cs[:-1])
    assert torch.isfinite(got[first:row]).all()
    if value != 3e38:
        if what == "v":      # (an infinite value's sums over channels and over tokens are an infinity here and none there: a head's norm makes zeros of its row or nothing)
            assert (~torch.isfinite(got[row:, 3])).all()
            got[row:, :dv], want[row:, :dv] = 0, 0
        _near(got, want), _near(gs, ws)
