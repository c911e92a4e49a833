"""The recurrences' form in tiles of 16 tokens (delta rule, linear attention with keys of its own) against the recurrence in 64 bits: runs that end
anywhere in a tile, fresh or continued, padded channel and column tiles, decays that underflow, and rows that hold no finite number."""
import pytest
import torch

from tests.test_gpu_fukatar import Rows

pytestmark = pytest.mark.gpu
F64 = torch.float64
RUNS = [(4, 0, 33), (1, 7, 1), (0, 3, 16), (3, 0, 17), (2, 50, 70), (5, 0, 15)]


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


def recurrence(q, k, v, beta, f, S):
    """[T, H, ...] in 64 bits; beta None: linear attention.  Returns the read-outs and the state behind them, S [H, dv, d]."""
    out = []
    for t in range(q.shape[0]):
        S = S * f[t].unsqueeze(1)
        u = v[t] if beta is None else beta[t].unsqueeze(-1) * (v[t] - (S * k[t].unsqueeze(1)).sum(-1))
        S = S + u.unsqueeze(-1) * k[t].unsqueeze(1)
        out.append((S * q[t].unsqueeze(1)).sum(-1))
    return torch.stack(out), S


def launch(dev, form, delta, channel, dims, r, X, Gt, F, S0):
    from vllm_i64_amd import _lib, ops_dense as D
    H, G, d, dv = dims
    S, O = S0.to(dev).clone(), torch.full((r.n, H * dv), 7.0, device=dev)
    work = torch.full((D.scan_work_floats(r.n, r.nseg, H, d),), float("nan"), device=dev)
    cols = dict(heads=H, dim=d, vdim=dv, seg_start=r.seg, nseg=r.nseg, positions=r.pos, slot_ids=r.slots, state=S, out=O, n=r.n, work=work)
    try:
        _lib.call_dense("i64h_set_gdn_scan_form", form)
        if delta:
            D.gdn_scan(X.to(dev), Gt.to(dev), f=F.to(dev) if channel else None, q_off=0, k_off=G * d, v_off=2 * G * d, kv_heads=G, **cols)
        else:
            D.gla_scan(X.to(dev), f=F.to(dev), q_off=0, k_off=G * d, f_off=0, v_off=2 * G * d, q_scale=0.3, **cols)
    finally:
        _lib.call_dense("i64h_set_gdn_scan_form", 0)
    return O.cpu(), S.cpu()


def inputs(dims, n, seed, low=0.0):
    H, G, d, dv = dims
    g = torch.Generator().manual_seed(seed)
    X = torch.randn(n, 2 * G * d + H * dv, generator=g)
    k = X[:, G * d:2 * G * d].view(n, G, d)
    k /= k.norm(dim=-1, keepdim=True)
    X[:, :G * d] *= d ** -0.5
    F = low + (1.0 - low) * torch.rand(n, H * d, generator=g)
    return X, torch.rand(n, 2 * H, generator=g), F, torch.randn(6, H, dv, d, generator=g)


def oracle(delta, channel, dims, X, Gt, F, S0):
    H, G, d, dv = dims
    own = torch.arange(H) // (H // G)
    O, S, at = [], S0.double().clone(), 0
    for slot, p, c in RUNS:
        x, gt, f = X[at:at + c].double(), Gt[at:at + c].double(), F[at:at + c].double()
        q, k, v = x[:, :G * d].reshape(c, G, d)[:, own], x[:, G * d:2 * G * d].reshape(c, G, d)[:, own], x[:, 2 * G * d:].reshape(c, H, dv)
        dec = f.reshape(c, H, d) if channel else gt[:, H:].unsqueeze(-1).expand(c, H, d)
        o, S[slot] = recurrence(q if delta else 0.3 * q, k, v, gt[:, :H] if delta else None, dec, S[slot] if p else torch.zeros(H, dv, d, dtype=F64))
        O.append(o.reshape(c, H * dv))
        at += c
    return torch.cat(O), S


def err(a, b):
    return float((a.double() - b).norm() / b.norm())


# a token's read-out and state are sums of at most dim + 16 products in 32 bits behind a chain of tiles that the decays keep from growing: a few hundred
# units of 2^-24 at the outside
TOL = 2e-5


@pytest.mark.parametrize("rule", ["delta, a decay per channel", "delta, a decay per head", "linear"])
@pytest.mark.parametrize("low", [0.0, 0.9])
@pytest.mark.parametrize("H,G,d,dv", [(4, 2, 64, 32), (3, 3, 40, 24), (8, 8, 128, 128), (2, 2, 200, 40), (1, 1, 12, 5), (2, 1, 256, 256), (2, 2, 132, 17)])
def test_tiles_against_64_bits(dev, rule, low, H, G, d, dv):
    delta, channel = rule != "linear", not rule.endswith("head")
    dims = (H, G if delta else H, d, dv)
    r = Rows(dev, RUNS)
    X, Gt, F, S0 = inputs(dims, r.n, d + dv, low)
    want, state = oracle(delta, channel, dims, X, Gt, F, S0)
    O, S = launch(dev, 5, delta, channel, dims, r, X, Gt, F, S0)
    O1, S1 = launch(dev, 1, delta, channel, dims, r, X, Gt, F, S0)
    print("tiles %.2e %.2e, token by token %.2e %.2e" % (err(O, want), err(S, state), err(O1, want), err(S1, state)))
    assert err(O, want) < TOL and err(S, state) < TOL


@pytest.mark.parametrize("delta", [True, False])
def test_decays_that_underflow(dev, delta):
    """Decays of 1e-6 and of zero: their products over a tile are no numbers that could be divided by."""
    dims = (2, 2, 64, 16)
    r = Rows(dev, RUNS)
    X, Gt, F, S0 = inputs(dims, r.n, 3, 0.9)
    F[:, ::3] = 1e-6
    F[::5, 1::7] = 0.0
    want, state = oracle(delta, True, dims, X, Gt, F, S0)
    O, S = launch(dev, 5, delta, True, dims, r, X, Gt, F, S0)
    assert err(O, want) < TOL and err(S, state) < TOL


@pytest.mark.parametrize("delta", [True, False])
@pytest.mark.parametrize("part", ["q", "k", "v", "decay", "state"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_no_finite_number_reaches_no_token_before_it(dev, delta, part, bad):
    """A value that is no finite number in the middle of a tile: what is finite token by token is the same finite number in tiles."""
    dims = (2, 2, 64, 32)
    r = Rows(dev, RUNS)
    X, Gt, F, S0 = inputs(dims, r.n, 5, 0.5)
    row = 33 + 1 + 5      # the sixth token of the third run
    if part == "decay":
        F[row, 70] = bad
    elif part == "state":
        S0[0, 1, 3, 9] = bad
    else:
        X[row, {"q": 3, "k": 128 + 70, "v": 256 + 5}[part]] = bad
    O, S = launch(dev, 5, delta, True, dims, r, X, Gt, F, S0)
    O1, S1 = launch(dev, 1, delta, True, dims, r, X, Gt, F, S0)
    for a, b in ((O, O1), (S, S1)):
        assert torch.equal(torch.isfinite(a), torch.isfinite(b))
        fine = torch.isfinite(b)
        assert not bool(fine.all()) or part == "q" and a is S
        assert err(a[fine], b[fine].double()) < TOL


def test_the_longest_runs_choose_the_tiles_and_need_their_workspace(dev):
    from vllm_i64_amd import _lib, ops_dense as D
    dims = (2, 2, 32, 16)
    r = Rows(dev, RUNS)
    X, Gt, F, S0 = inputs(dims, r.n, 9)
    a, b = launch(dev, 0, True, True, dims, r, X, Gt, F, S0), launch(dev, 5, True, True, dims, r, X, Gt, F, S0)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    with pytest.raises(_lib.I64HError):
        D.gdn_scan(X.to(dev), Gt.to(dev), f=F.to(dev), q_off=0, k_off=64, v_off=128, heads=2, kv_heads=2, dim=32, vdim=16, seg_start=r.seg, nseg=r.nseg, positions=r.pos,
                   slot_ids=r.slots, state=S0.to(dev), out=torch.empty(r.n, 32, device=dev), n=r.n, work=torch.empty(16, device=dev))


@pytest.mark.parametrize("delta", [True, False])
@pytest.mark.parametrize("singles,length,form", [(6, 15, 1), (6, 16, 2), (2, 40, 2), (3, 100, 2), (3, 150, 5)])
def test_single_rows_beside_a_prompt_whose_length_is_told(dev, delta, singles, length, form):
    """The longest run decides the form where the caller tells it, whatever the mean is: the bits are that form's, and the recurrence's in 64 bits."""
    from vllm_i64_amd import _lib, ops_dense as D
    H, d, dv = 4, 128, 16
    r = Rows(dev, [(1 + i, 9, 1) for i in range(singles)] + [(0, 0, length)])
    X, Gt, F, _ = inputs((H, H, d, dv), r.n, length, 0.9)
    S0 = torch.randn(singles + 1, H, dv, d, generator=torch.Generator().manual_seed(1))
    got = []
    for forced, longest in ((0, length), (form, 0)):
        S, O = S0.to(dev).clone(), torch.full((r.n, H * dv), 7.0, device=dev)
        cols = dict(heads=H, dim=d, vdim=dv, seg_start=r.seg, nseg=r.nseg, positions=r.pos, slot_ids=r.slots, state=S, out=O, n=r.n, longest=longest,
                    work=torch.full((D.scan_work_floats(r.n, r.nseg, H, d),), float("nan"), device=dev))
        try:
            _lib.call_dense("i64h_set_gdn_scan_form", forced)
            if delta:
                D.gdn_scan(X.to(dev), Gt.to(dev), f=F.to(dev), q_off=0, k_off=H * d, v_off=2 * H * d, kv_heads=H, **cols)
            else:
                D.gla_scan(X.to(dev), f=F.to(dev), q_off=0, k_off=H * d, f_off=0, v_off=2 * H * d, q_scale=0.3, **cols)
        finally:
            _lib.call_dense("i64h_set_gdn_scan_form", 0)
        got.append((O.cpu(), S.cpu()))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    for slot, at, c, fresh in ((0, singles, length, True), (2, 1, 1, False)):
        x = X[at:at + c].double()
        o, s = recurrence((1.0 if delta else 0.3) * x[:, :H * d].reshape(c, H, d), x[:, H * d:2 * H * d].reshape(c, H, d), x[:, 2 * H * d:].reshape(c, H, dv),
                          Gt[at:at + c, :H].double() if delta else None, F[at:at + c].double().reshape(c, H, d), torch.zeros(H, dv, d, dtype=F64) if fresh else S0[slot].double())
        assert err(got[0][0][at:at + c], o.reshape(c, H * dv)) < TOL and err(got[0][1][slot], s) < TOL


def test_the_forms_rules():
    """Runs are worth tiles from a length on that grows with their number, earlier from the projections; what the rules take they take for longer runs too."""
    from vllm_i64_amd import ops_dense as D
    for delta in (True, False):
        for H, d, dv in ((16, 128, 128), (8, 128, 128), (8, 64, 64), (4, 256, 64), (3, 70, 16)):
            for singles in (0, 7, 40):
                took = [(D.scan_in_tiles(singles + L, singles + 1, L, H, d, dv, delta=delta), D.rec_in_tiles(singles + L, singles + 1, L, H, d, dv, delta=delta)) for L in range(1, 1200)]
                assert all(b or not a for a, b in took)      # (alone: from the projections too)
                for rule in range(2):
                    on = [t[rule] for t in took]
                    assert on == sorted(on) and not on[0] and on[-1] == (d % 4 == 0)
