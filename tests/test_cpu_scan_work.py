"""Which steps hold a workspace for their recurrences' scans: those whose longest run is worth the form in tiles, for the step alone."""
import pytest
import torch

from vllm_i64_amd import ops_dense as D
from vllm_i64_amd.hybrid_runner import HybridRunner


def runner():
    r = HybridRunner.__new__(HybridRunner)
    r.device = torch.device("cpu")
    return r


# (runs, heads, dim, delta rule, linear attention): both sides of the line, from the smallest runs to the longest
STEPS = [([77], 8, 128, False, False), ([112], 8, 128, False, True), ([143], 8, 128, False, True), ([144], 8, 128, True, True), ([1] * 64, 8, 128, False, False),
         ([64] * 64, 16, 64, False, False), ([17] * 32, 32, 64, False, False), ([9] * 16, 16, 128, False, False), ([1] * 27 + [229, 256], 16, 128, True, True),
         ([1] * 40 + [200], 16, 128, False, False), ([512] * 8, 8, 128, True, True), ([192] * 32, 32, 64, False, False), ([192] * 32, 32, 128, True, True),
         ([1531], 16, 50, False, False), ([4096], 16, 128, True, True)]


@pytest.mark.parametrize("runs,heads,dim,delta,linear", STEPS)
def test_workspace_only_where_the_launch_takes_it(runs, heads, dim, delta, linear):
    n, nseg, key = sum(runs), len(runs), (heads, dim, dim)
    for rule, want in ((True, delta), (False, linear)):
        got = runner()._scan_work(n, nseg, max(runs), {key}, delta=rule)
        assert set(got) == ({key} if want else set())
        if want:
            assert got[key].numel() == D.scan_work_floats(n, nseg, heads, dim)


def test_scans_of_a_step_share_one():
    got = runner()._scan_work(600, 2, 512, {(4, 64, 64), (8, 128, 128), (4, 30, 30)}, delta=True)
    assert set(got) == {(4, 64, 64), (8, 128, 128)} and len({t.data_ptr() for t in got.values()}) == 1
    assert got[(4, 64, 64)].numel() == D.scan_work_floats(600, 2, 8, 128)


def test_no_room_is_no_error(monkeypatch):
    def full(*a, **k):
        raise torch.OutOfMemoryError("no room")
    r = runner()
    monkeypatch.setattr(torch, "empty", full)
    assert r._scan_work(600, 2, 512, {(8, 128, 128)}, delta=True) == {}


def test_longest_run():
    r = runner()
    r._arange = {}
    for tps, want in (([3, 0, 200, 5], 200), ([1, 1], 1), ([77], 77)):
        n = sum(tps)
        starts, nseg, longest = r._runs(n, None, tps, False)
        assert (nseg, longest) == (sum(t > 0 for t in tps), want) and starts.tolist()[-1] == n
    assert r._runs(6, torch.tensor([4, 4, 1, 1, 1, 0]), None, False)[1:] == (3, 3)
    assert r._runs(5, None, None, True)[1:] == (5, 1)


# heads, key heads, dim, vdim, taps (0: linear attention), prompt, whether the step holds a workspace
FROM_PROJECTIONS = [(8, 8, 128, 128, 4, 100, True), (8, 4, 128, 128, 4, 100, False), (8, 4, 128, 128, 4, 200, True), (8, 8, 128, 128, 5, 100, False), (8, 8, 128, 126, 4, 100, False),
                    (8, 8, 128, 128, 1, 100, False), (8, 8, 256, 128, 4, 100, False), (8, 8, 64, 64, 4, 100, True), (8, 8, 128, 128, 0, 100, True), (8, 8, 64, 64, 0, 100, False),
                    (8, 8, 64, 64, 0, 200, True), (8, 8, 128, 126, 0, 100, False), (8, 8, 128, 128, 4, 20, False)]


@pytest.mark.parametrize("heads,kv_heads,dim,vdim,taps,rows,held", FROM_PROJECTIONS)
def test_workspace_from_the_projections_only_where_it_is_read(monkeypatch, heads, kv_heads, dim, vdim, taps, rows, held):
    """A step's workspace is read by the tiles from the projections, or by a scan whose runs alone are worth it: no launch is handed one that it leaves."""
    from types import SimpleNamespace
    from vllm_i64_amd import hybrid_runner
    r = runner()
    r.exact, r.cfg, r.max_ff = False, SimpleNamespace(norm_eps=1e-6), 0
    delta = taps > 0
    m = SimpleNamespace(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, conv=taps, decay="channel", gate="sigmoid", conv_channels=2 * kv_heads * dim + heads * vdim)
    key = (heads, dim, vdim)
    recs = {key} if r._rec_tiles_take(m, taps) and (not delta or r._delta_recurs(m)) else set()
    work = r._scan_work(rows, 1, rows, {key}, delta=delta, recs=recs)
    assert bool(work) == held
    calls = []

    class Recorder:
        def __getattr__(self, name):
            if name in ("linear", "causal_conv", "gdn_gates", "gdn_scan", "gla_scan", "gate_norm", "rec_step", "rec_tiles"):
                return lambda *a, **kw: calls.append((name, kw))
            return getattr(D, name)

    monkeypatch.setattr(hybrid_runner, "D", Recorder())
    B = SimpleNamespace(**{k: torch.empty(rows * heads * 4 * 256) for k in ("a", "b", "c", "f", "g", "r", "rn", "z")})
    B.c16, B.rn16 = B.c.bfloat16(), B.rn.bfloat16()
    d = {k: 0 for k in ("r_off", "rb_off", "a1_off", "g1_off", "rq_off", "rk_off", "rv_off", "rg_off")}
    d.update({k: None for k in ("a2", "g2", "dt_bias", "a_rate", "conv_w", "r_norm", "o_right", "a2_b")})
    state = {"gdn": None, "gla": None, **({"conv": None} if taps > 1 else {})}
    args = (B, d, m, torch.empty(rows, 8), 0, rows, None, None, SimpleNamespace(state=[state]), None, 1)
    if delta:
        r._gated_delta(*args, False, None, work, rows)
    else:
        r._gated_linear(*args, None, 1.0, work, rows)
    took = [n for n, kw in calls if n == "rec_tiles" or (n in ("gdn_scan", "gla_scan") and kw["work"] is not None and D.scan_in_tiles(rows, 1, rows, *key, delta=delta))]
    assert bool(took) == held
