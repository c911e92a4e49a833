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
