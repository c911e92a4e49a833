"""Where a shared expert of the experts' size runs, and what its step buffers hold: the rows of one place only."""
import pytest
import torch

from tests import joined_shapes, pukatar_shapes, vepelix_shapes


def make(monkeypatch, design):
    from vllm_i64_amd.config import PukatarConfig, VepelixConfig
    from vllm_i64_amd.pukatar import PukatarModel
    from vllm_i64_amd.vepelix import VepelixModel
    joined_shapes.use(monkeypatch, design)
    shapes = vepelix_shapes if design == "vepelix" else pukatar_shapes
    model, config = (VepelixModel, VepelixConfig) if design == "vepelix" else (PukatarModel, PukatarConfig)
    return model(config.from_dict(shapes.config_of("joined")), shapes.make_weights("joined"), device="cpu", num_kv_blocks=4)


@pytest.mark.parametrize("design", ["vepelix", "pukatar"])
def test_apart_only_where_it_runs_beside_something(monkeypatch, design):
    m = make(monkeypatch, design)
    assert m.side is None and all(m._joins(n) for n in (1, 100, 1 << 20))      # no second stream: nothing to run beside
    m.side = object()
    m.FORK_WORK = 128 * 128 * 200
    assert m._joins(199) and m._joins(200) == (design == "pukatar")


@pytest.mark.parametrize("width,rows,exact", [(1024, 1574, False), (2048, 394, False), (1024, 787, True)])
def test_a_step_forks_where_its_launches_outlast_the_host(width, rows, exact):
    """Rows times the square of the width: a fork's events cost the host the same whatever the width."""
    from types import SimpleNamespace
    from vllm_i64_amd.hybrid_runner import HybridRunner
    r = HybridRunner.__new__(HybridRunner)
    r.cfg, r.exact, r.side = SimpleNamespace(width=width), exact, object()
    assert not r._heavy(rows - 1) and r._heavy(rows) and r._forks(rows)


@pytest.mark.parametrize("design", ["vepelix", "pukatar"])
def test_buffers_hold_the_rows_of_one_place(monkeypatch, design):
    m = make(monkeypatch, design)
    m.side = object()
    n, W = 200, 128
    for work, joined in ((1 << 40, True), (0, design == "pukatar")):
        m.FORK_WORK = work
        B = type(m).BUFFERS(m, n, 1)
        assert B.joined == joined
        # layer 3's shared expert is never in the stack; the widest grouped rows are layer 1's: three experts of 128, and the shared one where it joins
        assert B.ey.numel() == n * (4 if joined else 3) * W and B.act.numel() == n * (4 if joined else 3) * 128
        assert B.sact.numel() == n * ((96 if design == "vepelix" else 64) if joined else 128)
        assert B.pair_token.numel() == n * (4 if joined else 3) and B.group_off.numel() >= 7 + 1 + int(joined)
    m.cfg.layers = m.cfg.layers[:3]
    m._moe_sizes([l.mlp for l in m.cfg.layers])
    m.FORK_WORK = 1 << 40
    B = type(m).BUFFERS(m, n, 1)
    assert B.sact.numel() == n and (design == "vepelix" or B.y3.numel() == 0)      # every one joined: nothing beside the grouped rows
