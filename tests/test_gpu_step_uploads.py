"""What a step brings to the device: one upload of the engine's lists, run starts through page-locked memory; and a step that forks to the side stream or does
not, with the same results."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_engine_upload_parts():
    from vllm_i64_amd.engine import Engine
    e = Engine.__new__(Engine)
    e.device = torch.device("cuda:0")
    for n in (1, 2, 3, 4, 77, 1001):
        ids, pos, slots = [(1 << 40) + i for i in range(n)], list(range(5, 5 + n)), [i % 3 for i in range(n)]
        for rows in ([], [n - 1], list(range(n))):
            t = e._upload(ids, pos, slots, rows)
            assert [x.dtype for x in t] == [torch.int64] + [torch.int32] * 4 and all(x.is_contiguous() and x.data_ptr() % 16 == 0 for x in t)
            assert t[0].tolist() == ids and t[1].tolist() == pos and t[2].tolist() == slots and t[3].tolist() == [p + 1 for p in pos] and t[4].tolist() == (rows or [0])


def test_uploads_follow_each_other():
    """Page-locked memory that a finished call gave back is not written again before its copy has run."""
    from vllm_i64_amd.ops import upload
    dev = torch.device("cuda:0")
    x = torch.randn(2048, 2048, device=dev)
    got = []
    for i in range(50):
        x = torch.tanh(x @ x)      # (keeps the stream busy while the host runs ahead)
        got.append(upload([i] * 500, torch.int32, dev))
    assert all(t.tolist() == [i] * 500 for i, t in enumerate(got))


@pytest.mark.parametrize("design", ["vepelix", "pukatar"])
def test_forked_or_not(design):
    import importlib
    gpu = importlib.import_module("tests.test_gpu_%s" % design)
    dev = torch.device("cuda:0")
    outs = []
    for work in (0, 1 << 60):
        model = gpu.make_model("plain", "bfloat16", dev, max_tokens=256)
        model.FORK_WORK = work
        n = 100
        model.kv.reserve(0, n)
        assert model._forks(n) == (work == 0)
        ids = torch.randint(0, model.cfg.vocab, (n,), generator=torch.Generator().manual_seed(1)).to(dev)
        pos, slots = torch.arange(n, dtype=torch.int32, device=dev), torch.zeros(n, dtype=torch.int32, device=dev)
        outs.append(model.forward(ids, pos, slots, None, max_ctx_hint=n, tokens_per_seq=[n]).clone())
    assert torch.equal(*outs)
