"""Mixtures whose shared expert has the experts' size: joined to their grouped launches, beside them on the side stream, and with weights of its own - whole
steps against the 64-bit oracle and against each other, rows in fp32 and in bf16."""
import importlib

import pytest
import torch

from tests import joined_shapes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


@pytest.mark.parametrize("n", [7, 64, 200])
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("design", ["vepelix", "pukatar"])
def test_whole_steps(dev, monkeypatch, design, dtype, n):
    from vllm_i64_amd.hybrid_runner import HybridRunner
    gpu = importlib.import_module("tests.test_gpu_%s" % design)
    joined_shapes.use(monkeypatch, design)
    toks = gpu.tokens("joined", n, 5)
    got = {}
    for name, work in (("joined", 1 << 60), ("forked", 0), ("own", 1 << 60), ("thin", 1 << 60)):
        with monkeypatch.context() as mp:
            if name == "own":
                mp.setattr(HybridRunner, "_shared_in_stack", staticmethod(lambda f: False))
            if name == "thin":      # (as with many experts of a few rows each: fp32 rows beside the others' bf16)
                mp.setattr(HybridRunner, "_fills", staticmethod(lambda pairs, experts: False))
            model = gpu.make_model("joined", dtype, dev)
            model.FORK_WORK = work
            assert [d.get("merged") for d in model.layers] == [name != "own", name != "own", None, False]
            assert model._joins(n) == (work > 0 or design == "pukatar") and model._forks(n) == (work == 0)
            got[name] = gpu.whole_prompt(model, "joined", toks, dtype, layers_too=True)      # (checks against the oracle)
    assert all(gpu.same_to_rounding(got[k], got["joined"], dtype) for k in got)
    if design == "pukatar":      # (the same launches on one stream or two)
        assert torch.equal(got["forked"], got["joined"])


@pytest.mark.parametrize("design", ["vepelix", "pukatar"])
def test_captured_steps(dev, monkeypatch, design):
    """Captured decode steps of three sequences against the same tokens in one prompt each."""
    from vllm_i64_amd.model import GreedyDecoder
    gpu = importlib.import_module("tests.test_gpu_%s" % design)
    joined_shapes.use(monkeypatch, design)
    model = gpu.make_model("joined", "float32", dev, max_tokens=256, max_seqs=3)
    prompts = [gpu.tokens("joined", n, 40 + n) for n in (4, 11, 17)]
    dec = GreedyDecoder(model, 3, use_graph=True)
    dec.prefill([torch.tensor(p) for p in prompts], reserve_extra=12)
    seqs = [list(p) + [int(t)] for p, t in zip(prompts, dec.tokens.tolist())]
    for _ in range(5):
        dec.step()
        torch.cuda.synchronize()
        for s, t in zip(seqs, dec.tokens.tolist()):
            s.append(int(t))
    for p, s in zip(prompts, seqs):
        t = list(p)
        for _ in range(6):
            t.append(int(gpu.oracle_logits("joined", t)[-1].argmax()))
        assert s == t
