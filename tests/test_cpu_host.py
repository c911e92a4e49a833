"""CPU-side checks of the host code: the C ABI library loads and exports every declared symbol, header and binding agree,
the synthetic-weight generator follows the oracle's protocol, N>1 launch plumbing (gloo, world_size 2)."""
import os
import re
import subprocess
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol():
    import ctypes
    from vllm_i64_amd import _lib, build
    path = build.build(verbose=False)
    lib = ctypes.CDLL(path)
    hdr = open(os.path.join(ROOT, "include", "i64h.h")).read()
    declared = set(re.findall(r"\b(i64h_[a-z0-9_]+)\s*\(", hdr))
    assert declared, "no declarations parsed"
    for name in sorted(declared):
        assert hasattr(lib, name), f"{name} declared in include/i64h.h but not exported"
    bound = set(_lib.exported_symbols())
    assert bound <= declared, f"bound but not declared: {bound - declared}"
    assert declared <= bound, f"declared but not bound: {declared - bound}"


def test_binding_signature_lengths_match_header():
    from vllm_i64_amd import _lib
    hdr = open(os.path.join(ROOT, "include", "i64h.h")).read()
    hdr = re.sub(r"/\*.*?\*/", "", hdr, flags=re.S)
    for name, sig in _lib.SIGNATURES.items():
        m = re.search(r"\bint\s+" + name + r"\s*\((.*?)\)\s*;", hdr, flags=re.S)
        assert m, name
        nargs = len([a for a in m.group(1).split(",") if a.strip() and a.strip() != "void"])
        assert nargs == len(sig), f"{name}: header has {nargs} parameters, binding {len(sig)}"


def test_no_cpu_fallback_and_no_oracle_import_in_product():
    from vllm_i64_amd import kernels
    if not torch.cuda.is_available():
        assert kernels.get_i64_cuda_ops() is None
        with pytest.raises(RuntimeError):
            kernels.get_ops()
    pkg = os.path.join(ROOT, "vllm_i64_amd")
    for fn in os.listdir(pkg):
        if fn.endswith(".py"):
            src = open(os.path.join(pkg, fn)).read()
            assert "oracle" not in src.replace("the oracle's", "").replace("oracle's", ""), f"{fn} mentions the oracle package"


def test_synth_matches_oracle_protocol():
    from oracle import model_ref as M
    from vllm_i64_amd import synth
    from vllm_i64_amd.config import ModelConfig
    for name in ("tiny-moe", "tiny-cyclic", "tiny-dense"):
        ocfg = M.named_config(name)
        cfg = ModelConfig.from_any(ocfg)
        a, b = M.make_weights(ocfg, seed=0), synth.make_weights(cfg, seed=0)
        assert a.keys() == b.keys()
        for k in a:
            assert torch.equal(a[k], b[k]), k
        assert torch.equal(M.make_token_ids(ocfg, 50), synth.make_token_ids(cfg, 50))
    from vllm_i64_amd.config import trhash500m_synth
    c = trhash500m_synth()
    oc = M.named_config("trhash500m-synth")
    assert oc.num_parameters() == 492_100_608 or abs(oc.num_parameters() - 492.1e6) < 0.1e6
    assert c.route_weights == [0.5, 0.5]


_WORKER = r"""
import os, sys, time, torch, torch.distributed as dist
dist.init_process_group("gloo")
rank, world = dist.get_rank(), dist.get_world_size()
# same reduction bench.py does after the timed region: barrier, then MAX of the per-rank elapsed time
dist.barrier()
t = torch.tensor([0.1 * (rank + 1)], dtype=torch.float64)
dist.all_reduce(t, op=dist.ReduceOp.MAX)
tokens = 64 * world * 10 / float(t.item())
if rank == 0:
    print("RESULT", world, round(float(t.item()), 3), round(tokens, 1))
dist.destroy_process_group()
"""


def test_multi_rank_timing_reduction_gloo(tmp_path):
    """world_size-2 rehearsal of bench.py's N>1 protocol on CPU (gloo): every rank runs its own replica, elapsed = MAX over
    ranks, value = all ranks' tokens / that time."""
    script = tmp_path / "w.py"
    script.write_text(_WORKER)
    env = dict(os.environ, MASTER_ADDR="127.0.0.1")
    r = subprocess.run([sys.executable, "-m", "torch.distributed.run", "--nnodes=1", "--nproc-per-node", "2", "--master-addr", "127.0.0.1",
                        "--master-port", "29533", str(script)], capture_output=True, text=True, env=env, timeout=240)
    assert r.returncode == 0, r.stderr[-2000:]
    line = [l for l in r.stdout.splitlines() if l.startswith("RESULT")][0].split()
    assert int(line[1]) == 2 and float(line[2]) == 0.2 and float(line[3]) == 6400.0


def test_baseline_config_1_dense_batch1_greedy_on_the_cpu_engine():
    """BASELINE configuration 1 (dense-306, --quantization int8, CPU engine, greedy decode, batch 1): the plumbing case that runs
    without a GPU.  The oracle's engine with torch's own dynamic int8 Linears (the reference's quantized kernels) at the config's
    real width, four layers deep to keep the CPU suite short: deterministic, finite logits, and the numpy restatement of the
    quantized Linear gives the same greedy tokens."""
    import dataclasses
    from oracle import model_ref as M
    cfg = dataclasses.replace(M.named_config("dense306-synth"), num_layers=4, vocab_size=2048, name="dense306-4layer")
    w = M.make_weights(cfg, seed=0)
    prompt = M.make_token_ids(cfg, 24, seed=7)
    runs = []
    for mode in ("int8_torch", "int8_torch", "int8"):
        eng = M.OracleEngine(cfg, w, mode=mode, max_seqs=1, num_blocks=8)
        lg = eng.prefill([prompt])
        toks, logits = [], [lg]
        for _ in range(6):
            t = lg.argmax(-1)
            toks.append(int(t))
            lg = eng.decode(t)
            logits.append(lg)
        runs.append((toks, torch.cat(logits)))
    assert runs[0][0] == runs[1][0] and torch.equal(runs[0][1], runs[1][1])          # deterministic
    assert torch.isfinite(runs[0][1]).all()
    assert runs[2][0] == runs[0][0] and torch.equal(runs[2][1], runs[0][1])          # restatement == torch's kernels, bit for bit


def test_engine_adapter_per_sequence_position_maxima():
    """Host logic of the engine adapter: the highest position of each sequence of a step (what decides the blocks to allocate and
    the new seq_lens), with sequences that contribute no token and positions that are not ascending inside a sequence."""
    from vllm_i64_amd.engine_adapter import max_positions
    pos = torch.tensor([5, 6, 7, 40, 2, 9, 3, 11])
    assert max_positions(pos, [3, 1, 0, 4]) == [7, 40, -1, 11]
    assert max_positions(pos, [0, 8, 0]) == [-1, 40, -1]
    assert max_positions(pos[:0], []) == [] and max_positions(pos[:0], [0, 0]) == [-1, -1]
    assert max_positions(pos[:3], [0, 0, 3]) == [-1, -1, 7] and max_positions(pos[:1], [1]) == [5]


def test_attention_segments_of_a_step():
    """Host logic of the runner's attention plan: decode rows and prefill chunks of a mixed engine step become runs of a kind."""
    from vllm_i64_amd.model import attention_segments
    assert attention_segments([1] * 5, 5, 4) == [(0, 5, True)]
    assert attention_segments([512], 512, 4) == [(0, 512, False)]
    assert attention_segments([512, 1, 1, 0, 1], 515, 4) == [(0, 512, False), (512, 515, True)]
    assert attention_segments([1, 1, 20, 30, 1, 0, 7], 60, 4) == [(0, 2, True), (2, 52, False), (52, 53, True), (53, 60, False)]
    assert attention_segments([1, 17] * 40, 720, 4) == [(0, 720, False)]        # 80 runs: one launch, mostly chunk rows
    assert attention_segments([1, 1, 1, 2] * 10, 50, 4) == [(0, 50, True)]      # ... mostly decode rows
    assert attention_segments([], 0, 4) == [] and attention_segments([0, 0], 0, 4) == []
    with pytest.raises(ValueError):
        attention_segments([3, 1], 5, 4)


def test_linear_takes_numbers_of_any_kind(monkeypatch):
    """Switches and distances may come as numpy or float numbers, factors as tensors: a descriptor holds their values."""
    import numpy as np
    import torch
    from vllm_i64_amd import ops_dense as D
    seen = []
    for name, stand_in in (("_chk", lambda *a: None), ("_stream", lambda: 0), ("ptr", lambda t: 0), ("_ref", lambda d: d), ("call_dense", lambda name, d, stream: seen.append(d))):
        monkeypatch.setattr(D, name, stand_in)
    a, w, out = torch.zeros(3, 32), torch.zeros(2, 8, 32, dtype=torch.bfloat16), torch.zeros(3, 16)
    for exact, apart, scale in ((True, 8, 2.5), (np.bool_(True), np.int64(8), np.float32(2.5)), (1.0, 8.0, torch.tensor(2.5))):
        D.linear(a, w, out, n=8, batch=2, w_batch=256, c_batch=8, bias=torch.zeros(2, 8), bias_batch=apart, exact=exact, epilogue=D.EPI_SCALE, scale=scale)
        assert (seen[-1].exact, seen[-1].bias_batch, seen[-1].scale) == (1, 8, 2.5)


@pytest.mark.parametrize("top_k,experts,hidden,inter,shared,rows", [(2, 8, 1024, 512, 512, 362), (1, 256, 16, 16, 0, 42532), (2, 128, 64, 16, 0, 9551), (8, 32, 32, 16, 16, 3421), (2, 4, 128, 64, 64, 2843),
                                                                    (1, 64, 256, 128, 0, 4278)])
def test_rows_that_fit_the_library_s_own_scratch(top_k, experts, hidden, inter, shared, rows):
    """The entry point that allocates nothing takes so many rows of these layers, however many rows a wave of its plan counts."""
    import ctypes
    from vllm_i64_amd import _lib
    lib = _lib.load()
    L = _lib.MoeLayer(top_k=top_k, num_experts=experts, hidden=hidden, expert_inter=inter, shared_inter=shared)
    assert 0 < lib.i64h_moe_forward_workspace_bytes(rows, ctypes.addressof(L)) <= lib.i64h_moe_forward_static_max_bytes()


def test_operands_that_a_launch_would_read_or_write_out_of_bounds_are_refused():
    """C entries called past the Python checks: the refusal comes before anything is launched (addresses that are none)."""
    import ctypes
    from vllm_i64_amd import _lib
    at, lib, dense = 1 << 20, _lib.load(), _lib.load_dense()
    w8 = (ctypes.c_float * 8)()
    assert lib.i64h_fused_residual_norm_lm_rows(at, 0, 0, 0, 0, ctypes.addressof(w8), 0, 1.0, 1.0, 0, 1e-6, 4, 64, at, 2, at, 0) != 0
    assert b"norm's weights" in lib.i64h_last_error()
    base = dict(P=at, ldp=2048, heads=2, dim=64, vdim=64, a_off=384, a_rank=8, A=at, a_bias=at, a_rate=at, norm_w=at, positions=at, slot_ids=at, state=at, out=at, ldo=128, n=3, z_off=512)
    linear, delta = dict(base, k_off=128, v_off=256), dict(base, conv_w=at, conv=at, taps=4, Z=at, z_rank=8, b_off=600)
    for args in (dict(linear, ldo=127), dict(linear, k_off=2000), dict(linear, v_off=1924), dict(linear, z_off=1924), dict(linear, a_off=2044), dict(delta, q_off=1668), dict(delta, b_off=2047),
                 dict(delta, z_off=2044)):
        d = _lib.RecStep(**args)
        assert dense.i64h_rec_step(ctypes.addressof(d), 0) != 0 and b"behind the row's end" in dense.i64h_last_error(), args
    d = _lib.RecStep(**delta)
    for x in (dict(ldx=127), dict(ldx=128, v_off=4), dict(ldx=256, v_off=-4)):
        s = _lib.Gdn(**{**dict(X=at, seg_start=at, nseg=1, out=at, ldo=128, work=at, work_floats=1 << 40), **x})
        assert dense.i64h_rec_tiles(ctypes.addressof(d), ctypes.addressof(s), 0) != 0 and b"rows for the read-out" in dense.i64h_last_error(), x
