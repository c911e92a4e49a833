"""e4m3 products on rows quantized beforehand against the launches that quantize the rows themselves: the same codes, the same order of the sums, the same
bits - at sizes around the tiles' edges, row lengths of whole and half steps, gathered and grouped rows, the qkv tail, whole steps of a model."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


def weights(dev, g, *shape):
    from vllm_i64_amd import ops
    w = torch.randn(*shape, generator=g, device=dev) * 0.05
    q, s = ops.quantize_fp8_rows(w.reshape(-1, shape[-1]))
    return q.view(shape), s.view(shape[:-1])


@pytest.mark.parametrize("n0,K0,n1,K1", [(1, 4, 0, 4), (5, 448, 7, 1792), (64, 2048, 3, 2052), (9, 4100, 1, 64)])
def test_quantizer_of_two_matrices(dev, n0, K0, n1, K1):
    from vllm_i64_amd import ops
    g = torch.Generator(device=dev).manual_seed(n0 + K1)
    x0, x1 = torch.randn(n0, K0, generator=g, device=dev), torch.randn(max(n1, 1), K1, generator=g, device=dev)[:n1]
    x0[0, 0] = float("nan")
    if n0 > 3:
        x0[1, 1], x0[2] = float("inf"), 0.0
    outs = []
    for x in (x0, x1):
        outs += [torch.zeros(x.shape, dtype=torch.uint8, device=dev), torch.zeros(x.shape[0], device=dev)]
    ops.quantize_fp8_rows_pair(x0, outs[0], outs[1], *((x1, outs[2], outs[3]) if n1 else ()))
    for x, q, s in ((x0, outs[0], outs[1]), (x1, outs[2], outs[3])):
        if x.shape[0]:
            wq, ws = ops.quantize_fp8_rows(x)
            assert torch.equal(q, wq) and torch.equal(s.view(torch.int32), ws.view(torch.int32))


@pytest.mark.parametrize("M,N,K", [(1, 16, 64), (63, 48, 128), (64, 64, 192), (65, 80, 448), (130, 256, 640), (257, 1536, 1024)])
def test_same_bits_as_rows_quantized_in_the_launch(dev, M, N, K):
    from vllm_i64_amd import ops
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=dev)
    w, s = weights(dev, g, 2 * N, K)
    q, xs = ops.quantize_fp8_rows(x)
    for epi, rows in ((ops.EPI_STORE, N), (ops.EPI_SWIGLU, 2 * N)):
        want, got = torch.full((M + 1, N), 7.0, device=dev), torch.full((M + 1, N), 7.0, device=dev)
        ops.gemm_fp8_rows(x, w[:rows], s[:rows], want, epilogue=epi)
        ops.gemm_fp8_codes_pair(ops.fp8_codes_desc(q, xs, w[:rows], s[:rows], got), epilogue=epi)
        assert torch.equal(got, want)
    h = torch.randn(M, N, generator=g, device=dev)
    want, got = h.clone(), h.clone()
    ops.gemm_fp8_rows(x, w[:N], s[:N], want, c_add=want)
    ops.gemm_fp8_codes_pair(ops.fp8_codes_desc(q, xs, w[:N], s[:N], got, c_add=got))
    assert torch.equal(got, want)


@pytest.mark.parametrize("counts", [[5, 0, 70, 1], [0, 0, 0, 129], [64, 16, 128, 0], [1] * 70])
def test_rows_grouped_by_expert_beside_a_second_problem(dev, counts):
    from vllm_i64_amd import ops
    G, N, K, I, n = len(counts), 64, 192, 448, 150
    g = torch.Generator(device=dev).manual_seed(sum(counts))
    off = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(dev)
    R = int(off[-1])
    perm = torch.randint(0, 2 * n, (R,), generator=g, device=dev).to(torch.int32)
    x = torch.randn(n, K, generator=g, device=dev)
    q, xs = ops.quantize_fp8_rows(x)
    (we, se), (w2, s2) = weights(dev, g, G, 2 * N, K), weights(dev, g, 2 * N, K)
    outs = [torch.full((R, N), 7.0, device=dev) for _ in range(2)], [torch.full((n, N), 7.0, device=dev) for _ in range(2)]
    kw = dict(m=R, a_src_row=perm, a_src_mod=n, group_offsets=off)
    ops.gemm_fp8_rows_pair(ops.fp8_rows_desc(x, w2, s2, outs[1][0]), ops.fp8_rows_desc(x, we, se, outs[0][0], **kw), epilogue=ops.EPI_SWIGLU)
    ops.gemm_fp8_codes_pair(ops.fp8_codes_desc(q, xs, w2, s2, outs[1][1]), ops.fp8_codes_desc(q, xs, we, se, outs[0][1], **kw), epilogue=ops.EPI_SWIGLU)
    assert torch.equal(outs[0][0], outs[0][1]) and torch.equal(outs[1][0], outs[1][1])
    y = torch.randn(R, I, generator=g, device=dev)
    qy, ys = ops.quantize_fp8_rows(y)
    wd, sd = weights(dev, g, G, 96, I)
    place = torch.randperm(R, generator=g, device=dev).to(torch.int32)
    want, got = torch.full((R, 96), 7.0, device=dev), torch.full((R, 96), 7.0, device=dev)
    kw = dict(m=R, group_offsets=off, c_row_map=place)
    ops.gemm_fp8_rows_pair(ops.fp8_rows_desc(y, wd, sd, want, **kw))
    ops.gemm_fp8_codes_pair(ops.fp8_codes_desc(qy, ys, wd, sd, got, **kw))
    assert torch.equal(got, want)


@pytest.mark.parametrize("norm", [True, False])
@pytest.mark.parametrize("kv_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 64, 131])
def test_qkv_with_its_tail(dev, n, kv_dtype, norm):
    from vllm_i64_amd import ops
    from vllm_i64_amd.model import rope_table
    nh, kvh, hd, H = 4, 2, 64, 320
    g = torch.Generator(device=dev).manual_seed(n)
    x = torch.randn(n, H, generator=g, device=dev)
    w, s = weights(dev, g, (nh + 2 * kvh) * hd, H)
    q, xs = ops.quantize_fp8_rows(x)
    qw, kw = (torch.rand(hd, generator=g, device=dev) + 0.5 for _ in range(2))
    pos, slots = torch.arange(n, dtype=torch.int32, device=dev), torch.zeros(n, dtype=torch.int32, device=dev)
    blocks = (n + 15) // 16 + 1
    table = torch.arange(blocks, dtype=torch.int32, device=dev).flip(0).view(1, -1).contiguous()
    table[0, 1] = -1      # a page that the sequence does not own: nothing is written there
    rope = rope_table(256, hd, 10000.0).to(dev)
    res = []
    for codes in (False, True):
        k, v = (torch.full((blocks, 16, kvh, hd), 3.0, device=dev).to(kv_dtype) for _ in range(2))
        qo, qkv = torch.empty(n, nh, hd, device=dev), torch.empty(n, w.shape[0], device=dev)
        args = (qw if norm else None, kw if norm else None, 1e-6, rope, pos, slots, table, k, v, qo, nh, kvh, hd)
        if codes:
            ops.gemm_fp8_codes_qkv_rope_kv(ops.fp8_codes_desc(q, xs, w, s, None), *args)
        else:
            ops.gemm_fp8_rows_qkv_rope_kv(ops.fp8_rows_desc(x, w, s, qkv), *args)
        res.append((qo, k, v))
    assert all(torch.equal(a, b) for a, b in zip(*res))


@pytest.mark.parametrize("moe", [True, False])
def test_step_of_a_model(dev, moe):
    """A prompt of 300 rows on codes and with the rows quantized in front of every launch's tiles: the same logits and cache."""
    import dataclasses
    from oracle import model_ref as M
    from vllm_i64_amd.config import ModelConfig
    from vllm_i64_amd.model import I64MoEModel
    ocfg = dataclasses.replace(M.named_config("trhash500m-synth"), num_layers=2, vocab_size=500, name="cut", **({} if moe else dict(num_experts=1, shared_intermediate_size=0, top_k=1, intermediate_size=1024)))
    w = M.make_weights(ocfg, seed=1)
    model = I64MoEModel(ModelConfig.from_any(ocfg), w, device=dev, max_seqs=2, num_kv_blocks=64, quant="fp8")
    n = 300
    ids = torch.randint(0, 500, (n,), generator=torch.Generator().manual_seed(2)).to(dev)
    pos, slots = torch.arange(n, dtype=torch.int32, device=dev), torch.zeros(n, dtype=torch.int32, device=dev)
    model.kv.reserve(0, n)
    runs = []
    for tiles in (False, True):
        model.FP8_TILE_ROWS = model.FP8_TILE_ROWS_MOE = 1 if tiles else 1 << 30
        assert model._fp8_tiles(n) == tiles
        lg = model.forward(ids, pos, slots, (pos + 1).contiguous(), max_ctx_hint=n, tokens_per_seq=[n])
        runs.append([lg.clone()] + [t.clone() for t in (*model.kv.k, *model.kv.v)])
    assert all(torch.equal(a, b) for a, b in zip(*runs)) and bool(runs[0][0].isfinite().all())


@pytest.mark.parametrize("moe", [True, False])
@pytest.mark.parametrize("decode,prompt", [(31, 269), (40, 660), (7, 2093)])
def test_mixed_steps_of_a_model(dev, moe, decode, prompt):
    """Decoding sequences beside a new prompt on each of the three ways: rows quantized in front of every launch's tiles, once for the older tiled products, once for
    the 64 x 64 tiles.  The first and the last give the same logits and cache bit for bit."""
    import dataclasses
    from oracle import model_ref as M
    from vllm_i64_amd.config import ModelConfig
    from vllm_i64_amd.model import I64MoEModel
    ocfg = dataclasses.replace(M.named_config("trhash500m-synth"), num_layers=2, vocab_size=500, name="cut", **({} if moe else dict(num_experts=1, shared_intermediate_size=0, top_k=1, intermediate_size=1024)))
    model = I64MoEModel(ModelConfig.from_any(ocfg), M.make_weights(ocfg, seed=1), device=dev, max_seqs=decode + 1, num_kv_blocks=3 * decode + prompt // 16 + 2, quant="fp8")
    g = torch.Generator().manual_seed(decode)
    past = [5 + 2 * s % 30 for s in range(decode)]
    for s, p in enumerate(past + [0]):
        model.kv.reserve(s, p + (1 if s < decode else prompt))
    for t in (*model.kv.k, *model.kv.v):
        t.copy_(torch.randn(t.shape, generator=g))
    held = [t.clone() for t in (*model.kv.k, *model.kv.v)]
    ids = torch.randint(0, 500, (decode + prompt,), generator=g).to(dev)
    pos = torch.cat([torch.tensor(past), torch.arange(prompt)]).to(torch.int32).to(dev)
    slots = torch.cat([torch.arange(decode), torch.full((prompt,), decode)]).to(torch.int32).to(dev)
    tps = [1] * decode + [prompt]
    runs = []
    for tiles, fused in ((False, 1 << 30), (False, 0), (True, 1024)):
        model.FP8_TILE_ROWS = model.FP8_TILE_ROWS_MOE = 1 if tiles else 1 << 30
        model.FP8_FUSE_MAX_ROWS = fused
        for t, h in zip((*model.kv.k, *model.kv.v), held):
            t.copy_(h)
        lg = model.forward(ids, pos, slots, (pos + 1).contiguous(), max_ctx_hint=max(past + [prompt]) + 1, tokens_per_seq=tps)
        runs.append([lg.clone()] + [t.clone() for t in (*model.kv.k, *model.kv.v)])
    assert all(torch.equal(a, b) for a, b in zip(runs[2], runs[0]))
    # the older tiles add in another order: 2^-24 of a sum, and where that moves a code of the next product by a step (a sixteenth of one of 1024 or more terms) 2e-3 of a
    # row - a few rows of these steps at the outside
    assert all(float((a.double() - b.double()).norm() / b.double().norm()) < 1e-3 for a, b in zip(runs[2], runs[1]))
    assert bool(runs[2][0].isfinite().all())


def test_which_steps_take_the_tiles():
    """Neither an eager step that more launches bind to the host nor a recording one."""
    from oracle import model_ref as M
    from vllm_i64_amd.config import ModelConfig
    from vllm_i64_amd.model import I64MoEModel
    for moe, first in ((True, 256), (False, 176)):
        m = I64MoEModel.__new__(I64MoEModel)
        m.cfg = ModelConfig.from_any(M.named_config("trhash500m-synth" if moe else "dense306-synth"))
        m.layers = [dict(q_norm=None, k_norm=None)]
        assert [m._fp8_tiles(n) for n in (1, first - 1, first, 12288, 12289)] == [False, False, True, True, False]
