"""What is timed: steps of the framework's runners as a serving program makes them, through its public entry points.

A case names a model, the arithmetic of its Linears, and a batch.  A batch is written "sequences * new tokens @ tokens already cached", parts
joined by "+": "64*1@2048" is a decode step of 64 sequences with 2048 cached tokens each, "8*512@0" a prefill of eight 512-token prompts,
"31*1@700+1*481@0" the step of a continuous batch in which 31 sequences decode beside one new prompt.

models   moe, dense       token-routed mixture / plain feed-forward with quantized Linears ("int8": dynamic per call, "fp8": per token), the
                          layer sizes of trhash500m-synth and dense306-synth, two layers of them: behind more, a rounding tie of a 7-bit code
                          in one layer moves every later one, and nothing could be compared
         vepelix, pukatar hybrid designs at the layer sizes of `bench.py --design` (bf16 weights; "bf16": inputs of matrix products rounded to bf16,
                          "f32": true 32-bit products), one block of four layers, run `times` times
         sampler          the draw of the next tokens from a step's logits

drive    "graph"    GreedyDecoder: the captured decode step, put back to the same position before every pass
         "forward"  the runner's step interface, as the benchmark and a scheduler call it
         "engine"   Engine.step on token lists; the requests end with the step
"""
import math
import zlib

import torch

from vllm_i64_amd import ops_dense, synth
from vllm_i64_amd.config import ModelConfig
from vllm_i64_amd.engine import Engine
from vllm_i64_amd.model import GreedyDecoder, I64MoEModel
from vllm_i64_amd.pukatar import PukatarModel
from vllm_i64_amd.vepelix import VepelixModel

DEV = "cuda:0"
F64 = torch.float64
VOCAB, PAGE, RANK = 32000, 16, 128

MOE = {
    "moe": dict(name="moe", num_layers=2),      # the defaults are trhash500m-synth's
    "dense": dict(name="dense", num_layers=2, intermediate_size=4096, num_experts=1, shared_intermediate_size=0, top_k=1, primary_weight=1.0, table_routing=False),
}
VEPELIX = {
    1024: dict(width=1024, heads=16, dim=64, rot_dim=32, vdim=64, kv_rank=256, q_rank=512, left_heads=16, left_kv_heads=4, left_dim=64, left_vdim=64,
               window=1024, rec_heads=8, rec_dim=128, rec_vdim=128, ff=2752, experts=8, top=2, expert_ff=896, shared_ff=896),
    2048: dict(width=2048, heads=32, dim=64, rot_dim=32, vdim=64, kv_rank=256, q_rank=768, left_heads=32, left_kv_heads=8, left_dim=64, left_vdim=64,
               window=1024, rec_heads=16, rec_dim=128, rec_vdim=128, ff=5504, experts=8, top=2, expert_ff=1792, shared_ff=1792),
}
PUKATAR = {
    1024: dict(width=1024, heads=16, kv_heads=4, dim=64, vdim=64, rot_dims=64, window=1024, keep_first=4, rec_heads=8, rec_kv_heads=8, rec_dim=128,
               rec_vdim=128, taps=4, ff=2752, experts=8, top=2, expert_ff=896, shared_ff=896),
    2048: dict(width=2048, heads=32, kv_heads=8, dim=64, vdim=64, rot_dims=64, window=1024, keep_first=4, rec_heads=16, rec_kv_heads=16, rec_dim=128,
               rec_vdim=128, taps=4, ff=5504, experts=8, top=2, expert_ff=1792, shared_ff=1792),
}
EPS = 1e-6
OUT = 0.02 / 32 ** 0.5      # of matrices that write the residual: the usual 1 / sqrt(2 layers) at sixteen layers


def _case(model, batch, drive, arith="bf16", width=1024, times=1):
    return dict(model=model, batch=batch, drive=drive, arith=arith, width=width, times=times)


def listed():
    c = _case
    return [
        # the headline workload's decode step: 64 conversations, 2048 tokens in
        dict(name="moe_decode_64", **c("moe", "64*1@2048", "graph", "int8")),
        # one interactive user of the plain model: latency
        dict(name="dense_decode_1", **c("dense", "1*1@517", "graph", "int8")),
        # the headline workload's prefill chunk: eight 2048-token prompts
        dict(name="moe_prefill_8x2048", **c("moe", "8*2048@0", "forward", "int8")),
        # continuous batching with fp8 Linears: the scheduler's default step, 31 decoding sequences beside the rest of a 512-token budget
        dict(name="moe_fp8_mixed", **c("moe", "31*1@700+1*481@0", "forward", "fp8")),
        # a hybrid design's prefill step of 4096 rows
        dict(name="vepelix_prefill_8x512", **c("vepelix", "8*512@0", "forward", width=1024, times=2)),
        # its decode step at full batch, the wide size
        dict(name="vepelix_decode_64", **c("vepelix", "64*1@2048", "graph", width=2048, times=2)),
        # time to the first token of one short prompt through the engine
        dict(name="vepelix_first_token_77", **c("vepelix", "1*77@0", "engine", width=1024)),
        # 32-bit products (evaluation runs): three prompts, the shortest of one token
        dict(name="vepelix_f32_prompts", **c("vepelix", "1*300@0+1*75@0+1*1@0", "forward", "f32", width=1024)),
        # ragged prompts in one step, two of them longer than the window with the first positions kept
        dict(name="pukatar_prefill_ragged", **c("pukatar", "1*1531@0+1*257@0+1*64@0+1*3@0+1*1101@0", "forward", width=2048, times=2)),
        # a small decode batch
        dict(name="pukatar_decode_7", **c("pukatar", "7*1@1500", "graph", width=1024, times=2)),
        # continuous batching: decoding sequences beside a second portion of a long prompt and a new one
        dict(name="pukatar_mixed", **c("pukatar", "27*1@900+1*229@512+1*256@0", "forward", width=2048)),
        # the draw of 64 next tokens: temperature, top-k, top-p
        dict(name="sample_64", **c("sampler", "64*1@0", "forward", "f32")),
    ]


def draw(rng):
    """Models by the share of the list that they have; batch sizes and lengths over their logarithm, odd ones among them."""
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    model = rng.choice(["moe", "moe", "dense", "vepelix", "vepelix", "vepelix", "pukatar", "pukatar", "pukatar", "sampler"])
    quantized = model in MOE
    if model == "sampler":
        return _case(model, "%d*1@0" % log(1, 64), "forward", "f32")
    arith = rng.choice(["int8", "int8", "fp8"]) if quantized else rng.choice(["bf16", "bf16", "bf16", "bf16", "f32"])
    width = 1024 if quantized or arith == "f32" else rng.choice([1024, 2048])
    times = 1 if quantized or arith == "f32" else rng.choice([1, 2])
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "mixed"])
    if kind == "decode":
        return _case(model, "%d*1@%d" % (log(1, 64), log(16, 2048)), "graph", arith, width, times)
    most = 16384 if quantized else (600 if arith == "f32" else 3500)
    if kind == "mixed":
        return _case(model, "%d*1@%d+1*%d@0" % (log(1, 40), log(16, 1500), log(17, 480)), "forward", arith, width, times)
    if rng.random() < 0.25:
        return _case(model, "1*%d@0" % log(5, 400), "engine", arith, width, times)
    parts, left = [], log(64, most)
    for _ in range(rng.choice([1, 2, 3, 5])):
        n = min(left, log(1, 2048))
        if n > 0:
            parts.append("1*%d@0" % n)
            left -= n
    return _case(model, "+".join(parts), "forward", arith, width, times)


# ---- inputs, from the seed alone ---------------------------------------------------------------------------------------------------------
def _sequences(case):
    """[(new tokens, cached tokens)] in slot order."""
    out = []
    for part in case["batch"].split("+"):
        count, rest = part.split("*")
        new, past = rest.split("@")
        out += [(int(new), int(past))] * int(count)
    return out


class _Draws:
    """Random tensors on the GPU, a generator per seed and purpose."""

    def __init__(self, seed, tag):
        self.g = torch.Generator(device=DEV).manual_seed((int(seed) * 1000003 + zlib.crc32(tag.encode())) % (1 << 62))

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.float32):
        return torch.randn(*shape, generator=self.g, device=DEV).mul_(std).add_(mean).to(dtype)

    def ints(self, n, top):
        return torch.randint(0, top, (n,), generator=self.g, device=DEV)

    def order(self, n):
        return torch.randperm(n, generator=self.g, device=DEV)


def _tokens(case, seed):
    return _Draws(seed, "tokens").ints(sum(n for n, _ in _sequences(case)), VOCAB)


def _past(seed, run, part, rows, width, std=0.7):
    """What earlier steps left in a layer run's cache or state, sequences one behind the other."""
    return _Draws(seed, "past %d %s" % (run, part)).normal(rows, width, std=std)


def _quantized_config(case):
    need = max(n + p for n, p in _sequences(case))
    return ModelConfig(max_pos=max(2304, need + 16), **MOE[case["model"]])


def _quantized_weights(case, seed):
    """N(0, 0.02) matrices, those that write the residual scaled down with a usual depth (OUT), norm weights near one; balanced routing
    tables, the routes of a token on different experts."""
    cfg, r = _quantized_config(case), _Draws(seed, "weights")
    H, kv, hd, E = cfg.hidden_size, cfg.num_kv_heads * cfg.head_dim, cfg.head_dim, cfg.num_experts
    mat = lambda *s: r.normal(*s, std=0.02)
    out = lambda *s: r.normal(*s, std=OUT)
    norm = lambda n: r.normal(n, std=0.1, mean=1.0)
    w = {"embed": r.normal(VOCAB, H, std=0.2), "final_norm": norm(H)}
    for l in range(cfg.num_layers):
        p = "l%d." % l
        w.update({p + "ln1": norm(H), p + "qkv": mat(H + 2 * kv, H), p + "q_norm": norm(hd), p + "k_norm": norm(hd), p + "o": out(H, H), p + "ln2": norm(H)})
        if E > 1:
            ei, S = cfg.intermediate_size // E, cfg.shared_intermediate_size
            first = r.order(VOCAB) % E
            w.update({p + "exp_gate_up": mat(E, 2 * ei, H), p + "exp_down": out(E, H, ei), p + "sh_gate_up": mat(2 * S, H), p + "sh_down": out(H, S),
                      p + "table": torch.stack([first, (first + 1 + r.order(VOCAB) % (E - 1)) % E])})
        else:
            w.update({p + "gate_up": mat(2 * cfg.intermediate_size, H), p + "down": out(H, cfg.intermediate_size)})
    return w


def _layers(case):
    """One block's layers: (mixer, feed-forward)."""
    if case["model"] == "vepelix":
        return [("latent", "dense"), ("parallel", "moe"), ("latent", "moe"), ("parallel", "moe")]
    return [("delta", "dense"), ("delta", "moe"), ("window", "dense"), ("delta", "moe")]


def _hybrid_weights(case, seed):
    """N(0, 0.02) matrices in bf16, those that write the residual scaled down (OUT), small vectors spread around where training leaves them,
    a router wide enough to tell tokens apart."""
    vep = case["model"] == "vepelix"
    z = (VEPELIX if vep else PUKATAR)[case["width"]]
    r, W = _Draws(seed, "weights"), case["width"]
    bf = torch.bfloat16
    mat = lambda *s: r.normal(*s, std=0.02, dtype=bf)
    out = lambda *s: r.normal(*s, std=OUT, dtype=bf)
    vec = lambda n, mean=0.0, std=0.1: r.normal(n, std=std, mean=mean, dtype=bf)
    w = {"embed": r.normal(VOCAB, W, std=2.0, dtype=bf), "head": mat(VOCAB, W)}
    if vep:
        w["final.norm"] = vec(W)
    else:
        for name in ("embed.norm", "final.norm", *("l%d.norm1" % i for i in range(4))):
            w.update({name: vec(W, 1.0), name + ".b": vec(W)})
        if case["times"] > 1:
            w.update({"loop.in": mat(W, 2 * W), "loop.step": r.normal(case["times"], W, std=0.1, dtype=bf)})

    def glu(p, ff):
        w.update({p + "gate": mat(ff, W), p + "up": mat(ff, W), p + "down": out(W, ff)})

    for i, (mixer, mlp) in enumerate(_layers(case)):
        p = "l%d." % i
        m = p + "mix."
        if vep:
            w.update({p + "norm1": vec(W), p + "norm2": vec(W), p + "ls1": vec(W, 1.0), p + "ls2": vec(W, 1.0)})
        if mixer == "latent":
            H, rank = z["heads"], z["kv_rank"]
            w.update({m + "dq": mat(z["q_rank"], W), m + "dq.norm": vec(z["q_rank"], 1.0), m + "uq": mat(H * (z["dim"] + z["rot_dim"]), z["q_rank"]),
                      m + "dkv": mat(rank + z["rot_dim"], W), m + "dkv.norm": vec(rank, 1.0), m + "uk": mat(H * z["dim"], rank), m + "uv": mat(H * z["vdim"], rank),
                      m + "sink": vec(H, std=0.5), m + "g": mat(H, W), m + "o": out(W, H * z["vdim"])})
        elif mixer == "parallel":
            H, G, d, dv = z["left_heads"], z["left_kv_heads"], z["left_dim"], z["left_vdim"]
            rk, rv = z["rec_heads"] * z["rec_dim"], z["rec_heads"] * z["rec_vdim"]
            a, b = m + "left.", m + "right."
            w.update({a + "q": mat(H * d, W), a + "k": mat(G * d, W), a + "v": mat(G * dv, W), a + "q.norm": vec(d, 1.0), a + "k.norm": vec(d, 1.0), a + "o": out(W, H * dv),
                      b + "q": mat(rk, W), b + "k": mat(rk, W), b + "v": mat(rv, W), b + "g": mat(rv, W), b + "a1": mat(RANK, W), b + "a2": mat(rk, RANK),
                      b + "a2.b": torch.linspace(-2.0, 6.0, rk, device=DEV).to(bf), b + "norm": vec(z["rec_vdim"], 1.0), b + "o": out(W, rv)})
        elif mixer == "window":
            H, G, d, dv = z["heads"], z["kv_heads"], z["dim"], z["vdim"]
            w.update({m + "q": mat(H * d, W), m + "k": mat(G * d, W), m + "v": mat(G * dv, W), m + "sink": vec(H, std=0.5), m + "o": out(W, H * dv)})
        else:
            H = z["rec_heads"]
            rk, rv, nd = z["rec_kv_heads"] * z["rec_dim"], H * z["rec_vdim"], H * z["rec_dim"]
            tap = lambda n: r.normal(n, z["taps"], std=0.3, dtype=bf)
            w.update({m + "q": mat(rk, W), m + "k": mat(rk, W), m + "v": mat(rv, W), m + "q.conv": tap(rk), m + "k.conv": tap(rk), m + "v.conv": tap(rv), m + "b": mat(H, W),
                      m + "A_log": torch.linspace(-4.0, 0.0, H, device=DEV).to(bf), m + "dt_bias": vec(nd), m + "norm": vec(z["rec_vdim"], 1.0), m + "a1": mat(RANK, W),
                      m + "a2": mat(nd, RANK), m + "g1": mat(RANK, W), m + "g2": mat(rv, RANK), m + "o": out(W, rv)})
        f = p + "mlp."
        if mlp == "dense":
            glu(f, z["ff"])
        else:
            w[f + "router"] = r.normal(z["experts"], W, std=0.1, dtype=bf)
            for e in range(z["experts"]):
                glu("%se%d." % (f, e), z["expert_ff"])
            glu(f + "shared.", z["shared_ff"])
            if not vep:
                w.update({f + "router.b": vec(z["experts"]), f + "shared.sg": mat(1, W)})
    return w


def _cached(case, run, mixer):
    """{part: width} of what a layer run keeps per cached token, and of its state per sequence."""
    z = (VEPELIX if case["model"] == "vepelix" else PUKATAR)[case["width"]]
    if mixer == "latent":
        return {"rows": z["kv_rank"] + z["rot_dim"]}, {}
    if mixer == "parallel":
        return {"rows": z["left_kv_heads"] * (z["left_vdim"] + z["left_dim"])}, {"gla": (z["rec_heads"], z["rec_vdim"], z["rec_dim"])}
    if mixer == "window":
        return {"rows": z["kv_heads"] * (z["vdim"] + z["dim"])}, {}
    conv = 2 * z["rec_kv_heads"] * z["rec_dim"] + z["rec_heads"] * z["rec_vdim"]
    return {}, {"gdn": (z["rec_heads"], z["rec_vdim"], z["rec_dim"]), "conv": (z["taps"] - 1, conv)}


def _runs(case):
    """[(layer, pass)] in the order they run."""
    return [(i, t) for t in range(case["times"]) for i in range(4)]


def _scatter(kv, seqs, pool, values):
    """Rows of the cached tokens, sequences one behind the other, into the pages that the sequences own."""
    flat, at = pool.view(-1, *pool.shape[2:]), 0
    for s, (_, past) in enumerate(seqs):
        if past:
            pos = torch.arange(past, device=DEV)
            page = kv.block_table[s].long()[pos // PAGE]
            flat[page * PAGE + pos % PAGE] = values[at:at + past].view(past, *pool.shape[2:]).to(pool.dtype)
            at += past


STATE_STD = {"gla": 0.1, "gdn": 0.1, "conv": 0.7}


def _build(case, seed, seqs):
    blocks = sum((n + p + PAGE - 1) // PAGE for n, p in seqs) + 1
    past = sum(p for _, p in seqs)
    if case["model"] in MOE:
        cfg = _quantized_config(case)
        model = I64MoEModel(cfg, _quantized_weights(case, seed), device=DEV, kv_dtype=torch.bfloat16, max_seqs=len(seqs), num_kv_blocks=blocks, quant=case["arith"])
        if case["drive"] != "engine":
            for s, (n, p) in enumerate(seqs):
                model.kv.reserve(s, n + p)
        width = cfg.num_kv_heads * cfg.head_dim
        for l in range(cfg.num_layers) if past else ():
            _scatter(model.kv, seqs, model.kv.k[l], _past(seed, l, "k", past, width, 1.0))
            _scatter(model.kv, seqs, model.kv.v[l], _past(seed, l, "v", past, width))
        return model
    vep = case["model"] == "vepelix"
    z = (VEPELIX if vep else PUKATAR)[case["width"]]
    cfg = (synth.vepelix_config if vep else synth.pukatar_config)(blocks=1, loop_blocks=int(case["times"] > 1), vocab=VOCAB, **z)
    model = (VepelixModel if vep else PukatarModel)(cfg, _hybrid_weights(case, seed), device=DEV, dtype="float32" if case["arith"] == "f32" else "bfloat16",
                                                    max_seqs=len(seqs), num_kv_blocks=blocks, kv_block=PAGE)
    if case["drive"] != "engine":
        for s, (n, p) in enumerate(seqs):
            model.kv.reserve(s, n + p)
    if past:
        carried = [s for s, (_, p) in enumerate(seqs) if p]
        for run, (i, _) in enumerate(_runs(case)):
            rows, state = _cached(case, run, _layers(case)[i][0])
            if rows:
                _scatter(model.kv, seqs, model.kv.rows[run], _past(seed, run, "rows", past, rows["rows"]))
            for name, shape in state.items():
                model.kv.state[run][name][carried] = _past(seed, run, name, len(carried), math.prod(shape), STATE_STD[name]).view(-1, *shape)
    return model


def prepare(case, seed):
    """The runner with its weights, the pages and states that earlier steps filled, and the step's token ids."""
    seqs = _sequences(case)
    if case["model"] == "sampler":
        n, r = len(seqs), _Draws(seed, "logits")
        top = r.normal(n, VOCAB, std=2.0)      # a trained model's logits: a wide body and a few tokens far above it
        top.scatter_add_(1, r.ints(n * 12, VOCAB).view(n, 12), r.normal(n, 12, std=2.0, mean=8.0))
        return dict(case=case, logits=top, temperature=torch.full((n,), 0.8, device=DEV), top_k=torch.full((n,), 50, dtype=torch.int32, device=DEV),
                    top_p=torch.full((n,), 0.95, device=DEV), u=torch.rand(n, generator=r.g, device=DEV))
    model, ids = _build(case, seed, seqs), _tokens(case, seed)
    if case["drive"] == "graph":
        dec = GreedyDecoder(model, len(seqs), use_graph=True)
        lens = [p for _, p in seqs]
        dec.set_state(ids, lens, reserve_extra=1)
        dec.prepare()
        here = [dec.tokens.clone(), dec.positions.clone(), dec.ctx_len.clone()]
        return dict(case=case, model=model, dec=dec, lens=lens, here=here)
    if case["drive"] == "engine":
        cuts, at = [], 0
        host = ids.tolist()
        for s, (n, _) in enumerate(seqs):
            cuts.append(("r%d" % s, host[at:at + n], [n - 1]))
            at += n
        return dict(case=case, model=model, engine=Engine(model, max_batch_tokens=4096), entries=cuts, ends=[c[0] for c in cuts])
    new = [n for n, _ in seqs]
    pos = torch.cat([torch.arange(p, p + n, dtype=torch.int32) for n, p in seqs]).to(DEV)
    slots = torch.cat([torch.full((n,), s, dtype=torch.int32) for s, n in enumerate(new)]).to(DEV)
    last = (torch.cumsum(torch.tensor(new), 0) - 1).to(torch.int32).to(DEV)
    return dict(case=case, model=model, args=(ids, pos, slots, (pos + 1).contiguous()),
                kw=dict(logit_rows=last, max_ctx_hint=max(n + p for n, p in seqs), tokens_per_seq=new))


def run(state):
    case = state["case"]
    if case["model"] == "sampler":
        return ops_dense.sample_rows(state["logits"], temperature=state["temperature"], top_k=state["top_k"], top_p=state["top_p"], u=state["u"])
    if case["drive"] == "graph":
        dec = state["dec"]
        # back to the position in front of the step: its token is decoded again over the same cached rows
        torch._foreach_copy_([dec.tokens, dec.positions, dec.ctx_len], state["here"])
        dec.host_lens = list(state["lens"])
        logits = dec.step()
    elif case["drive"] == "engine":
        logits = state["engine"].step(state["entries"], end=state["ends"])
    else:
        logits = state["model"].forward(*state["args"], **state["kw"])
    kv = state["model"].kv      # what the step leaves for the next one: pages of cached rows, the recurrences' states
    if case["model"] in MOE:
        return {"logits": logits, "cache": [*kv.k, *kv.v]}
    return {"logits": logits, "cache": [t for t in kv.rows if t is not None], "state": [d[name] for d in kv.state for name in sorted(d)]}


# ---- what a step cannot do without -------------------------------------------------------------------------------------------------------
def _seen(n, p, window, keep):
    """(query, key) pairs of n new rows behind p cached ones, and the cached rows that any of them sees."""
    if not window:
        return n * p + n * (n + 1) // 2, p
    pairs = sum(min(j + 1, window) + min(keep, max(0, j + 1 - window)) for j in range(p, p + n))
    return pairs, min(p, window - 1 + keep)


def work(case):
    seqs = _sequences(case)
    rows, outs = sum(n for n, _ in seqs), len(seqs)
    if case["model"] == "sampler":
        return {"bytes": outs * VOCAB * 4 + outs * 24, "flops": outs * VOCAB * 4}
    if case["model"] in MOE:
        cfg = _quantized_config(case)
        H, kv, E = cfg.hidden_size, cfg.num_kv_heads * cfg.head_dim, cfg.num_experts
        fixed = H * (H + 2 * kv) + H * H
        if E > 1:
            one = 3 * H * (cfg.intermediate_size // E)
            read, mult = fixed + 3 * H * cfg.shared_intermediate_size + one * min(E, rows * cfg.top_k), fixed + 3 * H * cfg.shared_intermediate_size + one * cfg.top_k
        else:
            read = mult = fixed + 3 * H * cfg.intermediate_size
        pairs = sum(_seen(n, p, 0, 0)[0] for n, p in seqs)
        cached = sum(n + p for n, p in seqs) * 2 * kv * 2
        return {"bytes": cfg.num_layers * (read + cached) + VOCAB * H * 4 + min(rows, VOCAB) * H * 4 + rows * 8 + outs * VOCAB * 4,
                "flops": cfg.num_layers * (2 * rows * mult + 4 * pairs * H) + 2 * outs * VOCAB * H}
    vep = case["model"] == "vepelix"
    z, W = (VEPELIX if vep else PUKATAR)[case["width"]], case["width"]
    row_bytes = 4 if case["arith"] == "f32" else 2
    nbytes, flops = VOCAB * W * 2 + min(rows, VOCAB) * W * 2 + rows * 8 + outs * VOCAB * 4, 2 * outs * VOCAB * W
    for run, (i, t) in enumerate(_runs(case)):
        mixer, mlp = _layers(case)[i]
        pairs, cached = 0, 0
        window, keep = (0, 0) if mixer == "latent" else (z["window"], z.get("keep_first", 0))
        for n, p in seqs:
            a, b = _seen(n, p, window, keep)
            pairs, cached = pairs + a, cached + n + b
        if mixer == "latent":
            H = z["heads"]
            qw = H * (z["dim"] + z["rot_dim"])
            par = W * (z["q_rank"] + z["kv_rank"] + z["rot_dim"] + H) + z["q_rank"] * qw + z["kv_rank"] * H * (z["dim"] + z["vdim"]) + W * H * z["vdim"]
            flops += 2 * pairs * H * (z["dim"] + z["rot_dim"] + z["vdim"])
        elif mixer == "window" or mixer == "parallel":
            s = "left_" if mixer == "parallel" else ""
            H, G, d, dv = z[s + "heads"], z[s + "kv_heads"], z[s + "dim"], z[s + "vdim"]
            par = W * (H * d + G * (d + dv) + H * dv)
            flops += 2 * pairs * H * (d + dv)
        else:
            par = 0
        rows_kept, state = _cached(case, run, mixer)
        nbytes += cached * rows_kept.get("rows", 0) * row_bytes
        if state:
            H, d, dv = z["rec_heads"], z["rec_dim"], z["rec_vdim"]
            G = z.get("rec_kv_heads", H)
            par += W * (2 * G * d + H * dv + RANK) + RANK * H * d + W * H * dv + (W * H * dv if mixer == "parallel" else W * (RANK + H) + RANK * H * dv)
            flops += rows * H * d * dv * (5 if mixer == "parallel" else 8)
            nbytes += sum(math.prod(s) * 4 * (1 + (p > 0)) for s in state.values() for _, p in seqs)
        read = par
        if mlp == "dense":
            par, read = par + 3 * W * z["ff"], read + 3 * W * z["ff"]
        else:
            par += 3 * W * (z["shared_ff"] + z["top"] * z["expert_ff"]) + W * z["experts"]
            read += 3 * W * (z["shared_ff"] + min(z["experts"], rows * z["top"]) * z["expert_ff"]) + W * z["experts"]
        if not vep and case["times"] > 1 and i == 0:
            par, read = par + W * W, read + W * W
        flops += 2 * rows * par
        nbytes += 2 * read if t == 0 else 0      # (a further pass has the same weights)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the distance from the same step in 64 bits: int8 and fp8 0.004 to 0.019 (codes on a rounding tie), bf16 0.002 to 0.0045 with
    single values up to 0.12, 32 bits 1.2e-6 with single values up to 2e-5."""
    if case["model"] == "sampler":
        return {"rel": 0.0, "differ": 0.01}      # a draw that falls on the border of two tokens
    return {"int8": {"rel": 0.03, "max": 0.5}, "fp8": {"rel": 0.03, "max": 0.5}, "bf16": {"rel": 0.02, "max": 0.5}, "f32": {"rel": 5e-6, "max": 1e-4}}[case["arith"]]


# ---- the same steps in 64 bits -----------------------------------------------------------------------------------------------------------
def _rms(x, eps=EPS):
    return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _attend(q, k, v, scale, p, window=0, keep=0, sink=None):
    """q [n, H, d] at positions p .. against k [p + n, G, d], v [p + n, G, dv]; sink [H]: one more term in the denominator."""
    n, H, G = q.shape[0], q.shape[1], k.shape[1]
    k, v = k.repeat_interleave(H // G, 1), v.repeat_interleave(H // G, 1)
    s = torch.matmul(q.transpose(0, 1), k.permute(1, 2, 0).contiguous()) * scale      # [H, n, p + n]
    i, j = torch.arange(p, p + n, device=DEV)[:, None], torch.arange(p + n, device=DEV)[None, :]
    see = j <= i
    if window:
        see = see & ((i - j < window) | (j < keep))
    s = s.masked_fill(~see, -math.inf)
    if sink is not None:
        s = torch.cat([s, sink.view(H, 1, 1).expand(H, n, 1)], -1)
    a = torch.softmax(s, -1)[..., :p + n]
    return torch.matmul(a, v.transpose(0, 1).contiguous()).transpose(0, 1)      # [n, H, dv]


def _exact_quantized(case, seed):
    cfg, w, seqs = _quantized_config(case), _quantized_weights(case, seed), _sequences(case)
    ids, total = _tokens(case, seed), sum(p for _, p in seqs)
    pos = torch.cat([torch.arange(p, p + n, device=DEV) for n, p in seqs])
    H, hd, nh, G, E = cfg.hidden_size, cfg.head_dim, cfg.num_heads, cfg.num_kv_heads, cfg.num_experts

    def linear8(x, wt):
        """The whole call has one scale and zero point of seven bits, the matrix one scale."""
        ws = wt.abs().max() / 127.5
        wq = torch.clamp(torch.round(wt / ws), -128, 127)
        lo, hi = x.min().clamp(max=0.0), x.max().clamp(min=0.0)
        s = (hi - lo) / 127.0
        a, b = lo.abs() / s, 127.0 - hi / s
        zp = torch.round(torch.where(-a < 127.0 - (hi / s).abs(), a, b)).clamp(0, 127)
        return ((torch.round(x / s + zp).clamp(0, 255) - zp) @ wq.T) * (s * ws)

    def linear_fp8(x, wt):
        def codes(t):
            s = t.abs().amax(-1, keepdim=True).clamp(min=1e-12) / 448.0
            return (t / s).clamp(-448.0, 448.0).float().to(torch.float8_e4m3fn).double(), s
        (xq, xs), (wq, ws) = codes(x), codes(wt)
        return (xq @ wq.T) * xs * ws.T

    linear = linear8 if case["arith"] == "int8" else linear_fp8
    M = lambda name: w[name].double()

    def glu(x, gate_up, down):
        g, u = linear(x, gate_up).chunk(2, -1)
        return linear(_silu(g) * u, down)

    def rotate(x):
        f = cfg.rope_theta ** (-torch.arange(0, hd, 2, dtype=F64, device=DEV) / hd)
        a = (pos.double()[:, None] * f)[:, None, :]
        u, v = x.chunk(2, -1)
        return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()], -1)

    x = M("embed")[ids]
    for l in range(cfg.num_layers):
        p_ = "l%d." % l
        q, k, v = linear(_rms(x) * M(p_ + "ln1"), M(p_ + "qkv")).split((H, G * hd, G * hd), -1)
        q = rotate(_rms(q.view(-1, nh, hd)) * M(p_ + "q_norm"))
        k = rotate(_rms(k.view(-1, G, hd)) * M(p_ + "k_norm"))
        v = v.view(-1, G, hd)
        pk = _past(seed, l, "k", total, G * hd, 1.0).bfloat16().double().view(-1, G, hd)
        pv = _past(seed, l, "v", total, G * hd).bfloat16().double().view(-1, G, hd)
        out, at, old = [], 0, 0
        for n, p in seqs:
            kk, vv = torch.cat([pk[old:old + p], k[at:at + n]]), torch.cat([pv[old:old + p], v[at:at + n]])
            out.append(_attend(q[at:at + n], kk, vv, hd ** -0.5, p))
            at, old = at + n, old + p
        x = x + linear(torch.cat(out).reshape(-1, H), M(p_ + "o"))
        h = _rms(x) * M(p_ + "ln2")
        if E > 1:
            route = w[p_ + "table"][:, ids]
            gu, dn = M(p_ + "exp_gate_up"), M(p_ + "exp_down")
            y = glu(h, M(p_ + "sh_gate_up"), M(p_ + "sh_down")) * cfg.shared_scale
            for r in range(cfg.top_k):
                for e in range(E):
                    mine = (route[r] == e).nonzero().flatten()
                    if mine.numel():
                        y[mine] += cfg.routed_scale * cfg.primary_weight * glu(h[mine], gu[e], dn[e])      # (two routes of one half each)
        else:
            y = glu(h, M(p_ + "gate_up"), M(p_ + "down"))
        x = x + y
    last = torch.cumsum(torch.tensor([n for n, _ in seqs], device=DEV), 0) - 1
    return {"logits": (_rms(x[last]) * M("final_norm")) @ M("embed").T, "cache": None}      # (which page holds what is the runner's business)


def _scaled_frequencies(dims):
    """Pairs that turn often within 1024 positions keep their frequency, slow ones run four times slower, a ramp between them."""
    base, factor, original, fast, slow = 100000.0, 4.0, 1024.0, 32.0, 1.0
    index = lambda turns: dims * math.log(original / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
    lo, hi = max(math.floor(index(fast)), 0), min(math.ceil(index(slow)), dims - 1)
    i = torch.arange(dims // 2, dtype=F64, device=DEV)
    plain, ramp = base ** (-2.0 * i / dims), ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    return ramp * plain / factor + (1.0 - ramp) * plain, 1.0 + 0.1 * math.log(factor)


def _exact_hybrid(case, seed):
    vep = case["model"] == "vepelix"
    z, W, seqs = (VEPELIX if vep else PUKATAR)[case["width"]], case["width"], _sequences(case)
    w, ids, total = _hybrid_weights(case, seed), _tokens(case, seed), sum(p for _, p in seqs)
    pos = torch.cat([torch.arange(p, p + n, device=DEV) for n, p in seqs])
    rounded = (lambda t: t.double()) if case["arith"] == "f32" else (lambda t: t.bfloat16().double())
    M = lambda name: w[name].double()
    N = ids.numel()
    starts = [0]
    for n, _ in seqs:
        starts.append(starts[-1] + n)

    def pairs(x):      # neighbours turn against each other
        f, mult = _scaled_frequencies(x.shape[-1])
        a = (pos.double()[:, None] * f)[:, None, :]
        c, s, u, v = a.cos() * mult, a.sin() * mult, x[..., 0::2], x[..., 1::2]
        return torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)

    def halves(x):
        d = x.shape[-1]
        a = (pos.double()[:, None] * 10000.0 ** (-2.0 * torch.arange(d // 2, dtype=F64, device=DEV) / d))[:, None, :]
        u, v = x.chunk(2, -1)
        return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()], -1)

    def per_sequence(run, width, f):
        """f(rows of a sequence, its cached rows, their number), results one behind the other."""
        past, old, out = rounded(_past(seed, run, "rows", total, width)), 0, []
        for s, (n, p) in enumerate(seqs):
            out.append(f(slice(starts[s], starts[s + 1]), past[old:old + p], p))
            old += p
        return torch.cat(out)

    def values_keys(run, q, k, v, **kw):
        G, dv, d = v.shape[1], v.shape[2], k.shape[2]

        def one(rows, past, p):
            past = past.view(p, G, dv + d)
            return _attend(q[rows], torch.cat([past[..., dv:], k[rows]]), torch.cat([past[..., :dv], v[rows]]), d ** -0.5, p, **kw)
        return per_sequence(run, G * (dv + d), one).flatten(1)

    def latent(run, m, h):
        H, d, dr, dv, r = z["heads"], z["dim"], z["rot_dim"], z["vdim"], z["kv_rank"]
        q = ((_rms(h @ M(m + "dq").T) * M(m + "dq.norm")) @ M(m + "uq").T).view(-1, H, d + dr)
        q = torch.cat([q[..., :d], pairs(q[..., d:])], -1)
        down = h @ M(m + "dkv").T
        c, kr = _rms(down[:, :r]) * M(m + "dkv.norm"), pairs(down[:, None, r:])[:, 0]
        uk, uv = M(m + "uk"), M(m + "uv")

        def one(rows, past, p):
            cc, kk = torch.cat([past[:, :r], c[rows]]), torch.cat([past[:, r:], kr[rows]])
            keys = torch.cat([(cc @ uk.T).view(-1, H, d), kk[:, None].expand(-1, H, dr)], -1)
            return _attend(q[rows], keys, (cc @ uv.T).view(-1, H, dv), (d + dr) ** -0.5, p, sink=M(m + "sink"))
        o = per_sequence(run, r + dr, one) * torch.sigmoid(h @ M(m + "g").T).unsqueeze(-1)
        return o.flatten(1) @ M(m + "o").T

    def recur(run, name, shape, q, k, v, decay, beta=None):
        """q, k, decay [N, H, d], v [N, H, dv]; sequences of one length together.  Returns the rows read and the states left."""
        H, dv, d = shape
        state = torch.zeros(len(seqs), H, d, dv, dtype=F64, device=DEV)
        carried = [s for s, (_, p) in enumerate(seqs) if p]
        if carried:
            state[carried] = _past(seed, run, name, len(carried), math.prod(shape), STATE_STD[name]).double().view(-1, H, dv, d).transpose(2, 3)
        out = torch.zeros(N, H, dv, dtype=F64, device=DEV)
        for n in {n for n, _ in seqs}:
            who = [s for s, (m, _) in enumerate(seqs) if m == n]
            first, S = torch.tensor([starts[s] for s in who], device=DEV), state[who]
            for t in range(n):
                at = first + t
                S = S * decay[at].unsqueeze(-1)
                u = v[at]
                if beta is not None:
                    u = beta[at].unsqueeze(-1) * (u - (S * k[at].unsqueeze(-1)).sum(-2))
                S = S + k[at].unsqueeze(-1) * u.unsqueeze(-2)
                out[at] = (S * q[at].unsqueeze(-1)).sum(-2)
            state[who] = S
        return out, state.transpose(2, 3)

    def linear_attention(run, m, h, states):
        H, d, dv = z["rec_heads"], z["rec_dim"], z["rec_vdim"]
        q, k, v = (h @ M(m + "q").T).view(N, H, d) * d ** -0.5, (h @ M(m + "k").T).view(N, H, d), (h @ M(m + "v").T).view(N, H, dv)
        decay = torch.sigmoid((h @ M(m + "a1").T) @ M(m + "a2").T + M(m + "a2.b")) ** (1.0 / 8.0)
        o, s = recur(run, "gla", (H, dv, d), q, k, v, decay.view(N, H, d))
        states.append(s)
        return ((_rms(o) * M(m + "norm")).flatten(1) * _silu(h @ M(m + "g").T)) @ M(m + "o").T

    def convolve(run, m, h, states):
        """Silu of the causal convolution over [q | k | v], and the inputs that the next step needs."""
        x = torch.cat([h @ M(m + n).T for n in "qkv"], -1)
        taps = torch.cat([M(m + n + ".conv") for n in "qkv"])
        T, C = taps.shape[1], taps.shape[0]
        held = torch.zeros(len(seqs), T - 1, C, dtype=F64, device=DEV)
        carried = [s for s, (_, p) in enumerate(seqs) if p]
        if carried:
            held[carried] = _past(seed, run, "conv", len(carried), (T - 1) * C, STATE_STD["conv"]).double().view(-1, T - 1, C)
        out, kept = [], []
        for s in range(len(seqs)):
            y = torch.cat([held[s], x[starts[s]:starts[s + 1]]])
            n = y.shape[0] - (T - 1)
            out.append(sum(y[j:j + n] * taps[:, j] for j in range(T)))
            kept.append(y[-(T - 1):])
        states.append(torch.stack(kept))
        return _silu(torch.cat(out))

    def delta(run, m, h, states):
        H, G, d, dv = z["rec_heads"], z["rec_kv_heads"], z["rec_dim"], z["rec_vdim"]
        q, k, v = convolve(run, m, h, states).split((G * d, G * d, H * dv), -1)
        unit = lambda t: (t / torch.sqrt(t.pow(2).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 1)
        q, k = unit(q.reshape(N, G, d)) * d ** -0.5, unit(k.reshape(N, G, d))
        step = torch.nn.functional.softplus((h @ M(m + "a1").T) @ M(m + "a2").T + M(m + "dt_bias"), threshold=700.0).view(N, H, d)
        o, s = recur(run, "gdn", (H, dv, d), q, k, v.reshape(N, H, dv), torch.exp(-torch.exp(M(m + "A_log")).view(1, H, 1) * step), torch.sigmoid(h @ M(m + "b").T))
        states.append(s)
        o = (_rms(o) * M(m + "norm")).flatten(1) * torch.sigmoid((h @ M(m + "g1").T) @ M(m + "g2").T)
        return o @ M(m + "o").T

    def clamped(p, h):
        g, u = (h @ M(p + "gate").T).clamp(max=7.0), (h @ M(p + "up").T).clamp(-7.0, 7.0)
        return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ M(p + "down").T

    def plain(p, h):
        return (_silu(h @ M(p + "gate").T) * (h @ M(p + "up").T)) @ M(p + "down").T

    def mixture(p, h):
        zr = h @ M(p + "router").T
        if not vep:
            zr = zr + M(p + "router.b")
        best, who = zr.topk(z["top"], -1)
        weight = torch.sigmoid(best) if vep else torch.softmax(best, -1)
        y = plain(p + "shared.", h) if vep else torch.sigmoid(h @ M(p + "shared.sg").T) * clamped(p + "shared.", h)
        for e in range(z["experts"]):
            row, at = (who == e).nonzero(as_tuple=True)
            if row.numel():
                g = weight[row, at].unsqueeze(-1)
                q = "%se%d." % (p, e)
                y[row] += plain(q, g * h[row]) if vep else g * clamped(q, h[row])
        return y

    def norm(name, x):
        if vep:
            return _rms(x) * (1.0 + M(name))
        return _rms(x - x.mean(-1, keepdim=True)) * M(name) + M(name + ".b")

    x = M("embed")[ids]
    if not vep:
        x = norm("embed.norm", x)
    x0, states = x, []
    for run, (i, t) in enumerate(_runs(case)):
        mixer, mlp = _layers(case)[i]
        p = "l%d." % i
        m = p + "mix."
        if vep and t and i == 0:
            x = x + x0
        elif not vep and case["times"] > 1 and i == 0:
            x = torch.cat([x, x0], -1) @ M("loop.in").T + M("loop.step")[t]
        h = norm(p + "norm1", x)
        if mixer == "latent":
            y = latent(run, m, h)
        elif mixer == "delta":
            y = delta(run, m, h, states)
        elif mixer == "window":
            H, G, d, dv = z["heads"], z["kv_heads"], z["dim"], z["vdim"]
            q, k = halves((h @ M(m + "q").T).view(N, H, d)), halves((h @ M(m + "k").T).view(N, G, d))
            y = values_keys(run, q, k, (h @ M(m + "v").T).view(N, G, dv), window=z["window"], keep=z["keep_first"], sink=M(m + "sink")) @ M(m + "o").T
        else:
            H, G, d, dv, a = z["left_heads"], z["left_kv_heads"], z["left_dim"], z["left_vdim"], m + "left."
            q, k = ((_rms((h @ M(a + n).T).view(N, c, d)) * M(a + n + ".norm")) for n, c in (("q", H), ("k", G)))
            left = values_keys(run, pairs(q), pairs(k), (h @ M(a + "v").T).view(N, G, dv), window=z["window"]) @ M(a + "o").T
            y = 0.7 * left + 0.6 * linear_attention(run, m + "right.", h, states)
        f = p + "mlp."
        if vep:
            x = x + M(p + "ls1") * y
            h = norm(p + "norm2", x)
            x = x + M(p + "ls2") * (clamped(f, h) if mlp == "dense" else mixture(f, h))
        else:
            x = x + (y + (plain(f, h) if mlp == "dense" else mixture(f, h)))
    last = torch.tensor(starts[1:], device=DEV) - 1
    return {"logits": norm("final.norm", x[last]) @ M("head").T, "cache": None, "state": states}


@torch.no_grad()
def exact(case, seed):
    if case["model"] == "sampler":
        return None
    return _exact_quantized(case, seed) if case["model"] in MOE else _exact_hybrid(case, seed)
