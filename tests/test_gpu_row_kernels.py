"""Row kernels that give a row more waves in launches of few rows: both forms at the edges of the rule, widths and alignments that take whole
vectors and those that do not, against 64-bit references."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


def close(got, ref, tol=2e-5):
    # sums of at most a few thousand fp32 terms of order one: 2^-24 each, far below tol
    assert torch.allclose(got.double().cpu(), ref, atol=tol, rtol=tol), float((got.double().cpu() - ref).abs().max())


@pytest.mark.parametrize("n", [1, 256, 257])
@pytest.mark.parametrize("width,groups,period,off", [(2048, 16, 2048, 0), (1028, 1, 1028, 4), (96, 16, 96, 0), (2056, 4, 257, 0), (260, 5, 52, 3)])
@pytest.mark.parametrize("after", [False, True])
def test_gate_norm(dev, n, width, groups, period, off, after):
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(width + n)
    y, z, w = torch.randn(n, width, generator=g), torch.randn(n, width + off + 5 * (off == 3), generator=g), torch.rand(period, generator=g)
    out = torch.empty(n, width, device=dev)
    D.gate_norm(y.to(dev), w.to(dev), out, groups=groups, eps=1e-6, z=z.to(dev), z_off=off, ldz=z.shape[1], gate_after=after, width=width)
    gate = torch.nn.functional.silu(z[:, off:off + width].double())
    v = (y.double() if after else y.double() * gate).view(n, groups, -1)
    v = (v / (v.square().mean(-1, keepdim=True) + 1e-6).sqrt()).view(n, width) * w.double().repeat(width // period)
    close(out, v * gate if after else v)


@pytest.mark.parametrize("width", [2048, 1028, 10])
@pytest.mark.parametrize("top", [1, 3, 4, 9])
@pytest.mark.parametrize("weighted,shared", [(True, True), (False, False)])
def test_moe_combine(dev, width, top, weighted, shared):
    from vllm_i64_amd import ops_dense as D
    g, n = torch.Generator().manual_seed(width + top), 5
    y, h, s = torch.randn(n * top, width, generator=g), torch.randn(n, width, generator=g), torch.randn(n, width, generator=g)
    rows = torch.randperm(n * top, generator=g).to(torch.int32).view(n, top)
    rows[2, top - 1] = -1      # a choice without a row: the input itself
    w, gate = torch.rand(n, top, generator=g), torch.rand(n, generator=g)
    out = torch.empty(n, width, device=dev)
    D.moe_combine(y.to(dev), rows.to(dev), w.to(dev) if weighted else None, h.to(dev), s.to(dev) if shared else None, out, n=n, top=top, width=width,
                  shared_gate=gate.to(dev) if shared else None)
    v = torch.where((rows >= 0)[..., None], y[rows.clamp(min=0).long()], h[:, None]).double()
    ref = (v * w.double()[..., None]).sum(1) if weighted else v.sum(1)
    close(out, ref + gate.double()[:, None] * s.double() if shared else ref)


@pytest.mark.parametrize("n", [1, 256, 257, 512, 513, 1024, 1025])
@pytest.mark.parametrize("E,K", [(5, 100), (32, 1028), (33, 130), (64, 2048)])
@pytest.mark.parametrize("gated", [False, True])
def test_route_topk(dev, n, E, K, gated):
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(E + n)
    # logits of order one: with a spread above 87 the smallest of a softmax's fp32 scores are all zero and tie
    h, w = torch.randn(n, K, generator=g), (torch.randn(E + gated, K, generator=g) * K ** -0.5).bfloat16()
    idx, wgt, gate = torch.empty(n, 4, dtype=torch.int32, device=dev), torch.empty(n, 4, device=dev), torch.empty(n, device=dev) if gated else None
    D.route_topk(None, entries=E, correction=None, groups=1, keep=1, top=4, scale=2.0, idx=idx, wgt=wgt, h=h.to(dev), w=w.to(dev), gate_out=gate)
    z = h.double() @ w.double().t()
    p = torch.softmax(z[:, :E], -1)
    best, order = p.sort(-1, descending=True)
    # fp32 products: a logit of order one is off by at most about K * 2^-24 = 1.2e-4, so entries as near as that may trade places
    assert bool((torch.gather(p, 1, idx.long().cpu()) >= best[:, :4] * (1 - 1e-3)).all())
    chosen = torch.gather(p, 1, idx.long().cpu())
    close(wgt, 2 * chosen / chosen.sum(-1, keepdim=True), 2e-3)
    if gated:
        close(gate, torch.sigmoid(z[:, E]), 1e-3)


@pytest.mark.parametrize("H,G,dim,vdim,rot,turned,heads", [(32, 8, 64, 64, 32, True, False), (3, 1, 40, 24, 40, False, True), (16, 4, 64, 64, 64, False, False)])
def test_rot_prep_forms(dev, H, G, dim, vdim, rot, turned, heads):
    """257 rows in one launch, and in launches of 256 and 1: the same rows, up to the order of a row's sum of squares."""
    from vllm_i64_amd import ops_dense as D
    g, n = torch.Generator().manual_seed(H), 257
    P = torch.randn(n, (H + G) * dim + G * vdim, generator=g).to(dev)
    pos, sl, bt = torch.arange(n, dtype=torch.int32, device=dev) % 32, torch.arange(n, dtype=torch.int32, device=dev), torch.arange(2 * n, dtype=torch.int32, device=dev).view(n, 2)
    w1, w2 = torch.rand(dim if heads else H * dim, device=dev), torch.rand(dim if heads else G * dim, device=dev)
    fr, vfr = torch.rand(rot // 2, device=dev), torch.rand(vdim // 2, device=dev) if turned else None
    def run(cuts):
        cache, q = torch.zeros(2 * n, 16, G * (vdim + dim), device=dev), torch.empty(n, H * (vdim + dim), device=dev)
        for a, b in cuts:
            D.rot_prep(P[a:b], q_off=0, k_off=H * dim, v_off=(H + G) * dim, heads=H, kv_heads=G, dim=dim, vdim=vdim, q_norm_w=w1, k_norm_w=w2, eps=1e-6, rot_dims=rot, interleaved=False,
                       inv_freq=fr, rot_mult=1.0, head_norm=not heads, v_freq=vfr, scale=0.1, positions=pos[a:b], slot_ids=sl[a:b], block_table=bt, cache=cache, q=q[a:b], n=b - a, norm_heads=heads)
        return cache, q
    one, two = run([(0, n)]), run([(0, 256), (256, n)])
    for a, b in zip(one, two):
        close(a, b.double().cpu(), 2e-6)


@pytest.mark.parametrize("H,G,dim,vdim,rot,inter", [(3, 1, 64, 16, 64, True), (16, 4, 64, 64, 32, False), (33, 3, 128, 32, 8, False), (2, 2, 16, 256, 12, True), (1, 1, 256, 64, 0, False), (70, 10, 64, 64, 64, False)])
@pytest.mark.parametrize("norm", ["", "heads", "behind"])
@pytest.mark.parametrize("n,dtype", [(1, torch.bfloat16), (37, torch.float32)])
def test_rot_prep_of_whole_heads(dev, H, G, dim, vdim, rot, inter, norm, n, dtype):
    """Heads whose sizes are powers of two: against the same in 64 bits, and against rows at an offset that only four-byte loads can read."""
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(H * dim + rot)
    W = (H + G) * dim + G * vdim
    P, pos = torch.randn(n, W, generator=g), torch.randint(0, 32, (n,), generator=g, dtype=torch.int32)
    sl, bt = torch.arange(n, dtype=torch.int32), torch.randperm(2 * n, generator=g).to(torch.int32).view(n, 2)
    w1, w2, fr, mult = torch.rand(dim, generator=g), torch.rand(dim, generator=g), torch.rand(max(rot // 2, 1), generator=g), 1.1
    def run(shift):
        buf = torch.zeros(n, W + 4, device=dev)
        buf[:, shift:shift + W] = P.to(dev)
        cache, q = torch.zeros(2 * n, 16, G * (vdim + dim), device=dev, dtype=dtype), torch.empty(n, H * (vdim + dim), device=dev)
        D.rot_prep(buf, q_off=shift, k_off=shift + H * dim, v_off=shift + (H + G) * dim, heads=H, kv_heads=G, dim=dim, vdim=vdim, q_norm_w=w1.to(dev) if norm == "heads" else None,
                   k_norm_w=w2.to(dev) if norm == "heads" else None, eps=1e-6, rot_dims=rot, interleaved=inter, inv_freq=fr.to(dev), rot_mult=mult, head_norm=norm == "behind", v_freq=None,
                   scale=0.25, positions=pos.to(dev), slot_ids=sl.to(dev), block_table=bt.to(dev), cache=cache, q=q, n=n, norm_heads=norm == "heads")
        return q.view(n, H, vdim + dim), cache[bt.to(dev).long()[torch.arange(n), pos.long() // 16], pos.long() % 16].view(n, G, vdim + dim)
    def turned(x, w):
        if norm == "heads":
            x = x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()
        if rot:
            a = (pos.float()[:, None] * fr).double()[:, None, :]      # (the kernel's angle is a 32-bit product)
            c, s, r = a.cos() * mult, a.sin() * mult, x[..., :rot]
            u, v = (r[..., 0::2], r[..., 1::2]) if inter else r.chunk(2, -1)
            p1, p2 = u * c - v * s, v * c + u * s
            x = torch.cat([torch.stack([p1, p2], -1).flatten(-2) if inter else torch.cat([p1, p2], -1), x[..., rot:]], -1)
        if norm == "behind":
            x = x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6)
        return x
    x = P.double()
    q, k, v = x[:, :H * dim].view(n, H, dim), x[:, H * dim:(H + G) * dim].view(n, G, dim), x[:, (H + G) * dim:].view(n, G, vdim)
    want = [torch.cat([torch.zeros(n, H, vdim).double(), 0.25 * turned(q, w1)], -1), torch.cat([v, turned(k, w2)], -1)]
    tol = 1e-5      # values of order one through about ten 32-bit operations, sines and cosines of angles to 32
    for a, b, c, t in zip(run(0), run(1), want, (tol, tol if dtype == torch.float32 else 2.0 ** -8)):
        assert torch.allclose(a.double().cpu(), c, atol=t * (4 if t > tol else 1), rtol=t), float((a.double().cpu() - c).abs().max())
        assert torch.allclose(a.float(), b.float(), atol=t * (4 if t > tol else 1), rtol=t)
