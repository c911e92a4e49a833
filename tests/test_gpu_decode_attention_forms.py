"""Decode rows over bf16 caches on the matrix cores: the instances for rows of exactly their size (a latent row of 256 + 32, values and keys of 64 and
of 128) and the general one beside them, against attention in 64 bits on the same cached rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def oracle(q, rows, r, koff, scale, seen, sink):
    """q [H, D], rows [T, D] (columns < r are the values, from koff on the keys), seen [T] bool, sink [H] or None; 64 bits."""
    s = (q[:, koff:].double() @ rows[:, koff:].double().T) * scale
    s = s.masked_fill(~seen, float("-inf"))
    if sink is not None:
        s = torch.cat([s, sink.double().view(-1, 1)], 1)
    return torch.softmax(s, -1)[:, :rows.shape[0]] @ rows[:, :r].double()


# the query travels as two bf16 terms (2^-17 of it), as do the weights: scores of at most 10 are off by 8e-5, and so are the weights
TOL = 2e-4


@pytest.mark.parametrize("form,r,rot", [("latent", 256, 32), ("latent", 256, 40), ("latent", 240, 48), ("kattn", 64, 64), ("kattn", 128, 128), ("kattn", 64, 48)])
@pytest.mark.parametrize("heads", [1, 5, 16, 34])
@pytest.mark.parametrize("window,keep", [(0, 0), (40, 3)])
@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("bad", [False, True])
def test_decode_rows(form, r, rot, heads, window, keep, splits, bad):
    """r, rot: a latent row's two parts, or the width of a head's values and of its keys; heads per key head; contexts that end at the edges of the
    tiles of 32 keys; a key outside the window may hold no finite number in pages that the row's tiles do not touch."""
    from vllm_i64_amd import ops_dense as D
    dev, block, G, lens = torch.device("cuda:0"), 16, 2 if form == "kattn" else 1, [1, 31, 32, 33, 64, 97, 200]
    if form == "latent" and keep:
        keep = 0
    g = torch.Generator().manual_seed(r + heads)
    n, H, width, scale = len(lens), heads * G, r + rot, 0.1
    per = (max(lens) + block - 1) // block
    bt = torch.randperm(n * per, generator=g).int().view(n, per)
    cache = torch.randn(n * per, block, G * width, generator=g).to(torch.bfloat16)
    if bad:      # behind every context, and (windows) in the first page's middle
        for s, T in enumerate(lens):
            flat = bt[s].long().repeat_interleave(block) * block + torch.arange(block).repeat(per)
            cache.view(n * per * block, -1)[flat[T:]] = float("nan")
            if window and T - window > 64:
                cache.view(n * per * block, -1)[flat[32:T - window - 33]] = float("inf")
    Q = torch.randn(n, H, width, generator=g)
    koff = 0 if form == "latent" else r
    if koff:
        Q[:, :, :koff] = 0.0
    sink = torch.linspace(-2.0, 2.0, H)
    pos = torch.tensor([T - 1 for T in lens], dtype=torch.int32, device=dev)
    slots = torch.arange(n, dtype=torch.int32, device=dev)
    out = torch.full((n, H * r), 7.0, device=dev)
    kw = dict(window=window, heads=H, out=out, n=n, mode=2, splits=splits)
    if form == "latent":
        ws = torch.empty(max(1, D.latent_attn_workspace_floats(n, H, r, splits)), device=dev)
        D.latent_attn(Q.to(dev), cache.to(dev), bt.to(dev), slots, pos, scale=scale, kv_rank=r, rot_dim=rot, sink=sink.to(dev), workspace=ws, **kw)
    else:
        ws = torch.empty(max(1, D.kattn_workspace_floats(n, H, G, r, splits)), device=dev)
        D.kattn((Q * scale).view(n, H * width).to(dev), cache.to(dev), None, bt.to(dev), slots, pos, chunk=0, bias=None, sink=True, sink_w=sink.to(dev), kv_heads=G, dim=rot, vdim=r,
                keep_first=keep, workspace=ws, **kw)
    got = out.cpu().double().view(n, H, r)
    for s, T in enumerate(lens):
        j = torch.arange(T)
        seen = (j > T - 1 - window) | (j < keep) if window else j >= 0
        rows = cache.view(n * per * block, G, width)[(bt[s].long()[j // block] * block + j % block)]
        rows = torch.where(seen.view(-1, 1, 1), rows, torch.zeros((), dtype=rows.dtype))
        for h in range(H):
            want = oracle(Q[s, h:h + 1], rows[:, h // heads], r, koff, scale, seen, sink[h:h + 1])
            assert float((got[s, h] - want[0]).abs().max() / want.abs().max()) < TOL, (T, h)


@pytest.mark.parametrize("cap", [0.0, 2.5])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("r,rot", [(64, 64), (32, 24), (128, 128), (48, 80)])
def test_options_of_the_scores(r, rot, cap, bias, scaled):
    """Key scales, soft cap and distance bias, in that order, alone and together; contexts that end at the edges of the tiles of 32 keys."""
    from vllm_i64_amd import ops_dense as D
    dev, block, G, H, lens = torch.device("cuda:0"), 16, 2, 10, [1, 31, 32, 33, 64, 97, 200]
    g = torch.Generator().manual_seed(r + rot)
    n, width, per = len(lens), r + rot, (max(lens) + block - 1) // block
    bt = torch.randperm(n * per, generator=g).int().view(n, per)
    cache = torch.randn(n * per, block, G * width, generator=g).to(torch.bfloat16)
    ks = torch.rand(n * per, block, generator=g) + 0.5
    table = torch.randn(70, H, generator=g)      # (distances beyond take its last row)
    Q = torch.randn(n, H, width, generator=g) * 0.1
    Q[:, :, :r] = 0.0
    pos, slots, out = torch.tensor([T - 1 for T in lens], dtype=torch.int32, device=dev), torch.arange(n, dtype=torch.int32, device=dev), torch.full((n, H * r), 7.0, device=dev)
    ws = torch.empty(D.kattn_workspace_floats(n, H, G, r, 3), device=dev)
    D.kattn(Q.view(n, -1).to(dev), cache.to(dev), ks.to(dev) if scaled else None, bt.to(dev), slots, pos, chunk=0, bias=table.to(dev) if bias else None, sink=False, heads=H, kv_heads=G,
            dim=rot, vdim=r, out=out, n=n, mode=2, splits=3, workspace=ws, softcap=cap)
    got = out.cpu().double().view(n, H, r)
    for s, T in enumerate(lens):
        j = torch.arange(T)
        at = bt[s].long()[j // block] * block + j % block
        rows = cache.view(-1, G, width)[at].double()
        for h in range(H):
            z = rows[:, h // (H // G), r:] @ Q[s, h, r:].double()
            z = z * ks.view(-1)[at].double() if scaled else z
            z = cap * torch.tanh(z / cap) if cap else z
            z = z + table.double()[(T - 1 - j).clamp(max=69), h] if bias else z
            want = torch.softmax(z, 0) @ rows[:, h // (H // G), :r]
            assert float((got[s, h] - want).abs().max() / want.abs().max()) < TOL, (T, h)
