"""The matrix-core attention of prompt portions (bf16 and 32-bit caches) against 64-bit attention over the same rows: every number of heads that shares a workgroup, key widths
that are no multiple of a step, pages of any size, tiles that hold rows of several sequences, cached tokens in front, windows, kept
first positions, sinks, soft cap."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


def pages(lens, past, block, g):
    need = [(n + p + block - 1) // block for n, p in zip(lens, past)]
    order = torch.randperm(sum(need), generator=g).to(torch.int32)
    bt, at = torch.zeros(len(lens), max(need), dtype=torch.int32), 0
    for i, k in enumerate(need):
        bt[i, :k] = order[at:at + k]
        at += k
    pos = torch.cat([torch.arange(p, p + n, dtype=torch.int32) for n, p in zip(lens, past)])
    slots = torch.cat([torch.full((n,), i, dtype=torch.int32) for i, n in enumerate(lens)])
    return bt, pos, slots, sum(need)


def reference(q, keys, values, pos, scale, window, keep, cap, sink):
    """q [n, H, d], keys [H, T, d], values [H, T, v]: one sequence, 64 bits."""
    s = torch.einsum("nhd,htd->hnt", q.double(), keys.double()) * scale
    if cap:
        s = cap * torch.tanh(s / cap)
    j = torch.arange(keys.shape[1])[None, :]
    i = pos[:, None].long()
    see = (j <= i) if not window else (j <= i) & ((i - j < window) | (j < keep))
    s = torch.cat([s.masked_fill(~see, -math.inf), sink.double().view(-1, 1, 1).expand(-1, s.shape[1], 1)], -1)
    return torch.einsum("hnt,htv->nhv", torch.softmax(s, -1)[..., :-1], values.double())


# (the last one: more portions in a tile of 64 rows than workgroups that they are dealt to)
LENS = [([1, 15, 16, 17, 40], [0, 3, 0, 31, 0]), ([70], [0]), ([33, 2], [64, 5]), ([2, 1] * 40 + [70], [3, 40] * 40 + [0])]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("lens,past", LENS)
@pytest.mark.parametrize("H,G,dim,vdim", [(4, 1, 64, 64), (2, 1, 32, 32), (3, 1, 64, 16), (8, 2, 24, 48), (6, 2, 128, 128), (12, 3, 8, 64)])
@pytest.mark.parametrize("block,window,keep,cap", [(16, 0, 0, 0.0), (16, 20, 3, 0.0), (6, 33, 40, 0.0), (16, 0, 0, 2.0)])
def test_keys_and_values(dev, lens, past, H, G, dim, vdim, block, window, keep, cap, dtype):
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(H + dim + window)
    bt, pos, slots, blocks = pages(lens, past, block, g)
    n, w = int(pos.numel()), vdim + dim
    cache = torch.randn(blocks, block, G * w, generator=g).to(dtype)
    q = torch.randn(n, H, w, generator=g)
    q[:, :, :vdim] = 0
    sink = torch.randn(H, generator=g)
    out = torch.full((n, H * vdim), 7.0, device=dev)
    D.kattn(q.to(dev), cache.to(dev), None, bt.to(dev), slots.to(dev), pos.to(dev), chunk=0, bias=None, sink=True, heads=H, kv_heads=G, dim=dim, vdim=vdim, out=out, n=n, mode=3,
            window=window, keep_first=keep, softcap=cap, sink_w=sink.to(dev))
    # the prep kernel's scale is in the query: the launch has none of its own
    at = 0
    for i, (m, p) in enumerate(zip(lens, past)):
        j = torch.arange(m + p)
        rows = cache[bt[i].long()[j // block], j % block].view(m + p, G, w).repeat_interleave(H // G, 1).transpose(0, 1)
        ref = reference(q[at:at + m, :, vdim:], rows[..., vdim:], rows[..., :vdim], pos[at:at + m], 1.0, window, keep, cap, sink)
        got = out[at:at + m].view(m, H, vdim).double().cpu()
        # two bf16 terms of query and weight: 2^-16 relative each, scores of up to sqrt(dim) * 4; 32-bit products: 2^-24 times the score
        tol = 1e-3 if dtype == torch.bfloat16 else 2e-5
        assert torch.allclose(got, ref, atol=2 * tol, rtol=tol), float((got - ref).abs().max())
        at += m


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("lens,past", LENS)
@pytest.mark.parametrize("H,r,e", [(4, 256, 32), (5, 256, 64), (8, 32, 8), (16, 128, 0), (2, 64, 64), (4, 144, 24)])
@pytest.mark.parametrize("window", [0, 25])
def test_latent_rows(dev, lens, past, H, r, e, window, dtype):
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(H + r + e)
    bt, pos, slots, blocks = pages(lens, past, 16, g)
    n = int(pos.numel())
    cache = torch.randn(blocks, 16, r + e, generator=g).to(dtype)
    q = torch.randn(n, H, r + e, generator=g)
    sink = torch.randn(H, generator=g)
    out = torch.full((n * H * r,), 7.0, device=dev)
    D.latent_attn(q.to(dev).flatten(), cache.to(dev), bt.to(dev), slots.to(dev), pos.to(dev), window=window, scale=0.1, heads=H, kv_rank=r, rot_dim=e, out=out, n=n, mode=3, sink=sink.to(dev))
    at = 0
    for i, (m, p) in enumerate(zip(lens, past)):
        j = torch.arange(m + p)
        rows = cache[bt[i].long()[j // 16], j % 16].expand(H, -1, -1)
        ref = reference(q[at:at + m], rows, rows[..., :r], pos[at:at + m], 0.1, window, 0, 0.0, sink)
        got = out.view(n, H, r)[at:at + m].double().cpu()
        tol = 5e-4 if dtype == torch.bfloat16 else 1e-5
        assert torch.allclose(got, ref, atol=tol, rtol=tol), float((got - ref).abs().max())
        at += m


UNSEEN = [(4, 1, 32, 64, 0, 0), (2, 1, 32, 32, 9, 2), (3, 1, 32, 256, 0, 0)]


@pytest.mark.parametrize("bad", [math.inf, math.nan])
@pytest.mark.parametrize("H,G,dim,vdim,window,keep", UNSEEN)
def test_unseen_values_of_32_bits(dev, H, G, dim, vdim, window, keep, bad):
    """A key that a row does not see adds nothing to the row, also where its value is no finite number."""
    unseen_values(dev, H, G, dim, vdim, window, keep, bad, torch.float32, 2e-5)


@pytest.mark.parametrize("bad", [math.inf, -math.inf, math.nan])
@pytest.mark.parametrize("H,G,dim,vdim,window,keep", UNSEEN + [(12, 3, 8, 64, 0, 0)])
def test_unseen_values_of_bf16(dev, H, G, dim, vdim, window, keep, bad):
    """The same over a bf16 cache: rows of another sequence and earlier rows of the same one are right beside such a value."""
    unseen_values(dev, H, G, dim, vdim, window, keep, bad, torch.bfloat16, 1e-3)


def unseen_values(dev, H, G, dim, vdim, window, keep, bad, dtype, tol):
    from vllm_i64_amd import ops_dense as D
    lens, past, at_key = [40, 30, 5], [0, 3, 0], [33, 4, 2]
    g = torch.Generator().manual_seed(H + vdim)
    bt, pos, slots, blocks = pages(lens, past, 16, g)
    n, w = int(pos.numel()), vdim + dim
    cache = torch.randn(blocks, 16, G * w, generator=g).to(dtype)
    for i, j in enumerate(at_key):
        cache[bt[i, j // 16], j % 16, i] = bad
    q = torch.randn(n, H, w, generator=g)
    q[:, :, :vdim] = 0
    out = torch.full((n, H * vdim), 7.0, device=dev)
    D.kattn(q.to(dev), cache.to(dev), None, bt.to(dev), slots.to(dev), pos.to(dev), chunk=0, bias=None, sink=False, heads=H, kv_heads=G, dim=dim, vdim=vdim, out=out, n=n, mode=3,
            window=window, keep_first=keep)
    at = 0
    for i, (m, p) in enumerate(zip(lens, past)):
        j = torch.arange(m + p)
        rows = cache[bt[i].long()[j // 16], j % 16].view(m + p, G, w).repeat_interleave(H // G, 1).transpose(0, 1)
        values = rows[..., :vdim].clone()
        values[:H // G, at_key[i], i] = 0.0
        ref = reference(q[at:at + m, :, vdim:], rows[..., vdim:], values, pos[at:at + m], 1.0, window, keep, 0.0, torch.full((H,), -math.inf))
        got = out[at:at + m].view(m, H, vdim).double().cpu()
        d = pos[at:at + m].long() - at_key[i]
        sees = (d >= 0) & ((d < window) | (at_key[i] < keep)) if window else d >= 0
        group = got[:, :H // G]      # (the value lies in the first key head's columns)
        assert bool((~torch.isfinite(group[sees][..., i])).all())
        ref[:, :H // G, i] = torch.where(sees[:, None], 0.0, ref[:, :H // G, i])
        group[:, :, i] = torch.where(sees[:, None], 0.0, group[:, :, i])
        assert torch.allclose(got, ref, atol=2 * tol, rtol=tol), float((got - ref).abs().max())
        at += m


def test_options_of_key_heads_stay_refused_over_32_bits(dev):
    from vllm_i64_amd import _lib
    from vllm_i64_amd import ops_dense as D
    f, i = torch.zeros(4096, device=dev), torch.zeros(64, dtype=torch.int32, device=dev)
    for option in ({"kv_groups": 2}, {"row_stride": 64}, {"chunk": 16}, {"kscale": D.ptr(f)}, {"bias": D.ptr(f), "bias_rows": 4}):
        d = _lib.LatentAttn(Q=D.ptr(f), cache=D.ptr(f), cache_dtype=0, block_table=D.ptr(i), max_blocks_per_seq=1, block_size=16, slot_ids=D.ptr(i), positions=D.ptr(i), scale=1.0,
                            out=D.ptr(f), n=1, heads=2, kv_rank=32, rot_dim=0, mode=3, **option)
        with pytest.raises(_lib.I64HError, match="matrix-core form only"):
            D.call_dense("i64h_latent_attn", D._ref(d), D._stream())


def test_a_score_of_minus_infinity_is_a_weight_of_zero(dev):
    """An infinite first column of a key meets negative queries only: the columns past a key's end, which a step of the products takes along, add nothing to its score.  (32-bit products: two bf16 terms of a query may differ in sign, and then meet an infinity as both.)"""
    from vllm_i64_amd import ops_dense as D
    H, dim, vdim, n = 4, 24, 48, 20
    g = torch.Generator().manual_seed(5)
    bt, pos, slots, blocks = pages([n], [0], 16, g)
    cache = torch.randn(blocks, 16, vdim + dim, generator=g)
    cache[bt[0, 0], 3, vdim] = math.inf
    q = torch.randn(n, H, vdim + dim, generator=g)
    q[:, :, :vdim] = 0
    q[:, :, vdim] = -q[:, :, vdim].abs() - 0.1
    out = torch.empty(n, H * vdim, device=dev)
    D.kattn(q.to(dev), cache.to(dev), None, bt.to(dev), slots.to(dev), pos.to(dev), chunk=0, bias=None, sink=False, heads=H, kv_heads=1, dim=dim, vdim=vdim, out=out, n=n, mode=3)
    j = torch.arange(n)
    rows = cache[bt[0].long()[j // 16], j % 16].expand(H, -1, -1)
    ref = reference(q[:, :, vdim:], rows[..., vdim:], rows[..., :vdim], pos, 1.0, 0, 0, 0.0, torch.full((H,), -math.inf))
    assert torch.allclose(out.view(n, H, vdim).double().cpu(), ref, atol=4e-5, rtol=2e-5)


@pytest.mark.parametrize("dim,vdim", [(24, 64), (40, 32), (8, 256)])
def test_an_infinite_first_column_of_a_bf16_key(dev, dim, vdim):
    """A step of the products takes columns past a key's end along, as zeros: beside an infinite first column they would make a score of minus infinity
    no number.  (The first column's queries are such that both of their bf16 terms, after the factor log2(e), are negative.)"""
    from vllm_i64_amd import ops_dense as D
    H, n = 4, 20
    g = torch.Generator().manual_seed(5)
    bt, pos, slots, blocks = pages([n], [0], 16, g)
    cache = torch.randn(blocks, 16, vdim + dim, generator=g).to(torch.bfloat16)
    cache[bt[0, 0], 3, vdim] = math.inf
    q = torch.randn(n, H, vdim + dim, generator=g)
    q[:, :, :vdim] = 0
    q[:, :, vdim] = -(1.0 + 2.0 ** -10) / math.log2(math.e)
    out = torch.empty(n, H * vdim, device=dev)
    D.kattn(q.to(dev), cache.to(dev), None, bt.to(dev), slots.to(dev), pos.to(dev), chunk=0, bias=None, sink=False, heads=H, kv_heads=1, dim=dim, vdim=vdim, out=out, n=n, mode=3)
    j = torch.arange(n)
    rows = cache[bt[0].long()[j // 16], j % 16].expand(H, -1, -1)
    ref = reference(q[:, :, vdim:], rows[..., vdim:], rows[..., :vdim], pos, 1.0, 0, 0, 0.0, torch.full((H,), -math.inf))
    assert torch.allclose(out.view(n, H, vdim).double().cpu(), ref, atol=2e-3, rtol=1e-3)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_without_a_sequence(dev, dtype):
    """Rows whose slot is -1 see no key, also where rows are summed key by key because a value of their tile is no finite number: the sink alone, zeros."""
    from vllm_i64_amd import ops_dense as D
    H, dim, vdim, n = 4, 32, 64, 24
    g = torch.Generator().manual_seed(7)
    bt, pos, slots, blocks = pages([n], [0], 16, g)
    cache = torch.randn(blocks, 16, vdim + dim, generator=g).to(dtype)
    q = torch.randn(n, H, vdim + dim, generator=g)
    q[:, :, :vdim] = 0
    slots[[2, 5, 20]] = -1
    cache[bt[0, 0], 9, 7] = math.inf
    out = torch.empty(n, H * vdim, device=dev)
    D.kattn(q.to(dev), cache.to(dev), None, bt.to(dev), slots.to(dev), pos.to(dev), chunk=0, bias=None, sink=True, heads=H, kv_heads=1, dim=dim, vdim=vdim, out=out, n=n, mode=3)
    rows = cache[bt[0].long()[torch.arange(n) // 16], torch.arange(n) % 16].expand(H, -1, -1)
    values = rows[..., :vdim].clone()
    values[:, 9, 7] = 0.0
    ref = reference(q[:, :, vdim:], rows[..., vdim:], values, pos, 1.0, 0, 0, 0.0, torch.zeros(H))
    ref[slots < 0] = 0.0
    got = out.view(n, H, vdim).double().cpu()
    sees = (pos >= 9) & (slots >= 0)
    assert bool((~torch.isfinite(got[sees][..., 7])).all())
    got[sees, :, 7] = ref[sees, :, 7] = 0.0
    tol = 1e-3 if dtype == torch.bfloat16 else 2e-5
    assert torch.allclose(got, ref, atol=2 * tol, rtol=tol), float((got - ref).abs().max())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_scores_of_minus_infinity_beside_a_value_that_is_no_number(dev, dtype):
    """Rows that are summed key by key, because a later key's value in their tile is no finite number, while a distance bias of minus infinity hides all
    but their last keys: the first 64 scores are minus infinity, weights of zero."""
    from vllm_i64_amd import ops_dense as D
    H, dim, vdim, n, past, reach = 4, 32, 64, 16, 144, 5
    g = torch.Generator().manual_seed(6)
    bt, pos, slots, blocks = pages([n], [past], 16, g)
    cache = torch.randn(blocks, 16, vdim + dim, generator=g).to(dtype)
    last = past + n - 1
    cache[bt[0, last // 16], last % 16, 7] = math.nan      # seen by the last row only
    q = torch.randn(n, H, vdim + dim, generator=g)
    q[:, :, :vdim] = 0
    bias = torch.randn(reach + 1, H, generator=g)
    bias[reach:] = -math.inf      # (the table's last row stands for all distances behind it)
    out = torch.empty(n, H * vdim, device=dev)
    D.kattn(q.to(dev), cache.to(dev), None, bt.to(dev), slots.to(dev), pos.to(dev), chunk=0, bias=bias.to(dev), sink=False, heads=H, kv_heads=1, dim=dim, vdim=vdim, out=out, n=n, mode=3)
    j = torch.arange(past + n)
    rows = cache[bt[0].long()[j // 16], j % 16].double()
    s = torch.einsum("nhd,td->hnt", q[:, :, vdim:].double(), rows[:, vdim:])
    d = pos[:, None].long() - j[None, :]
    s = (s + bias.double()[d.clamp(0, reach)].permute(2, 0, 1)).masked_fill(d < 0, -math.inf)
    ref = torch.einsum("hnt,tv->nhv", torch.softmax(s, -1)[:, :-1], rows[:, :vdim].nan_to_num())
    got = out.view(n, H, vdim).double().cpu()
    assert bool(got[-1, :, 7].isnan().all())
    tol = 1e-3 if dtype == torch.bfloat16 else 2e-5
    assert torch.allclose(got[:-1], ref, atol=2 * tol, rtol=tol), float((got[:-1] - ref).abs().max())


# (one to seven tiles of 32 keys, a last one of one key and of all, several runs a tile of rows; the sizes whose tiles go from memory to LDS by themselves)
TILES = [([1, 16, 31], [0, 15, 1]), ([2, 17, 5, 3], [30, 48, 91, 93]), ([40, 3], [88, 157]), ([7, 64], [0, 150])]


@pytest.mark.parametrize("lens,past", TILES)
@pytest.mark.parametrize("H,G,w,r,off", [(4, 1, 288, 256, 0), (3, 1, 288, 256, 0), (8, 2, 128, 64, 64), (2, 2, 128, 64, 64), (6, 3, 256, 128, 128), (4, 1, 256, 128, 128)])
@pytest.mark.parametrize("block,window,keep", [(16, 0, 0), (5, 0, 0), (16, 45, 3), (12, 33, 40)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_of_exact_sizes(dev, lens, past, H, G, w, r, off, block, window, keep, dtype):
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(H + w + window)
    bt, pos, slots, blocks = pages(lens, past, block, g)
    n = int(pos.numel())
    cache = torch.randn(blocks, block, G * w, generator=g).to(dtype)
    q = torch.randn(n, H, w, generator=g)
    q[:, :, :off] = 0
    sink = torch.randn(H, generator=g)
    out = torch.full((n * H * r,), 7.0, device=dev)
    args = (q.to(dev).flatten(), cache.to(dev), bt.to(dev), slots.to(dev), pos.to(dev))
    if off:
        D.kattn(args[0].view(n, -1), args[1], None, *args[2:], chunk=0, bias=None, sink=True, heads=H, kv_heads=G, dim=w - r, vdim=r, out=out.view(n, -1), n=n, mode=3, window=window,
                keep_first=keep, sink_w=sink.to(dev))
        scale = 1.0
    else:
        keep, scale = 0, 0.1
        D.latent_attn(*args, window=window, scale=scale, heads=H, kv_rank=r, rot_dim=w - r, out=out, n=n, mode=3, sink=sink.to(dev))
    at = 0
    for i, (m, p) in enumerate(zip(lens, past)):
        j = torch.arange(m + p)
        rows = cache[bt[i].long()[j // block], j % block].view(m + p, G, w).repeat_interleave(H // G, 1).transpose(0, 1)
        ref = reference(q[at:at + m, :, off:], rows[..., off:], rows[..., :r], pos[at:at + m], scale, window, keep, 0.0, sink)
        got = out.view(n, H, r)[at:at + m].double().cpu()
        # two bf16 terms of query and weight: 2^-16 relative each, scores of up to sqrt(dim) * 4; 32-bit products: 2^-24 times the score
        tol = 1e-3 if dtype == torch.bfloat16 else 2e-5
        assert torch.allclose(got, ref, atol=2 * tol, rtol=tol), float((got - ref).abs().max())
        at += m


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,G,dim,vdim,window,keep", [(4, 1, 64, 64, 0, 0), (2, 1, 128, 128, 9, 2), (8, 2, 64, 64, 9, 2)])
def test_unseen_values_in_rows_of_exact_sizes(dev, H, G, dim, vdim, window, keep, dtype):
    for bad in (math.inf, -math.inf, math.nan):
        unseen_values(dev, H, G, dim, vdim, window, keep, bad, dtype, 1e-3 if dtype == torch.bfloat16 else 2e-5)


def test_many_32_bit_rows_of_exact_sizes(dev):
    """Enough workgroups for the form that gives each wave its own rows: 1700 rows of 16 heads over 4, the same rows in one launch and in portions."""
    from vllm_i64_amd import ops_dense as D
    H, G, w, n = 16, 4, 128, 1700
    g = torch.Generator().manual_seed(3)
    bt, pos, slots, blocks = pages([n], [0], 16, g)
    args = [torch.randn(n, H * w, generator=g).to(dev), torch.randn(blocks, 16, G * w, generator=g).to(dev)]
    args[0].view(n, H, w)[:, :, :64] = 0
    def run(cuts):
        out = torch.empty(n, H * 64, device=dev)
        for a, b in cuts:
            D.kattn(args[0][a:b], args[1], None, bt.to(dev), slots[a:b].to(dev), pos[a:b].to(dev), chunk=0, bias=None, sink=False, heads=H, kv_heads=G, dim=64, vdim=64, out=out[a:b],
                    n=b - a, mode=3, window=100, keep_first=2)
        return out
    one, cut = run([(0, n)]), run([(0, 700), (700, 1501), (1501, n)])
    assert torch.allclose(one, cut, atol=4e-5, rtol=2e-5), float((one - cut).abs().max())


@pytest.mark.parametrize("mode,splits", [(3, 1), (2, 1), (2, 3)])
@pytest.mark.parametrize("H,G,dim,vdim", [(4, 2, 64, 64), (6, 3, 128, 128), (3, 1, 32, 48)])
def test_kattn_result_in_bf16(dev, mode, splits, H, G, dim, vdim):
    """A result asked for in bf16 is the 32-bit one, rounded once: rows of whole tiles and rest, whole prompts and one row a sequence, its keys in one part or
    several; nothing beyond the rows is written, and the forms that have no such result say so."""
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(H)
    lens, past = ([1, 15, 17, 40, 70], [0, 3, 31, 0, 9]) if mode == 3 else ([1] * 5, [0, 3, 31, 130, 200])
    bt, pos, slots, blocks = pages(lens, past, 16, g)
    n, w = int(pos.numel()), vdim + dim
    cache = torch.randn(blocks, 16, G * w, generator=g).bfloat16().to(dev)
    q = torch.randn(n, H, w, generator=g)
    q[:, :, :vdim] = 0
    kw = dict(chunk=0, bias=None, sink=False, heads=H, kv_heads=G, dim=dim, vdim=vdim, n=n, mode=mode, splits=splits)
    args = (q.to(dev), cache, None, bt.to(dev), slots.to(dev), pos.to(dev))
    out = D.kattn(*args, out=torch.empty(n, H * vdim, device=dev), **kw)
    out16 = D.kattn(*args, out=torch.full((n + 1, H * vdim), 7.0, device=dev, dtype=torch.bfloat16), **kw)
    assert torch.equal(out16[:n], out.bfloat16()) and bool((out16[n] == 7).all())
    if mode == 2:      # (the knob that keeps such rows off the matrix cores leaves a launch with this result where it is)
        D.call_dense("i64h_set_latent_attn_decode_form", 0)
        try:
            again = D.kattn(*args, out=torch.empty_like(out16), **kw)
        finally:
            D.call_dense("i64h_set_latent_attn_decode_form", 1)
        assert torch.equal(again[:n], out16[:n])
    with pytest.raises(Exception, match="bf16"):
        D.kattn(*args, out=out16, **{**kw, "mode": 1, "splits": 1})
    with pytest.raises(Exception, match="bf16"):
        D.kattn(args[0], cache.float(), *args[2:], out=out16, **kw)


@pytest.mark.parametrize("mode,splits", [(3, 1), (2, 1), (2, 3)])
@pytest.mark.parametrize("H,r,e", [(16, 256, 32), (4, 128, 16), (5, 64, 32)])
def test_latent_result_in_bf16(dev, mode, splits, H, r, e):
    """The same of latent rows."""
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(H + r)
    lens, past = ([1, 15, 17, 40, 70], [0, 3, 31, 0, 9]) if mode == 3 else ([1] * 5, [0, 3, 31, 130, 200])
    bt, pos, slots, blocks = pages(lens, past, 16, g)
    n = int(pos.numel())
    cache = torch.randn(blocks, 16, r + e, generator=g).bfloat16().to(dev)
    args = (torch.randn(n * H * (r + e), generator=g).to(dev), cache, bt.to(dev), slots.to(dev), pos.to(dev))
    kw = dict(window=0, scale=0.1, heads=H, kv_rank=r, rot_dim=e, n=n, mode=mode, splits=splits)
    out = D.latent_attn(*args, out=torch.empty(n * H * r, device=dev), **kw)
    out16 = D.latent_attn(*args, out=torch.full(((n + 1) * H * r,), 7.0, device=dev, dtype=torch.bfloat16), **kw)
    assert torch.equal(out16[: n * H * r], out.bfloat16()) and bool((out16[n * H * r:] == 7).all())
    with pytest.raises(Exception, match="bf16"):
        D.latent_attn(args[0], cache.float(), *args[2:], out=out16, **kw)
    with pytest.raises(Exception, match="bf16"):
        D.latent_attn(*args, out=out16, **{**kw, "mode": 1, "splits": 1})


@pytest.mark.parametrize("H,G,dim", [(32, 8, 64), (8, 2, 64), (16, 4, 128)])
@pytest.mark.parametrize("lens,past", [([3] * 64, 40), ([2] * 150, 9), ([16] * 24, 0)])
def test_32_bit_rows_of_many_sequences_by_their_number(dev, H, G, dim, lens, past):
    """The number of sequences chooses between forms whose sums run in another order, and nothing else: with and without it, against 64 bits."""
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(len(lens))
    bt, pos, slots, blocks = pages(lens, [past] * len(lens), 16, g)
    n, w = int(pos.numel()), 2 * dim
    cache = torch.randn(blocks, 16, G * w, generator=g)
    q = torch.randn(n, H, w, generator=g) * dim ** -0.5
    q[:, :, :dim] = 0
    sink = torch.randn(H, generator=g)
    args = (q.to(dev).view(n, -1), cache.to(dev), None, bt.to(dev), slots.to(dev), pos.to(dev))
    got = [D.kattn(*args, chunk=0, bias=None, sink=True, sink_w=sink.to(dev), heads=H, kv_heads=G, dim=dim, vdim=dim, out=torch.full((n, H * dim), 7.0, device=dev), n=n, mode=3, seqs=k).double().cpu().view(n, H, dim)
           for k in (0, len(lens))]
    at = 0
    for i, m in enumerate(lens):
        j = torch.arange(m + past)
        rows = cache[bt[i].long()[j // 16], j % 16].view(m + past, G, w).repeat_interleave(H // G, 1).transpose(0, 1)
        ref = reference(q[at:at + m, :, dim:], rows[..., dim:], rows[..., :dim], pos[at:at + m], 1.0, 0, 0, 0.0, sink)
        for x in got:
            assert torch.allclose(x[at:at + m], ref, atol=4e-5, rtol=2e-5), (i, float((x[at:at + m] - ref).abs().max()))
        at += m
