"""The matrix-core tile forms of i64h_linear_run against 64-bit products of the same bf16 values: every form at sizes around its tiles' edges,
ragged k, column offsets, gathered rows, rows dealt to experts, gate / up pairs, the normed input."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

# (one more than the form of the block kernel; "rows": the fragment-streaming kernel for at most 64 rows, the block kernel by size beyond)
FORMS = {"128x128": 1, "64x128 (32x64 in 32 bits)": 2, "64x64": 3, "64x64/2": 4, "32x64/4": 5, "16x64/4": 6, "16x128/2 pair": 7, "32x128/2": 8, "by size": 0, "rows": -1}


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


@pytest.fixture
def use_form():
    from vllm_i64_amd import ops_dense as D
    yield lambda name: D.call_dense("i64h_set_linear_skinny", {-1: 4, 0: 3}.get(FORMS[name], 16 * FORMS[name]))
    D.call_dense("i64h_set_linear_skinny", 3)


def bf16(t):
    return t.to(torch.bfloat16)


def close(got, ref, K):
    """fp32 sums of exact products of order one over sqrt(K): a rounding of 2^-24 of the running sum per term at most."""
    return torch.allclose(got.double().cpu(), ref, atol=K ** 0.5 * 2e-6, rtol=2e-5)


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("M,N,K", [(3, 4, 8), (17, 63, 72), (65, 129, 128), (130, 196, 1000), (129, 64, 64), (256, 260, 192)])
def test_tiles_and_ends(dev, use_form, form, M, N, K, exact):
    from vllm_i64_amd import ops_dense as D
    use_form(form)
    g = torch.Generator().manual_seed(M + N + K)
    a, w = torch.randn(M, K + 8, generator=g), bf16(torch.randn(2 * N, K, generator=g) / math.sqrt(K))
    b = torch.randn(N, generator=g)
    e = torch.randn(M, N + 3, generator=g)
    rounded = (lambda t: t.double()) if exact else (lambda t: bf16(t).double())
    A = rounded(a[:, 4:4 + K])
    ref, up = A @ w[:N].double().T, A @ w[N:].double().T
    ad, wd = a.to(dev), w.to(dev)
    out = torch.full((M, N + 5), 7.0, device=dev)
    kw = dict(n=N, k=K, a_off=4, lda=K + 8, exact=exact)
    D.linear(ad, wd, out, c_off=2, ldc=N + 5, **kw)
    assert close(out[:, 2:2 + N], ref, K) and bool((out[:, :2] == 7).all()) and bool((out[:, 2 + N:] == 7).all())
    out = torch.empty(M, N, device=dev)
    D.linear(ad, wd, out, bias=b.to(dev), epilogue=D.EPI_ADD, e=e.to(dev), e_off=1, lde=N + 3, **kw)
    assert close(out, ref + b.double() + e[:, 1:1 + N].double(), K)
    s = torch.rand(M, generator=g) + 0.5
    D.linear(ad, wd, out, epilogue=D.EPI_SILU_MUL, row_scale=s.to(dev), **kw)
    z, u = ref * s[:, None].double(), up * s[:, None].double()
    assert torch.allclose(out.double().cpu(), z * torch.sigmoid(z) * u, atol=1e-4, rtol=1e-4)
    if K % 8 == 0 and M > 2:
        nw = torch.rand(K, generator=g) + 0.5
        D.linear(ad, wd, out, in_norm_w=nw.to(dev), in_eps=1e-6, **kw)
        x = a[:, 4:4 + K]
        f = 1.0 / torch.sqrt(x.double().pow(2).mean(-1, keepdim=True) + 1e-6)
        assert close(out, (rounded(x * nw) @ w[:N].double().T) * f, K)


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("counts", [[5, 0, 70, 1], [0, 0, 0, 129], [64, 16, 128, 0], [1, 1, 1, 1]])
def test_rows_dealt_to_experts(dev, use_form, form, counts, exact):
    """Gathered rows into a gate / up pair with a factor per row, and rows as they lie; empty batches; a larger bound than there are rows."""
    from vllm_i64_amd import ops_dense as D
    use_form(form)
    rounded = (lambda t: t.double()) if exact else (lambda t: bf16(t).double())
    E, N, K, n = len(counts), 72, 136, 150
    g = torch.Generator().manual_seed(sum(counts))
    off = torch.tensor([0] + counts).cumsum(0).to(torch.int32)
    R = int(off[-1])
    rows = torch.randint(0, n, (R + 9,), generator=g).to(torch.int32)
    h, s = torch.randn(n, K, generator=g), torch.rand(R, generator=g) + 0.5
    w = bf16(torch.randn(E, 2 * N, K, generator=g) / math.sqrt(K))
    out = torch.full((R + 3, N), 7.0, device=dev)
    D.linear(h.to(dev), w.to(dev), out, m=max(counts), n=N, k=K, a_rows=rows.to(dev), batch=E, w_batch=2 * N * K, group_off=off.to(dev), row_scale=s.to(dev),
             epilogue=D.EPI_CLAMP_GLU, act_a=1.702, act_b=7.0, exact=exact)
    A = rounded(h)[rows[:R].long()]
    e_of = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    z = torch.einsum("rk,rnk->rn", A, w.double()[e_of]) * s[:, None].double()
    u, v = z[:, :N].clamp(max=7.0), z[:, N:].clamp(-7.0, 7.0)
    assert torch.allclose(out[:R].double().cpu(), u * torch.sigmoid(1.702 * u) * (v + 1), atol=1e-4, rtol=1e-4) and bool((out[R:] == 7).all())
    wd = bf16(torch.randn(E, K, N, generator=g) / math.sqrt(N))
    down = torch.full((R + 3, K), 7.0, device=dev)
    D.linear(out[:R], wd.to(dev), down, m=max(counts), n=K, k=N, batch=E, w_batch=K * N, group_off=off.to(dev), exact=exact)
    ref = torch.einsum("rn,rkn->rk", rounded(out[:R].cpu()), wd.double()[e_of])
    assert close(down[:R], ref, N) and bool((down[R:] == 7).all())


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("M", [5, 100])
def test_batched_over_heads(dev, use_form, form, M):
    from vllm_i64_amd import ops_dense as D
    use_form(form)
    H, n, k = 3, 40, 64
    g = torch.Generator().manual_seed(M)
    a, w = torch.randn(M, H * k, generator=g), bf16(torch.randn(H, n, k, generator=g) / 8)
    out = torch.empty(M, H * n, device=dev)
    D.linear(a.to(dev), w.to(dev), out, m=M, n=n, k=k, lda=H * k, ldc=H * n, batch=H, a_batch=k, w_batch=n * k, c_batch=n)
    for h in range(H):
        assert close(out[:, h * n:(h + 1) * n], bf16(a[:, h * k:(h + 1) * k]).double() @ w[h].double().T, k)


def test_not_a_number_stays_in_its_row(dev, use_form):
    """Rows past the end repeat the last one, chunks past k read as zeros: an infinity or NaN touches no other row."""
    from vllm_i64_amd import ops_dense as D
    a, w = torch.ones(66, 72), bf16(torch.ones(64, 72))
    a[65, 71], a[3, 0] = math.nan, math.inf
    for form in FORMS:
        use_form(form)
        out = torch.empty(66, 64, device=dev)
        D.linear(a.to(dev), w.to(dev), out)
        bad = ~torch.isfinite(out.cpu())
        assert bool(bad[[3, 65]].all()) and int(bad.sum()) == 128 and bool((out.cpu()[:3] == 72).all())


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("m", [2, 16, 40])
def test_no_more_rows_of_a_batch_than_the_launch_says(dev, use_form, form, m, exact):
    """Rows that a batch has beyond m are left alone, and those of the batches behind it are found all the same."""
    from vllm_i64_amd import ops_dense as D
    use_form(form)
    counts, N, K = [70, 3, 0, 45], 72, 136
    g = torch.Generator().manual_seed(m)
    off = torch.tensor([0] + counts).cumsum(0).to(torch.int32)
    R = int(off[-1])
    a, w = torch.randn(R, K, generator=g), bf16(torch.randn(len(counts), N, K, generator=g) / math.sqrt(K))
    out = torch.full((R, N), 7.0, device=dev)
    D.linear(a.to(dev), w.to(dev), out, m=m, n=N, k=K, batch=len(counts), w_batch=N * K, group_off=off.to(dev), exact=exact)
    got = out.cpu()
    for e, c in enumerate(counts):
        rows, o = min(c, m), int(off[e])
        A = a[o:o + rows].double() if exact else bf16(a[o:o + rows]).double()
        assert close(got[o:o + rows], A @ w[e].double().T, K) and bool((got[o + rows:o + c] == 7).all()), e


@pytest.mark.parametrize("M", [3, 64, 100])
def test_a_weight_of_more_than_4_gib(dev, use_form, M):
    """A tile's weights are addressed from the tile's first row: every column of a product whose weight does not fit 32-bit offsets."""
    from vllm_i64_amd import ops_dense as D
    use_form("by size")
    N, K = 262400, 8192
    g = torch.Generator().manual_seed(M)
    a, row = torch.randn(M, K, generator=g), bf16(torch.randn(K, generator=g) / math.sqrt(K))
    f = bf16(torch.arange(N) % 61 - 30)      # (row n of the weight: one row times a whole number)
    w = torch.empty(N, K, dtype=torch.bfloat16, device=dev)
    torch.mul(f.to(dev)[:, None], row.to(dev)[None, :], out=w)
    out = torch.empty(M, N, device=dev)
    D.linear(a.to(dev), w, out)
    cols = torch.cat([torch.arange(0, N, 997), torch.arange(N - 70, N)])
    ref = bf16(a).double() @ w[cols.to(dev)].cpu().double().T
    # (terms up to 30 times those of `close`)
    assert torch.allclose(out[:, cols.to(dev)].double().cpu(), ref, atol=30 * K ** 0.5 * 2e-6, rtol=2e-5)


# sizes that take a large form by their rule: 128 x 128 tiles (at least 200), 64 x 128 (at least 250, and fewer than 200 of the former), the 64 x 64 tile kernel (short
# k and many tiles, or k up to 32), 64-column tiles for narrow batches of many rows
LARGE = {"128x128": (1700, 1990, 136, 1), "64x128": (1000, 1996, 200, 1), "short k": (1500, 1990, 128, 1), "k 24": (70, 1000, 24, 1), "narrow": (1100, 60, 264, 16)}


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("size,epilogue", [(s, e) for s in LARGE for e in ("plain", "pair", "normed") if LARGE[s][3] == 1 or e == "plain"])      # (batches are plain products)
def test_large_forms_by_size(dev, use_form, size, epilogue, exact):
    from vllm_i64_amd import ops_dense as D
    use_form("by size")
    M, N, K, H = LARGE[size]
    g = torch.Generator().manual_seed(M + N)
    a, nw = torch.randn(M, H * K, generator=g), torch.rand(K, generator=g) + 0.5
    w = bf16(torch.randn(H, (2 if epilogue == "pair" else 1) * N, K, generator=g) / math.sqrt(K))
    out = torch.empty(M, H * N, device=dev)
    kw = {"plain": {}, "pair": {"epilogue": D.EPI_SILU_MUL}, "normed": {"in_norm_w": nw.to(dev), "in_eps": 1e-6}}[epilogue]
    D.linear(a.to(dev), w.to(dev), out, m=M, n=N, k=K, lda=H * K, ldc=H * N, batch=H, a_batch=K, w_batch=w[0].numel(), c_batch=N, exact=exact, **kw)
    for h in range(H):
        x = a[:, h * K:(h + 1) * K]
        x = x * nw if epilogue == "normed" else x
        ref = (x if exact else bf16(x)).double() @ w[h].double().T
        got = out[:, h * N:(h + 1) * N]
        if epilogue == "pair":
            ref = ref[:, :N] * torch.sigmoid(ref[:, :N]) * ref[:, N:]
            assert torch.allclose(got.double().cpu(), ref, atol=1e-4, rtol=1e-4)
        else:
            ref = ref / torch.sqrt(a.double().pow(2).mean(-1, keepdim=True) + 1e-6) if epilogue == "normed" else ref
            assert close(got, ref, K)


@pytest.mark.parametrize("M", [3, 8, 9, 64])
def test_gathered_rows_of_a_matrix_of_unknown_height(dev, use_form, M):
    """A caller that does not say how many rows the list may name: 64-bit addresses."""
    from vllm_i64_amd import _lib
    from vllm_i64_amd import ops_dense as D
    use_form("by size")
    n, N, K = 300, 5000, 264
    g = torch.Generator().manual_seed(M)
    a, w, rows = torch.randn(n, K, generator=g), bf16(torch.randn(N, K, generator=g) / math.sqrt(K)), torch.randint(0, n, (M,), generator=g).to(torch.int32)
    ad, wd, rd, out = a.to(dev), w.to(dev), rows.to(dev), torch.empty(M, N, device=dev)
    d = _lib.Linear(A=D.ptr(ad), lda=K, a_rows=D.ptr(rd), W=D.ptr(wd), C=D.ptr(out), ldc=N, M=M, N=N, K=K, batch=1)
    D.call_dense("i64h_linear_run", D._ref(d), D._stream())
    assert close(out, bf16(a[rows.long()]).double() @ w.double().T, K)


@pytest.mark.parametrize("form", ["64x64", "64x128 (32x64 in 32 bits)", "32x64/4", "16x64/4", "16x128/2 pair", "32x128/2", "by size"])
def test_parts_of_32_bit_rows(dev, use_form, form):
    """Rows of 32-bit values as three bf16 parts: values of all magnitudes keep their 24 bits, infinities and NaN stay what a product term by term makes of them, in rows and in weights."""
    from vllm_i64_amd import ops_dense as D
    use_form(form)
    M, N, K = 37, 72, 200
    g = torch.Generator().manual_seed(5)
    a = torch.randn(M, K, generator=g) * 10.0 ** torch.randint(-18, 18, (M, 1), generator=g)
    w = bf16(torch.randn(2 * N, K, generator=g))
    a[3] = torch.randint(-(1 << 24) + 1, 1 << 24, (K,), generator=g).float()      # all 24 bits used
    w[5] = 0
    w[5, 7] = 1
    out = torch.empty(M, N, device=dev)
    D.linear(a.to(dev), w[:N].contiguous().to(dev), out, exact=True)
    ref = a.double() @ w[:N].double().T
    assert torch.equal(out.cpu()[:, 5], a[:, 7])                                 # a value comes through as it is
    scale = a.double().abs() @ w[:N].double().abs().T
    assert ((out.double().cpu() - ref).abs() <= scale * 2.0 ** -23).all()        # (a sum of K terms rounded a few dozen times, each time by 2^-24 of a partial sum)
    a[1, 3], a[2, 4], a[4, 5], a[4, 6], a[6, 8] = float("inf"), float("-inf"), float("inf"), float("-inf"), float("nan")
    a[8, 0] = 3.3e38
    w[9, 11], w[10, 0], w[N + 9, 11] = float("inf"), float("-inf"), float("inf")
    D.linear(a.to(dev), w[:N].contiguous().to(dev), out, exact=True)
    ref = (a[:, None, :].double() * w[None, :N].double()).sum(-1).float()
    got = out.cpu()
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got[ref.isinf()], ref[ref.isinf()])
    D.linear(a.to(dev), w.to(dev), out, exact=True, epilogue=D.EPI_SILU_MUL)
    up = (a[:, None, :].double() * w[None, N:].double()).sum(-1).float()
    z = ref.double()
    want = (z * torch.sigmoid(z) * up.double()).float()
    ok = torch.isfinite(ref) & torch.isfinite(up)
    assert torch.equal(out.cpu()[ok].isnan(), want[ok].isnan()) and out.cpu()[(ref.isnan() | up.isnan())].isnan().all()


def test_a_row_of_nan_among_32_bit_rows_takes_no_longer(dev):
    """Sums that are no number are taken again term by term only where the row itself holds numbers: a sequence that is lost does not hold up the step's others (15 times as long if
    every sum is taken again; the smallest of some times each, and a bound far from both)."""
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(1)
    a, w, out = torch.randn(376, 1024, generator=g).to(dev), bf16(torch.randn(5760, 1024, generator=g)).to(dev), torch.empty(376, 5760, device=dev)

    def fastest():
        best = float("inf")
        for _ in range(8):
            e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            e[0].record()
            for _ in range(5):
                D.linear(a, w, out, exact=True)
            e[1].record()
            torch.cuda.synchronize()
            best = min(best, e[0].elapsed_time(e[1]))
        return best

    numbers = fastest()
    for lost in (slice(None), slice(1023, None)):
        a[3, lost] = float("nan")
        assert fastest() < 4 * numbers
        a[3] = 0
    a[3, 1023] = float("nan")
    D.linear(a, w, out, exact=True)
    assert out[3].isnan().all() and int(out.isnan().sum()) == 5760
