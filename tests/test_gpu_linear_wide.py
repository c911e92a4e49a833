"""Linears whose input rows come in bf16 against 64-bit products of the same values: every tile form around its tiles' edges, one to five steps of k,
gathered rows, rows dealt to batches, gate / up pairs, results in bf16."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

FORMS = {"by size": 3, "256x256": 16, "256x128": 32, "192x128": 48, "128x128": 64, "64x128": 80, "64x64": 96}


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


@pytest.fixture(params=FORMS)
def form(request):
    from vllm_i64_amd import ops_dense as D
    D.call_dense("i64h_set_linear_skinny", FORMS[request.param])
    yield request.param
    D.call_dense("i64h_set_linear_skinny", 3)


def close(got, ref, K):
    """fp32 sums of exact products of order one over sqrt(K): a rounding of 2^-24 of the running sum per term at most."""
    return torch.allclose(got.double().cpu(), ref, atol=K ** 0.5 * 2e-6, rtol=2e-5)


@pytest.mark.parametrize("M,N,K", [(1, 4, 64), (63, 63, 128), (65, 132, 192), (129, 64, 256), (193, 260, 320), (257, 129, 576)])
def test_tiles_and_ends(dev, form, M, N, K):
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randn(M, K + 16, generator=g).bfloat16()
    w, b, e = (torch.randn(2 * N, K, generator=g) / math.sqrt(K)).bfloat16(), torch.randn(N, generator=g), torch.randn(M, N, generator=g)
    A = a[:, 8:8 + K].double()
    ref, up = A @ w[:N].double().T, A @ w[N:].double().T
    ad, wd = a.to(dev), w.to(dev)
    kw = dict(a16=ad, n=N, k=K, a_off=8, lda=K + 16)
    out, out16 = torch.full((M, N + 3), 7.0, device=dev), torch.full((M, N + 3), 7.0, device=dev, dtype=torch.bfloat16)
    D.linear(None, wd, out, out16=out16, c_off=1, ldc=N + 3, **kw)
    assert close(out[:, 1:1 + N], ref, K) and torch.equal(out16, out.bfloat16()) and bool((out[:, 0] == 7).all()) and bool((out[:, 1 + N:] == 7).all())
    y = torch.empty(M, N, device=dev)
    D.linear(None, wd, y, bias=b.to(dev), epilogue=D.EPI_ADD, e=e.to(dev), lde=N, **kw)
    assert close(y, ref + b.double() + e.double(), K)
    y16 = torch.empty(M, N, device=dev, dtype=torch.bfloat16)
    D.linear(None, wd, None, out16=y16, epilogue=D.EPI_SCALE, scale=0.5, **kw)
    assert torch.allclose(y16.double().cpu(), 0.5 * ref, atol=1e-5, rtol=2.0 ** -8)      # (one rounding to eight bits)
    s = torch.rand(M, generator=g) + 0.5
    D.linear(None, wd, y, epilogue=D.EPI_SILU_MUL, row_scale=s.to(dev), **kw)
    z, u = ref * s[:, None].double(), up * s[:, None].double()
    assert torch.allclose(y.double().cpu(), z * torch.sigmoid(z) * u, atol=1e-4, rtol=1e-4)


def test_same_as_rows_rounded_while_staged(dev, form):
    """The sums run over k in one order in every form: the bits of a 128 x 128 tile that rounds its rows itself."""
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(3)
    a, w = torch.randn(300, 448, generator=g).to(dev), (torch.randn(200, 448, generator=g) / 20).bfloat16().to(dev)
    out, ref = torch.empty(300, 200, device=dev), torch.empty(300, 200, device=dev)
    D.linear(None, w, out, a16=a.bfloat16())
    D.call_dense("i64h_set_linear_skinny", 16)
    D.linear(a, w, ref)
    assert torch.equal(out, ref)


@pytest.mark.parametrize("counts", [[5, 0, 70, 1], [0, 0, 0, 259], [64, 16, 128, 0], [1, 1, 1, 1]])
def test_rows_dealt_to_experts(dev, form, counts):
    """Gathered rows into a gate / up pair with a factor per row, its bf16 results as they lie into the next; empty batches; a larger bound than there are rows."""
    from vllm_i64_amd import ops_dense as D
    E, N, K, n = len(counts), 128, 192, 150
    g = torch.Generator().manual_seed(sum(counts))
    off = torch.tensor([0] + counts).cumsum(0).to(torch.int32)
    R = int(off[-1])
    rows = torch.randint(0, n, (R + 9,), generator=g).to(torch.int32)
    h, s = torch.randn(n, K, generator=g).bfloat16(), torch.rand(R, generator=g) + 0.5
    w = (torch.randn(E, 2 * N, K, generator=g) / math.sqrt(K)).bfloat16()
    act = torch.full((R + 3, N), 7.0, device=dev, dtype=torch.bfloat16)
    D.linear(None, w.to(dev), None, a16=h.to(dev), out16=act, m=max(counts), n=N, k=K, a_rows=rows.to(dev), batch=E, w_batch=2 * N * K, group_off=off.to(dev), row_scale=s.to(dev),
             epilogue=D.EPI_CLAMP_GLU, act_a=1.702, act_b=7.0)
    e_of = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    z = torch.matmul(w.double()[e_of], h.double()[rows[:R].long()].unsqueeze(-1)).squeeze(-1) * s[:, None].double()
    u, v = z[:, :N].clamp(max=7.0), z[:, N:].clamp(-7.0, 7.0)
    assert torch.allclose(act[:R].double().cpu(), u * torch.sigmoid(1.702 * u) * (v + 1), atol=2e-4, rtol=2.0 ** -8) and bool((act[R:] == 7).all())
    wd = (torch.randn(E, K, N, generator=g) / math.sqrt(N)).bfloat16()
    down = torch.full((R + 3, K), 7.0, device=dev)
    D.linear(None, wd.to(dev), down, a16=act[:R], m=max(counts), n=K, k=N, batch=E, w_batch=K * N, group_off=off.to(dev))
    ref = torch.matmul(wd.double()[e_of], act[:R].double().cpu().unsqueeze(-1)).squeeze(-1)
    assert close(down[:R], ref, N) and bool((down[R:] == 7).all())


def test_not_a_number_stays_in_its_row(dev, form):
    from vllm_i64_amd import ops_dense as D
    a, w = torch.ones(66, 128).bfloat16(), torch.ones(64, 128).bfloat16()
    a[65, 127], a[3, 0] = math.nan, math.inf
    out = torch.empty(66, 64, device=dev)
    D.linear(None, w.to(dev), out, a16=a.to(dev))
    rest = [r for r in range(66) if r not in (3, 65)]
    assert bool((out[rest] == 128).all()) and bool(out[65].isnan().all()) and bool(out[3].isinf().all())


def test_refused(dev):
    from vllm_i64_amd import ops_dense as D
    a16, w, out = torch.ones(66, 96, device=dev).bfloat16(), torch.ones(64, 96, device=dev).bfloat16(), torch.empty(66, 64, device=dev)
    with pytest.raises(D._lib.I64HError):      # k no multiple of 64
        D.linear(None, w, out, a16=a16)
    a16, w = torch.ones(66, 128, device=dev).bfloat16(), torch.ones(64, 128, device=dev).bfloat16()
    for kw in (dict(exact=True), dict(epilogue=D.EPI_RELU_SQ), dict(in_norm_w=torch.ones(128, device=dev), in_eps=1e-6)):
        with pytest.raises(D._lib.I64HError):
            D.linear(None, w, out, a16=a16, **kw)
    with pytest.raises(D._lib.I64HError):      # a result in bf16 belongs to rows in bf16
        D.linear(a16.float(), w, out, out16=torch.empty(66, 64, device=dev).bfloat16())


def test_producers_round_once(dev):
    """The normed rows of the residual kernel (both forms) and of the gate norm, in bf16 beside fp32 and alone: the fp32 rows rounded."""
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator(device=dev).manual_seed(1)
    for W, S in ((96, 1), (1023, 1), (2048, 1), (64, 3)):
        x, w = torch.randn(S, 5, W, generator=g, device=dev), torch.rand(W, generator=g, device=dev)
        h, h16, alone = torch.empty(5, W, device=dev), *(torch.empty(5, W, device=dev, dtype=torch.bfloat16) for _ in range(2))
        D.streams_step(x, norm_w=w, eps=1e-6, h=h, h16=h16)
        D.streams_step(x, norm_w=w, eps=1e-6, h16=alone)
        assert torch.equal(h16, h.bfloat16()) and torch.equal(alone, h16)
    for width, n in ((128, 5), (130, 5), (512, 300)):
        y, z, w = (torch.randn(n, width, generator=g, device=dev) for _ in range(3))
        o, o16, alone = torch.empty(n, width, device=dev), *(torch.empty(n, width, device=dev, dtype=torch.bfloat16) for _ in range(2))
        kw = dict(groups=2, eps=1e-6, z=z, ldz=width, n=n, gate_after=True)
        D.gate_norm(y, w[0].contiguous(), o, out16=o16, **kw)
        D.gate_norm(y, w[0].contiguous(), None, out16=alone, **kw)
        assert torch.equal(o16, o.bfloat16()) and torch.equal(alone, o16)


@pytest.mark.parametrize("M,K", [(66, 64), (130, 256), (700, 128)])
def test_row_gates_over_rounded_rows(dev, M, K):
    """A head's value map over rows in bf16 with the head's gate per row: the fp32 result is that of the same numbers given in 32 bits, the bf16 one that, rounded."""
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(M)
    H, N = 5, 48
    a = torch.randn(M, H, K, generator=g).bfloat16().to(dev)
    w = torch.randn(H, N, K, generator=g).bfloat16().to(dev)
    e = torch.randn(M, H + 2, generator=g).to(dev)
    kw = dict(m=M, n=N, k=K, lda=H * K, ldc=H * N, batch=H, a_batch=K, w_batch=N * K, c_batch=N, epilogue=D.EPI_ROW_SIGMOID, e=e, e_off=1, lde=H + 2, e_batch=1)
    wide, wide16 = torch.empty(M, H * N, device=dev), torch.empty(M, H * N, device=dev, dtype=torch.bfloat16)
    D.linear(None, w, wide, a16=a.view(M, H * K), out16=wide16, **kw)
    ref = torch.matmul(a.double().transpose(0, 1), w.double().transpose(1, 2)).transpose(0, 1) * torch.sigmoid(e[:, 1:1 + H].double())[..., None]
    # K exact products summed in 32 bits: at most K 2^-24 of the sum of their magnitudes, below 6 sqrt(K)
    assert float((wide.view(M, H, N) - ref).abs().max()) <= K * 2.0 ** -24 * 6 * K ** 0.5 + 1e-5 and torch.equal(wide16, wide.bfloat16())


@pytest.mark.parametrize("M,N,pad", [(66, 8, 8), (65, 72, 4), (193, 132, 12), (257, 264, 8), (300, 384, 0)])
def test_lines_of_results(dev, form, M, N, pad):
    """Results that go out as whole lines: ends in rows and columns, both widths of a store, in fp32, in bf16 and in both; row gates, a bias, a pair; two batches beside
    each other.  What lies between the batches' columns and behind the rows stays."""
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(M + N)
    B, K, W = 2, 128, N + pad
    a = torch.randn(M, B * K, generator=g).bfloat16().to(dev)
    w = (torch.randn(B, 2 * N, K, generator=g) / 8).bfloat16().to(dev)
    e, bias = torch.randn(M, B, generator=g).to(dev), torch.randn(B, N, generator=g).to(dev)
    x = a.view(M, B, K).double().transpose(0, 1)
    first, second = torch.matmul(x, w[:, :N].double().transpose(1, 2)), torch.matmul(x, w[:, N:].double().transpose(1, 2))
    for opts, ref in ((dict(epilogue=D.EPI_ROW_SIGMOID, e=e, lde=B, e_batch=1, bias=bias, bias_batch=N), (first + bias[:, None].double()) * torch.sigmoid(e.double()).T[..., None]),
                      (dict(epilogue=D.EPI_SILU_MUL), first * torch.sigmoid(first) * second)):
        kw = dict(m=M, n=N, k=K, lda=B * K, ldc=B * W, batch=B, a_batch=K, w_batch=2 * N * K, c_batch=W, a16=a, **opts)
        out, out16 = torch.full((M + 1, B * W), 7.0, device=dev), torch.full((M + 1, B * W), 7.0, device=dev, dtype=torch.bfloat16)
        D.linear(None, w, out, out16=out16, **kw)
        alone, alone16 = torch.full_like(out, 7.0), torch.full_like(out16, 7.0)
        D.linear(None, w, alone, **kw)
        D.linear(None, w, None, out16=alone16, **kw)
        got = out[:M].view(M, B, W)
        # (the products below 64: their rounding through two factors)
        assert float((got[:, :, :N].transpose(0, 1) - ref).abs().max()) <= 64 * K * 2.0 ** -24
        assert bool((got[:, :, N:] == 7).all()) and bool((out[M] == 7).all())
        assert torch.equal(out16, out.bfloat16()) and torch.equal(alone, out) and torch.equal(alone16, out16)


@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 64, 65, 128, 150])
@pytest.mark.parametrize("N,K,B", [(16, 64, 1), (60, 256, 3), (130, 320, 1), (256, 1088, 2), (36, 2752, 1)])
def test_steps_of_k_dealt_to_waves(dev, M, N, K, B):
    """16 columns a workgroup, fewer and more steps of k than waves and stages, ends in rows and columns, one to three tiles of rows, batches; every epilogue, both results;
    and by size the same bits where the rule says so."""
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(M + N + K)
    W = N + 4
    a = torch.randn(M, B * K + 8, generator=g).bfloat16().to(dev)
    w = (torch.randn(B, N, K, generator=g) / math.sqrt(K)).bfloat16().to(dev)
    e, gate, bias = torch.randn(M, B * N, generator=g).to(dev), torch.randn(M, B, generator=g).to(dev), torch.randn(B, N, generator=g).to(dev)
    ref = torch.matmul(a[:, 8:].double().view(M, B, K).transpose(0, 1), w.double().transpose(1, 2)) + bias[:, None].double()
    kw = dict(m=M, n=N, k=K, a_off=8, lda=B * K + 8, ldc=B * W, batch=B, a_batch=K, w_batch=N * K, c_batch=W, bias=bias, bias_batch=N, a16=a)
    for opts, want in ((dict(), ref), (dict(epilogue=D.EPI_SCALE, scale=0.5), 0.5 * ref), (dict(epilogue=D.EPI_ADD, e=e, lde=B * N, e_batch=N), ref + e.double().view(M, B, N).transpose(0, 1)),
                       (dict(epilogue=D.EPI_ROW_SIGMOID, e=gate, lde=B, e_batch=1), ref * torch.sigmoid(gate.double()).T[..., None])):
        out, out16 = torch.full((M + 1, B * W), 7.0, device=dev), torch.full((M + 1, B * W), 7.0, device=dev, dtype=torch.bfloat16)
        D.call_dense("i64h_set_linear_skinny", 112)
        try:
            D.linear(None, w, out, out16=out16, **kw, **opts)
        finally:
            D.call_dense("i64h_set_linear_skinny", 3)
        got = out[:M].view(M, B, W)
        # (K products of about 1 / sqrt(K), their sum and what is added below 16: a rounding of 2^-24 each)
        assert float((got[:, :, :N].transpose(0, 1) - want).abs().max()) <= 2e-6 * K ** 0.5 + 1e-5
        assert bool((got[:, :, N:] == 7).all()) and bool((out[M] == 7).all()) and torch.equal(out16, out.bfloat16())
        if M <= 128 and K >= 256:
            sized = torch.full_like(out, 7.0)
            D.linear(None, w, sized, **kw, **opts)
            assert torch.equal(sized, out)


def test_rows_past_a_tiles_end(dev):
    """Infinities and NaN in rows behind a batch's last are none of its business."""
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(0)
    a = torch.randn(40, 256, generator=g).bfloat16()
    a[7:9] = float("nan")
    a[39] = float("inf")
    w = torch.randn(3, 128, 256, generator=g).bfloat16().to(dev)
    off = torch.tensor([0, 7, 9, 39], dtype=torch.int32, device=dev)
    out = torch.zeros(40, 128, device=dev)
    D.linear(None, w, out, a16=a.to(dev), m=40, batch=3, w_batch=128 * 256, group_off=off)
    assert torch.isfinite(out[:7]).all() and torch.isfinite(out[9:39]).all() and not torch.isfinite(out[7:9]).any() and not out[39].any()
    few = D.linear(None, w[0], torch.empty(7, 128, device=dev), a16=a[:7].to(dev))
    assert torch.isfinite(few).all()


def test_blocks_of_a_tile_follow_each_other(dev, form):
    """A wave hands itself one block of 16 rows after the other through the same LDS: whole numbers, exact in every sum and result, in all blocks of two tall tiles; several times."""
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(5)
    M, N, K = 512, 520, 64
    a, w = torch.randint(-2, 3, (M, K), generator=g), torch.randint(-1, 2, (N, K), generator=g)
    want = (a @ w.T).to(dev)      # at most 128: exact in bf16
    a16, w16 = a.bfloat16().to(dev), w.bfloat16().to(dev)
    for _ in range(5):
        out, out16 = torch.empty(M, N, device=dev), torch.empty(M, N, device=dev, dtype=torch.bfloat16)
        D.linear(None, w16, out, a16=a16, out16=out16)
        assert torch.equal(out.long(), want) and torch.equal(out16.long(), want)


@pytest.mark.parametrize("M,N,K", [(7, 64, 256), (16, 100, 576), (33, 48, 320), (70, 96, 1088), (128, 256, 256)])
def test_rows_that_are_no_numbers_beside_finite_ones(dev, M, N, K):
    """16 columns a workgroup: a row with an infinity or NaN is its own row's business, in the waves' sums as well, and a weight that is one its column's."""
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator().manual_seed(M)
    a, w = torch.randn(M, K, generator=g).bfloat16(), (torch.randn(N, K, generator=g) / math.sqrt(K)).bfloat16()
    clean = D.linear(None, w.to(dev), torch.empty(M, N, device=dev), a16=a.to(dev))
    assert torch.isfinite(clean).all()
    bad = torch.tensor([0, M // 2, M - 1])
    a[0, K - 1], a[M // 2, 0], a[M - 1, K // 2] = float("inf"), float("nan"), float("-inf")
    w[N - 1, 5] = float("nan")
    out, out16 = torch.full((M, N), 7.0, device=dev), torch.full((M, N), 7.0, device=dev, dtype=torch.bfloat16)
    D.linear(None, w.to(dev), out, a16=a.to(dev), out16=out16)
    good = torch.ones(M, dtype=torch.bool)
    good[bad] = False
    assert torch.equal(out.cpu()[good, :N - 1], clean.cpu()[good, :N - 1]) and not torch.isfinite(out.cpu()[bad]).any() and out[:, N - 1].isnan().all()
    assert torch.equal(out16.isnan(), out.isnan()) and torch.equal(out16.nan_to_num(0.0), out.bfloat16().nan_to_num(0.0))


@pytest.mark.parametrize("M,N,K,thin", [(3, 4112, 3072, True), (32, 8192, 3072, True), (33, 4112, 3072, False), (32, 8193, 3072, False), (32, 4112, 3008, False)])
def test_two_rounds_of_narrow_tiles_under_a_long_k(dev, M, N, K, thin):
    """Either side of the line up to which 16 columns a workgroup are taken for two rounds: the bits of that form, or of the 64 x 64 tiles; close to 64 bits."""
    from vllm_i64_amd import ops_dense as D
    g = torch.Generator(device=dev).manual_seed(M)
    a, w = torch.randn(M, K, generator=g, device=dev).bfloat16(), (torch.randn(N, K, generator=g, device=dev) / math.sqrt(K)).bfloat16()
    out, forced = torch.empty(M, N, device=dev), torch.empty(M, N, device=dev)
    D.linear(None, w, out, a16=a)
    D.call_dense("i64h_set_linear_skinny", 112 if thin else 96)
    try:
        D.linear(None, w, forced, a16=a)
    finally:
        D.call_dense("i64h_set_linear_skinny", 3)
    assert torch.equal(out, forced)
    assert float((out.double() - a.double() @ w.double().t()).abs().max()) <= 2e-6 * K ** 0.5 + 1e-5
