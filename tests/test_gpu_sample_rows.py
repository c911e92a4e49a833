"""The token draw against 64-bit softmax sums: vocabulary sizes around what a workgroup holds, every route (listed candidates, keys in registers, keys read
again), ties, masked and non-finite logits."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def draw(x, T, k, p, u):
    from vllm_i64_amd import ops_dense as D
    n = x.shape[0]
    dev = torch.device("cuda:0")
    f = lambda v, dt: torch.full((n,), v, dtype=dt, device=dev)
    return D.sample_rows(x.to(dev), temperature=f(T, torch.float32), top_k=f(k, torch.int32), top_p=f(p, torch.float32), u=u.to(dev)).cpu()


def check(x, T, k, p, u, got):
    """Every drawn token is kept, and u lies within fp32 rounding of the token's stretch of the running sum."""
    V = x.shape[1]
    for row, uu, tok in zip(x.double(), u.double(), got.tolist()):
        w = torch.exp((row - row.max()) / float(torch.tensor(T)))
        keep = torch.ones(V, dtype=torch.bool) if k <= 0 or k >= V else row >= row.topk(k).values[-1]
        if p < 1:
            order = row.masked_fill(~keep, -math.inf).argsort(descending=True)
            mass = torch.cumsum(torch.where(keep, w, 0.0)[order], 0)
            edge = row[order[min(int((mass < float(torch.tensor(p)) * mass[-1] * (1 - 1e-5)).sum()), V - 1)]]
            slack = row[order[min(int((mass < float(torch.tensor(p)) * mass[-1] * (1 + 1e-5)).sum()), V - 1)]]
            assert row[tok] >= slack
            keep &= row >= edge
        assert keep[tok] or p < 1
        cum = torch.cumsum(torch.where(keep, w, 0.0), 0)
        lo, hi = (cum[tok] - w[tok]) / cum[-1], cum[tok] / cum[-1]
        assert lo - 1e-4 <= uu <= hi + 1e-4, (V, k, p, float(uu), tok)


@pytest.mark.parametrize("V", [1, 5, 301, 1024, 4096, 4099, 32000, 32768, 32769, 50257])
@pytest.mark.parametrize("k", [0, 1, 50, 512, 513, 40000])
@pytest.mark.parametrize("p", [1.0, 0.9, 0.3])
def test_draw(V, k, p):
    g = torch.Generator().manual_seed(V + k)
    x = 2 * torch.randn(7, V, generator=g)
    u = torch.tensor([0.0, 0.1, 0.37, 0.5, 0.77, 0.95, 0.9999])
    check(x, 0.8, k, p, u, draw(x, 0.8, k, p, u))


@pytest.mark.parametrize("V", [300, 8192, 40000])
@pytest.mark.parametrize("k", [0, 3, 600])
def test_ties_masks_and_non_finite(V, k):
    u = torch.tensor([0.0, 0.26, 0.51, 0.99])
    same = torch.zeros(4, V)
    got = draw(same, 1.0, k, 1.0, u)      # (values equal to the k-th are all kept)
    assert torch.all((got - u.double() * V).abs() <= 2)
    x = torch.full((4, V), -math.inf)
    x[:, [7, 9, V - 1]] = torch.tensor([1.0, 1.0, 1.0])
    assert draw(x, 1.0, k, 1.0, torch.tensor([0.1, 0.5, 0.9, 0.33])).tolist() == [7, 9, V - 1, 7]
    assert draw(x, 1.0, k, 0.0, u).tolist() == [7] * 4      # no mass asked for: the first of the largest
    assert draw(torch.full((4, V), -math.inf), 1.0, k, 0.9, u).tolist() == [0] * 4
    x = torch.randn(4, V)
    x[:, 11] = math.inf
    assert draw(x, 1.0, k, 0.9, u).tolist() == [11] * 4
    x[:, 11], x[:, 5], x[:, 20] = 50.0, math.nan, 50.0
    assert draw(x, 1.0, k, 1.0, u).tolist() == [11] * 4      # a sum that is no number: the first of the largest
    assert draw(x, 0.0, k, 1.0, u).tolist() == [11] * 4      # greedy
    y = torch.randn(4, V)
    assert draw(y, 1.0, k, 0.9, torch.full((4,), -0.5)).tolist() == y.argmax(1).tolist()      # a draw below zero: the most likely token


@pytest.mark.parametrize("V", [300, 40000])
@pytest.mark.parametrize("k,p", [(0, 1.0), (0, 0.9), (600, 1.0)])
@pytest.mark.parametrize("bits", [0x7fc00000, -0x400000, -1])
def test_every_nan_counts(V, k, p, bits):
    """Quiet NaNs of either sign, all bits set among them (the smallest value of the order that the kernel bisects in): kept, the sum is no number and the
    first of the largest is drawn; top-k leaves a NaN with the sign bit out, as the smallest value, if there are enough others."""
    x = torch.randn(4, V, generator=torch.Generator().manual_seed(V))
    x.view(torch.int32)[:, 20] = bits
    if 0 < k < V and bits < 0:
        u = torch.tensor([0.0, 0.26, 0.51, 0.99])
        clean = x.clone()
        clean[:, 20] = -math.inf
        check(clean, 1.0, k, p, u, draw(x, 1.0, k, p, u))
    else:
        assert draw(x, 1.0, k, p, torch.tensor([0.1, 0.5, 0.9, 0.33])).tolist() == x.nan_to_num(-1e9).argmax(1).tolist()


@pytest.mark.parametrize("V", [130, 4095, 4096, 4097])
@pytest.mark.parametrize("k", [128, 129])
def test_draw_of_short_rows(V, k):
    """Around the longest row of the four-wave form and the largest top-k that it lists."""
    x = 2 * torch.randn(5, V, generator=torch.Generator().manual_seed(V + k))
    u = torch.tensor([0.0, 0.1, 0.5, 0.95, 0.9999])
    check(x, 0.8, k, 0.9, u, draw(x, 0.8, k, 0.9, u))


@pytest.mark.parametrize("V", [100, 5000, 40000])
@pytest.mark.parametrize("k", [1, 50, 64, 65, 100, 128, 129])
@pytest.mark.parametrize("p", [1.0, 0.9, 0.05])
def test_few_candidates_of_few_values(V, k, p):
    """Lists around one and two a lane of a wave, with the k-th value tied and with top-p's bound inside a run of equal values."""
    g = torch.Generator().manual_seed(V + k)
    x = (torch.randn(6, V, generator=g) * 4).round() / 4
    x[1] = torch.randn(V, generator=g) * 0.01
    x[2] = -0.0
    x[3] = -x[3].abs()
    u = torch.tensor([0.0, 0.1, 0.37, 0.5, 0.95, 0.9999])
    check(x, 0.8, k, p, u, draw(x, 0.8, k, p, u))


def test_first_of_the_largest():
    for V in (5, 3000, 40000):
        x = torch.full((5, V), -math.inf)
        x[0, 0], x[1], x[2, 2:4] = math.nan, math.nan, torch.tensor([-0.0, 0.0])
        x[3, 3:] = -1.0
        want = [1, 0, 2, 3, 0]
        assert draw(x, 0.0, 0, 1.0, torch.zeros(5)).tolist() == want


def test_first_of_two_zeros():
    """Zeros of either sign are one largest value, wherever they lie: in a thread's four values, in those it reads 4096 places on, with another thread."""
    for V in (3000, 40000, 70000):
        at = [(5, 6), (8, 8 + V // 4096 * 1024), (8, V - 1), (9, 1030), (V // 2, V // 2 + 4096 if V > 8192 else V // 2 + 3)]
        x = torch.full((2 * len(at), V), -1.0)
        for i, (a, b) in enumerate(at):
            for j, (p, q) in enumerate(((-0.0, 0.0), (0.0, -0.0))):
                x[2 * i + j, a], x[2 * i + j, b] = p, q
        assert draw(x, 0.0, 0, 1.0, torch.zeros(len(x))).tolist() == [a for a, _ in at for _ in range(2)]
