"""The gate / up epilogues over the whole range of a gate: its ends, infinities and NaN, in every form that multiplies out a gate."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

# (exact in bf16; around -87.3 the reciprocal of 1 + e^-z leaves the normal numbers, around -88.7 e^-z the range)
GATES = [0.0, -0.0, 1e-30, -1e-30, 0.5, -3.0, 20.0, -20.0, 86.0, -86.0, -86.5, 87.0, -87.0, -87.5, 88.0, -88.0, -88.5, 89.0, -89.0, -90.0, 104.0, -104.0, 1e4, -1e4, 2.0 ** 100, -(2.0 ** 100), 2.0 ** 127, -(2.0 ** 127),
         math.inf, -math.inf, math.nan]
BOUND = 2.0 ** 126
UPS = [1.0, -0.75, 2.0 ** 20]


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


@pytest.mark.parametrize("arith", ["rounded", "bf16", "exact"])
@pytest.mark.parametrize("rows", [1, 3, 5, 33, 100])
@pytest.mark.parametrize("epilogue", ["silu", "clamp"])
def test_ends_of_the_gate(dev, arith, rows, epilogue):
    """One weight column holds the gate, another the up value, and a row of ones and zeros asks for them: products are exact.  A gated result is as close to 64 bits as two roundings of
    the quotient and one of the product leave it, down to where it is below the normal numbers; what overflows in e^-z is zero; infinities and NaN are those of z / (1 + e^-z)."""
    from vllm_i64_amd import ops_dense as D
    K = 64
    z = torch.tensor([g for g in GATES for _ in UPS])
    u = torch.tensor(UPS * len(GATES))
    N = z.numel()
    w = torch.zeros(2 * N, K)
    w[:N, 0], w[N:, 0] = z, u      # (every other column zero: nothing but a number meets a row's zeros)
    a = torch.zeros(rows, K)
    a[:, 0] = 1.0
    w, a = w.bfloat16().to(dev), a.to(dev)
    kw = dict(epilogue=D.EPI_SILU_MUL) if epilogue == "silu" else dict(epilogue=D.EPI_CLAMP_GLU, act_a=1.0, act_b=BOUND)
    out = torch.full((rows, N), 7.0, device=dev)
    if arith == "rounded":
        D.linear(None, w, out, n=N, a16=a.bfloat16(), **kw)
    else:
        D.linear(a, w, out, n=N, exact=arith == "exact", **kw)
    assert torch.equal(out[:1].expand_as(out).nan_to_num(0.25), out.nan_to_num(0.25))
    got = out[0].double().cpu()
    z, u = z.bfloat16().double(), u.double()
    if epilogue == "clamp":
        z, u = z.nan_to_num(BOUND, math.inf, -math.inf).clamp(max=BOUND), u + 1.0      # (the bound takes the place of NaN)
    want = torch.where(z < -88.7228, torch.zeros_like(z), z / (1.0 + torch.exp(-z)))
    want = torch.where(z == -math.inf, torch.full_like(z, math.nan), want) * u
    finite = want.isfinite() & (want.abs() < 3.4e38)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got[~finite].nan_to_num(0.5, math.inf, -math.inf), torch.where(want.abs() >= 3.4e38, want.sign() * math.inf, want)[~finite].nan_to_num(0.5, math.inf, -math.inf))
    off = (got - want).abs()[finite]
    # 1 + e^-z, the quotient and the product by up: 3 roundings of 2^-24, e^-z itself good to four of them
    assert bool((off <= 2.0 ** -21 * want.abs()[finite] + 2.0 ** -149).all()), [(float(a), float(b), float(c)) for a, b, c in zip(z[finite], got[finite], want[finite]) if abs(b - c) > 2.0 ** -21 * abs(c) + 2.0 ** -149]
