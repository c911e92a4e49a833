"""The delta rule's unit vectors and gates: heads on 16 lanes (16-byte rows) and on a wave (any row), sizes at the edges of the stripes and rounds."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,G,d", [(4, 4, 64), (16, 16, 128), (6, 3, 4), (20, 20, 68), (34, 17, 132), (2, 1, 256), (3, 3, 260), (3, 3, 50)])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("unit", [True, False])
def test_unit_vectors(heads, G, d, shift, unit):
    """The factor is one over the root of a sum of `d` squares in 32 bits: a few units in the last place of it, and one of the product."""
    from vllm_i64_amd import ops_dense as D
    dev, n = torch.device("cuda:0"), 5
    g = torch.Generator().manual_seed(heads + d)
    ld = shift + 2 * G * d + 8
    ld += (-ld) % 4
    X, R = torch.randn(n, ld, generator=g), torch.randn(n, heads, generator=g)
    Xd, Gt = X.to(dev), torch.full((n, 2 * heads), 9.0, device=dev)
    D.gdn_gates(Xd, Gt, R.to(dev), q_off=shift, k_off=shift + G * d, v_off=0, heads=heads, kv_heads=G, dim=d, vdim=1, b_off=0, a_off=-1, a_log=None, dt_bias=None,
                unit_eps=1e-6 if unit else -1.0, q_scale=0.25, n=n)
    want = X.double().clone()
    x = want[:, shift:shift + 2 * G * d].view(n, 2 * G, d)
    if unit:
        x /= (x.pow(2).sum(-1, keepdim=True) + 1e-6).sqrt()
    x[:, :G] *= 0.25
    assert float((Xd.cpu().double() - want).abs().max() / want.abs().max()) < 1e-6
    assert torch.equal(Xd.cpu()[:, :shift], X[:, :shift]) and torch.equal(Xd.cpu()[:, shift + 2 * G * d:], X[:, shift + 2 * G * d:])
    assert float((Gt.cpu()[:, :heads] - torch.sigmoid(R)).abs().max()) < 1e-6
