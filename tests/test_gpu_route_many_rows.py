"""The router's own products in launches of many rows (a wave a row): entries in eights, a last one that goes with the eight before it, the gate's row
behind them, widths that 16-byte loads can and cannot read."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("entries", [3, 7, 8, 9, 16, 17, 24, 32])
@pytest.mark.parametrize("gate", [False, True])
@pytest.mark.parametrize("K", [36, 256, 260, 1024, 67])
def test_products_of_many_rows(entries, gate, K):
    from vllm_i64_amd import ops_dense as D
    dev, n, top = torch.device("cuda:0"), 515, 2      # (more rows than the form that splits a row takes)
    g = torch.Generator().manual_seed(entries * K)
    h, w = torch.randn(n, K, generator=g), (torch.randn(entries + int(gate), K, generator=g) * K ** -0.5).to(torch.bfloat16)
    idx, wgt = torch.full((n, top), -1, dtype=torch.int32, device=dev), torch.empty(n, top, device=dev)
    go = torch.full((n,), 9.0, device=dev) if gate else None
    D.route_topk(None, entries=entries, correction=None, groups=1, keep=1, top=top, scale=1.0, idx=idx, wgt=wgt, n=n, h=h.to(dev), w=w.to(dev), gate_out=go, sigmoid_scores=True,
                 raw_weights=True)
    z = h.double() @ w.double().T
    picked = z[:, :entries].gather(1, idx.cpu().long())
    best = z[:, :entries].topk(top).values
    # products of 32-bit values by bf16 ones, summed in 32 bits: K roundings of 2^-24 at the outside
    tol = (K + 8) * 2.0 ** -24 * 4
    assert float((picked - best).abs().max()) < tol and bool((idx[:, 0] != idx[:, 1]).all())
    assert float((wgt.cpu().double() - torch.sigmoid(picked)).abs().max()) < tol + 1e-6
    if gate:
        assert float((go.cpu().double() - torch.sigmoid(z[:, entries])).abs().max()) < tol + 1e-6
