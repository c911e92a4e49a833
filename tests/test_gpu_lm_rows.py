"""The tied lm_head at row counts around its fragments, and the final norm of the rows whose logits are wanted."""
import pytest
import torch

from vllm_i64_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("N,K", [(1, 32), (65, 288), (130, 1024), (63, 544), (200, 2080)])
@pytest.mark.parametrize("M", [1, 15, 16, 17, 31, 32, 33, 64, 65, 130])
def test_row_counts(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M * N + K)
    a, b = torch.randn(M, K, generator=g, device=DEV), torch.randn(N, K, generator=g, device=DEV)
    out = torch.full((M, N), float("nan"), device=DEV)
    ops.lm_head(a, b, out=out, workspace=torch.full((ops.lm_head_workspace_bytes(M, K),), 255, dtype=torch.uint8, device=DEV))
    ref = a.double() @ b.double().T
    # products exact to 2^-24 of the leading one, 32-bit sums of K of them
    assert ((out.double() - ref).abs() <= 2.0 ** -21 * (a.double().abs() @ b.double().abs().T)).all()


@pytest.mark.parametrize("moe", [False, True])
@pytest.mark.parametrize("n,H,wanted", [(1, 64, [0]), (5, 1024, [4, 0, 4]), (300, 96, [299, 7, 150]), (2500, 1024, list(range(0, 2500, 39)))])
def test_final_norm_of_wanted_rows(n, H, wanted, moe):
    g = torch.Generator(device=DEV).manual_seed(n + H)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)
    h, w, emb = r(n, H), r(H), r(70, H)
    rows = torch.tensor(wanted, dtype=torch.int32, device=DEV)
    kw = dict(add=r(n, H))
    if moe:
        inv = torch.randperm(2 * n, generator=g, device=DEV).to(torch.int32)
        kw = dict(moe_rows=r(2 * n, H), moe_inv=inv, moe_shared=r(n, H), route_weights=[0.7, 0.3], routed_scale=0.9, shared_scale=1.1)
    _, normed = ops.fused_residual_norm(h, w, 1e-6, **kw)
    M = len(wanted)
    ws = lambda: torch.zeros(ops.lm_head_workspace_bytes(M, H), dtype=torch.uint8, device=DEV)
    want = ops.lm_head(normed, emb, a_rows=rows, workspace=ws())
    planes, held, got = ws(), h.clone(), torch.empty(M, 70, device=DEV)
    ops.fused_residual_norm_lm_rows(h, w, 1e-6, rows, planes, **kw)
    ops.lm_head_planes(planes, emb, got)
    assert torch.equal(h, held) and torch.allclose(got, want, rtol=1e-5, atol=1e-5 * want.abs().max().item())      # (a row's squares may be summed in another order)
