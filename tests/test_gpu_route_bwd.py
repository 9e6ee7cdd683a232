"""Gradients of the routing rule for up to 8 experts, and the router's own gradients at batches of a few tokens per chunk."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,k", [(1, 8, 2), (63, 8, 8), (64, 5, 2), (65, 2, 1), (513, 8, 3), (100, 1, 1), (70, 9, 2)])
@pytest.mark.parametrize("mode", [0, 1])
def test_route_gradient_few_experts(gpu, T, E, k, mode):
    print("case route bwd", T, E, k, mode, flush=True)
    from adaptivetrainingsystem_amd import ops
    g = torch.Generator().manual_seed(T + E)
    z, usage, tau, lam = torch.randn(T, E, generator=g).double().requires_grad_(), torch.rand(E, generator=g).double(), 0.7, 0.3
    dw = torch.randn(T, k, generator=g)
    if mode == 0:
        p = torch.softmax(z / tau, -1)
        w, idx = torch.topk(p, k, -1)
        w = w / (w.sum(-1, keepdim=True) + 1e-9)
    else:
        v, idx = torch.topk(z, k, -1)
        w = torch.softmax(v / tau, -1)
    ((w * dw).sum() + lam * (torch.softmax(z, -1) * usage).sum()).backward()
    to = lambda t: t.detach().float().to(gpu)
    out = ops.route_bwd(to(z), idx.int().to(gpu), to(w), dw.to(gpu), tau, mode, logits_aux=to(z), usage=to(usage), aux_scale=lam,
                        aux_scale_dev=torch.ones(1, device=gpu))
    # float32: a few roundings of terms of the size of dw / tau
    assert (out.cpu().double() - z.grad).abs().max() <= 4e-6 * (dw.abs().max().item() / tau + 1)


# both ends of what each instance holds
@pytest.mark.parametrize("T,E,k", [(65, 1, 1), (129, 2, 2), (64, 3, 1), (200, 3, 3), (63, 4, 2), (65, 4, 4), (64, 5, 5)])
@pytest.mark.parametrize("mode", [0, 1])
def test_route_gradient_of_each_instance(gpu, T, E, k, mode):
    test_route_gradient_few_experts(gpu, T, E, k, mode)


@pytest.mark.parametrize("T,E,H,dtype", [(256, 8, 512, torch.float32), (257, 8, 4096, torch.bfloat16), (9, 3, 72, torch.float32),
                                         (1000, 64, 2048, torch.bfloat16), (5000, 8, 264, torch.bfloat16)])
def test_router_gradients_small_chunks(gpu, T, E, H, dtype):
    print("case router bwd", T, E, H, dtype, flush=True)
    from adaptivetrainingsystem_amd import ops
    g = torch.Generator().manual_seed(T)
    dz = torch.randn(T, E, generator=g)
    x, wg, base = (torch.randn(*s, generator=g).to(dtype) for s in ((T, H), (E, H), (T, H)))
    dx, dw = ops.router_bwd(dz.to(gpu), x.to(gpu), wg.to(gpu), base=base.to(gpu))
    ref_dx, ref_dw = base.double() + dz.double() @ wg.double(), dz.double().T @ x.double()
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23
    # float32 sums of E (T) products; dx is rounded once to its own type
    assert ((dx.cpu().double() - ref_dx).abs() <= eps * ref_dx.abs() + 2e-7 * E * 16).all()
    assert (dw.cpu().double() - ref_dw).norm() <= 2e-6 * ref_dw.norm()
