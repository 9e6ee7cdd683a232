"""Routing passes whose workgroup has 16 waves, gate products with an expert tile per workgroup, dispatch plans of 16 waves."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# tokens around one pass of four waves, one and several passes of sixteen; experts that fill a wave or part of one, and more
@pytest.mark.parametrize("T,E,k", [(4, 64, 6), (5, 64, 6), (17, 64, 16), (64, 64, 6), (64, 33, 5), (33, 8, 2), (512, 8, 2),
                                   (129, 16, 4), (65, 32, 3), (16, 128, 8), (16, 129, 8)])
@pytest.mark.parametrize("variant", [0, 1])
def test_route_topk_ties_and_sums(gpu, T, E, k, variant):
    print("case route waves", T, E, k, variant, flush=True)
    from adaptivetrainingsystem_amd import ops
    from oracle import sparse_layer_oracle as O
    g = torch.Generator().manual_seed(T * E)
    logits = torch.randint(-6, 7, (T, E), generator=g).float() / 2        # many equal values, zeros of both signs
    logits[::2][logits[::2] == 0] = -0.0
    r = ops.route_topk(logits.to(gpu), k, 1.0, variant)
    order = torch.sort(logits, dim=1, descending=True, stable=True).indices[:, :k]      # the lower id first among equals
    assert torch.equal(r["indices"].cpu().long(), order)
    z = logits.double()
    p = torch.softmax(z, 1)
    w = p.gather(1, order)
    w = w / (w.sum(1, keepdim=True) + 1e-9) if variant == 0 else torch.softmax(z.gather(1, order), 1)
    # an exponential, a sum of up to 128 terms and two divisions in float32: a few units of 6e-8 each
    assert (r["weights"].cpu().double() - w).abs().max() <= 1e-6 * w.max()
    assert torch.equal(r["hist"].cpu(), torch.bincount(order.flatten(), minlength=E).int())
    assert (r["prob_colsum"].cpu().double() - p.sum(0)).abs().max() <= 1e-6 * max(1.0, float(p.sum(0).max()))
    aux = O.aux_loss(logits, order, E, 0.01)
    assert abs(float(r["aux"].cpu()) - float(aux)) <= 1e-6


@pytest.mark.parametrize("n,k,E,C", [(256, 2, 8, 40), (258, 6, 64, 3), (1024, 2, 8, 100), (1020, 6, 64, 16), (1024, 4, 128, 5),
                                     (1024, 4, 129, 5)])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_dispatch_plan_waves(gpu, n, k, E, C, dtype):
    print("case plan waves", n, k, E, C, flush=True)
    from adaptivetrainingsystem_amd import ops
    from oracle import sparse_layer_oracle as O
    g = torch.Generator().manual_seed(n + E)
    idx = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(n // k)]) % max(1, E - 1)
    _, token_map = O.dispatch_loop(torch.zeros(n // k, 1), idx, E, C)
    plan = ops.dispatch_plan(idx.to(gpu, dtype), E, C)
    assert torch.equal(plan["token_map"].cpu(), token_map)
    hist = torch.bincount(idx.flatten(), minlength=E)
    assert torch.equal(plan["hist"].cpu().long(), hist) and torch.equal(plan["kept"].cpu().long(), hist.clamp(max=C))
    offsets = torch.cat([torch.zeros(1, dtype=torch.long), hist.clamp(max=C).cumsum(0)])
    assert torch.equal(plan["offsets"].cpu().long(), offsets)
    row_of = torch.full((n,), -1, dtype=torch.int32)
    for e in range(E):
        m = token_map[e][token_map[e] >= 0].long()
        row_of[m] = torch.arange(int(offsets[e]), int(offsets[e]) + len(m), dtype=torch.int32)
    assert torch.equal(plan["row_of"].cpu(), row_of) and int(plan["status"].cpu()) == 0


@pytest.mark.parametrize("T,H,E", [(1, 2048, 64), (17, 200, 33), (1024, 520, 64), (1025, 520, 64), (3, 128, 128)])
def test_router_logits_tiles(gpu, T, H, E):
    print("case gate tiles", T, H, E, flush=True)
    from adaptivetrainingsystem_amd import ops
    g = torch.Generator().manual_seed(T + E)
    x, w = torch.randn(T, H, generator=g).bfloat16(), (torch.randn(E, H, generator=g) * 0.05).bfloat16()
    bias = torch.randn(E, generator=g)
    out = ops.router_logits(x.to(gpu), w.to(gpu), bias.to(gpu)).cpu().double()
    ref = x.double() @ w.double().T + bias.double()
    # float32 sums of H exact products: sqrt(H) roundings of 6e-8 of a running sum
    scale = (x.double().abs() @ w.double().abs().T).max()
    assert (out - ref).abs().max() <= 1e-6 * scale
    # a token's logits do not depend on the batch that it is in
    big = torch.cat([x, torch.randn(2000, H, generator=g).bfloat16()]).to(gpu)
    assert torch.equal(ops.router_logits(big, w.to(gpu), bias.to(gpu)).cpu()[:T].double(), out)
