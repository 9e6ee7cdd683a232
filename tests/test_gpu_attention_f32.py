"""Float32 attention without materialised scores: against the formula in float64 and against the materialised route."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(q, k, v, dout, bias, scale):
    """Output and gradients in float64 through autograd, with the reference's fill of -1e4."""
    q, k, v = (t.double().requires_grad_() for t in (q, k, v))
    B, Hq, L, D = q.shape
    Lk, rep = k.shape[2], Hq // k.shape[1]
    s = (q @ k.repeat_interleave(rep, 1).transpose(-1, -2)) * scale
    future = torch.arange(Lk)[None, :] > torch.arange(L)[:, None] + (Lk - L)
    s = s.masked_fill(future, -1e4)
    if bias is not None:
        s = s + bias.double()[:, None, None, :]
    out = (torch.softmax(s, -1) @ v.repeat_interleave(rep, 1)).transpose(1, 2).reshape(B, L, Hq * D)
    out.backward(dout.double())
    return out.detach(), q.grad, k.grad, v.grad


# around tiles of 16 rows and keys, one row, fewer tiles than waves, keys before the first query, grouped heads
SIZES = [(1, 1, 1, 1, 1, 64), (1, 2, 1, 15, 15, 128), (2, 4, 2, 16, 16, 64), (2, 4, 2, 17, 33, 128), (1, 6, 2, 65, 65, 128),
         (3, 4, 4, 130, 200, 64), (1, 4, 2, 257, 257, 128), (1, 8, 1, 48, 511, 64)]


@pytest.mark.parametrize("B,Hq,Hkv,L,Lk,D", SIZES)
@pytest.mark.parametrize("masked", [False, True])
def test_fused_f32_attention(gpu, B, Hq, Hkv, L, Lk, D, masked):
    print("case f32 attention", B, Hq, Hkv, L, Lk, D, masked, flush=True)
    from adaptivetrainingsystem_amd import ops
    g = torch.Generator().manual_seed(L * 7 + Lk)
    q, k, v, dout = (torch.randn(*s, generator=g) for s in ((B, Hq, L, D), (B, Hkv, Lk, D), (B, Hkv, Lk, D), (B, L, Hq * D)))
    # (padding in front: the first rows see only masked keys, which share their weight with the future ones)
    bias = torch.zeros(B, Lk) if masked else None
    if masked:
        bias[:, 1:max(2, Lk // 3)] = -1e4
    G = [t.to(gpu) for t in (q, k, v)]
    kb = None if bias is None else bias.to(gpu)
    scale = D ** -0.5
    assert ops.attention_f32_fused_supported(*G, None, 0.0)
    out, stats = ops.attention_f32_fused(*G, scale, kb)
    grads = ops.attention_f32_fused_bwd(*G, out, stats, dout.to(gpu), scale, kb)
    # float32 sums of D and of Lk products against float64: a few units of 6e-8 times the square root of their number;
    # the materialised route measures 3e-7 at these sizes.  (A gradient of q or k is a difference of terms as large as dout.v
    # times k: with one key it is zero up to the rounding of those.)
    for a, r in zip((out, *grads), _reference(q, k, v, dout, bias, scale)):
        assert (a.cpu().double() - r).norm() <= 1.5e-6 * torch.maximum(r.norm(), dout.double().norm())
    # the inference entry point takes the same kernel
    assert torch.equal(ops.attention_f32(*G, key_bias=kb), out)


@pytest.mark.parametrize("shift", [0, 1])
def test_rows_whose_scores_lie_below_the_fill(gpu, shift):
    """All visible keys of the first rows are masked as deep as the causal fill (or deeper): the weights spread over the
    future keys as well, as the materialised softmax spreads them, and the gradients with them."""
    print("case f32 attention fill", shift, flush=True)
    from adaptivetrainingsystem_amd import ops
    B, Hq, Hkv, L, D = 2, 4, 2, 100, 64
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(B, h, L, D, generator=g).to(gpu) for h in (Hq, Hkv, Hkv))
    dout = torch.randn(B, L, Hq * D, generator=g).to(gpu)
    bias = torch.zeros(B, L)
    bias[:, :40] = -1e4 - shift
    bias = bias.to(gpu)
    scale = D ** -0.5
    want, state = ops.attention_f32(q, k, v, scale, key_bias=bias, return_weights=True)
    want_grads = ops.attention_f32_bwd(state, dout, B, Hq, Hkv, L, L, D, scale)
    out, stats = ops.attention_f32_fused(q, k, v, scale, bias)
    grads = ops.attention_f32_fused_bwd(q, k, v, out, stats, dout, scale, bias)
    # scores near 1e4 are known to 1e-3 in float32 on either route (one unit in the last place)
    for a, r in zip((out, *grads), (want, *want_grads)):
        assert (a - r).norm() <= 4e-3 * r.norm()


def test_routes_that_stay_materialised(gpu):
    from adaptivetrainingsystem_amd import ops
    t = torch.zeros(1, 2, 8, 64, device=gpu)
    assert not ops.attention_f32_fused_supported(t, t, t, torch.zeros(1, 8, 8, device=gpu), 0.0)
    assert not ops.attention_f32_fused_supported(t, t, t, None, 0.1)
    assert not ops.attention_f32_fused_supported(t[..., :32].contiguous(), t, t, None, 0.0)
    assert not ops.attention_f32_fused_supported(t.transpose(1, 2), t, t, None, 0.0)
