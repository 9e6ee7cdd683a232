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


@pytest.mark.parametrize("L,Lk,at,lift", [(100, 100, (0, 17, 50, 99), 1e4), (33, 70, (40, 69), 1.9e4), (20, 20, (16,), 9990.0),
                                          (64, 64, (63,), 1e9), (300, 300, (299, 150), 9.93e3), (48, 48, (5, 47), float("inf"))])
@pytest.mark.parametrize("masked", [False, True])
def test_future_keys_that_their_bias_lifts_above_the_fill(gpu, L, Lk, at, lift, masked):
    """The bias is added after the causal fill, so a future key whose bias outweighs the fill has weight in every row before it, in
    whatever tile it lies; with `masked` the row's own keys lie lower still."""
    print("case f32 attention lifted keys", L, Lk, at, lift, masked, flush=True)
    from adaptivetrainingsystem_amd import ops
    B, Hq, Hkv, D = 2, 4, 2, 64
    g = torch.Generator().manual_seed(L + Lk)
    q, dout = torch.randn(B, Hq, L, D, generator=g).to(gpu), torch.randn(B, L, Hq * D, generator=g).to(gpu)
    k, v = (torch.randn(B, Hkv, Lk, D, generator=g).to(gpu) for _ in range(2))
    bias = torch.zeros(B, Lk)
    if masked:
        bias[0, : Lk // 2] = -1e4
        bias[1] = -3e3
    for j in at:
        bias[j % B, j] = lift
    bias = bias.to(gpu)
    scale = D ** -0.5
    want, state = ops.attention_f32(q, k, v, scale, key_bias=bias, return_weights=True)
    want_grads = ops.attention_f32_bwd(state, dout, B, Hq, Hkv, L, Lk, D, scale)
    out, stats = ops.attention_f32_fused(q, k, v, scale, bias)
    grads = ops.attention_f32_fused_bwd(q, k, v, out, stats, dout, scale, bias)
    # scores near 1e4 .. 2e4 are known to 1e-3 .. 2e-3 in float32 on either route (one unit in the last place); where one key has all
    # the weight, the gradients of q and k are zero up to the rounding of terms as large as dout (1.5e-6, as above)
    for a, r in zip((out, *grads), (want, *want_grads)):
        assert torch.equal(a.isnan(), r.isnan())
        assert (a - r).nan_to_num().norm() <= 4e-3 * r.nan_to_num().norm() + 1.5e-6 * dout.norm()
    assert torch.equal(ops.attention_f32(q, k, v, scale, key_bias=bias).nan_to_num(), out.nan_to_num())


def test_a_mask_value_above_one_through_the_module(gpu):
    """An attention mask holds (1 - m) * -1e4 as a bias: a value of 2 lifts its key by 1e4."""
    from types import SimpleNamespace
    from adaptivetrainingsystem_amd import ops
    from adaptivetrainingsystem_amd.layers import GroupedQueryAttention
    torch.manual_seed(2)
    att = GroupedQueryAttention(SimpleNamespace(hidden_size=256, num_heads=4, num_kv_heads=2, seq_length=128)).to(gpu).eval()
    x, mask = torch.randn(2, 80, 256, device=gpu), torch.ones(2, 80, device=gpu)
    mask[:, 70] = 2.0
    with torch.no_grad():
        got = att(x, mask)
        cos, sin = att.rope(80, x.device)
        q, k, v = (ops.linear_nt(x.view(160, 256), p.weight).view(2, 80, -1, 64).transpose(1, 2) for p in (att.q_proj, att.k_proj, att.v_proj))
        q, k = ops.rope(q, k, cos, sin)
        a, _ = ops.attention_f32(q, k, v.contiguous(), 0.125, key_bias=(1.0 - mask) * -1e4, return_weights=True)
        want = ops.linear_nt(a.view(160, 256), att.o_proj.weight).view_as(got)
    assert (got - want).norm() <= 4e-3 * want.norm()


def test_the_scale_may_be_left_to_the_head_dim_and_saved_tensors_may_come_back_elsewhere(gpu):
    from adaptivetrainingsystem_amd.autograd import AttentionF32Function
    g = torch.Generator().manual_seed(9)
    q, k, v = (torch.randn(2, h, 20, 64, generator=g).to(gpu).requires_grad_() for h in (4, 2, 2))
    dout = torch.randn(2, 20, 256, generator=g).to(gpu)
    want = torch.autograd.grad(AttentionF32Function.apply(q, k, v, 0.125), (q, k, v), dout)

    def unpack(t):      # the same numbers behind another stride and alignment
        room = torch.empty(t.numel() + 1, device=gpu)[1:]
        return room.view(t.shape[::-1]).permute(*range(t.dim() - 1, -1, -1)).copy_(t)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        out = AttentionF32Function.apply(q, k, v, None)
    for a, b in zip(torch.autograd.grad(out, (q, k, v), dout), want):
        assert torch.equal(a, b)


# heads that divide by the XCDs (their tiles keep to one) and heads that do not, odd numbers of tiles
@pytest.mark.parametrize("B,Hq,Hkv,L,Lk,D", [(1, 8, 8, 40, 40, 64), (2, 12, 4, 100, 133, 64), (3, 16, 8, 17, 300, 128), (1, 24, 8, 257, 257, 128), (1, 9, 3, 65, 65, 64)])
def test_a_head_has_the_same_bits_alone(gpu, B, Hq, Hkv, L, Lk, D):
    from adaptivetrainingsystem_amd import ops
    print("case f32 heads", B, Hq, Hkv, L, Lk, D, flush=True)
    g = torch.Generator().manual_seed(L + Hq)
    q, k, v = (torch.randn(B, h, n, D, generator=g).to(gpu) for h, n in ((Hq, L), (Hkv, Lk), (Hkv, Lk)))
    dout, rep = torch.randn(B, L, Hq * D, generator=g).to(gpu), Hq // Hkv
    out, stats = ops.attention_f32_fused(q, k, v, None, None)
    grads = ops.attention_f32_fused_bwd(q, k, v, out, stats, dout, None, None)
    for b in range(B):
        for h in range(Hkv):
            heads, cols = slice(h * rep, (h + 1) * rep), slice(h * rep * D, (h + 1) * rep * D)
            one = [t[b:b + 1, s].contiguous() for t, s in ((q, heads), (k, slice(h, h + 1)), (v, slice(h, h + 1)))]
            o, st = ops.attention_f32_fused(*one, None, None)
            assert torch.equal(o, out[b:b + 1, :, cols])
            got = ops.attention_f32_fused_bwd(*one, o, st, dout[b:b + 1, :, cols].contiguous(), None, None)
            for t, whole, s in zip(got, grads, (heads, slice(h, h + 1), slice(h, h + 1))):
                assert torch.equal(t, whole[b:b + 1, s])
