"""The stacked projection of a training step: rotation between any layouts, weight gradients in K slices."""
import pytest
import torch

from tests.test_gpu_parity import BF16_TOL, F32_TOL, rel_err, same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L,nh,nkv,D", [(1, 1, 2, 1, 64), (2, 67, 4, 2, 128), (3, 130, 5, 5, 36)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("inverse", [False, True])
def test_rope_strided(gpu, B, L, nh, nkv, D, dtype, inverse):
    print("case rope strided", B, L, nh, nkv, D, dtype, inverse, flush=True)
    from adaptivetrainingsystem_amd import ops
    g = torch.Generator().manual_seed(7)
    cos, sin = ops.rope_table(L, D)
    n = nh + 2 * nkv
    y = torch.randn(B, L, n, D, generator=g).to(dtype).to(gpu).transpose(1, 2)
    q, k, v = y[:, :nh], y[:, nh:nh + nkv], y[:, nh + nkv:]
    if inverse:      # contiguous gradients into the projection's layout
        q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
        buf = torch.full((B, L, n, D), 7.0, dtype=dtype, device=gpu)
        o = buf.transpose(1, 2)
        outs = (o[:, :nh], o[:, nh:nh + nkv], o[:, nh + nkv:])
    else:
        outs = tuple(torch.full((B, h, L, D), 7.0, dtype=dtype, device=gpu) for h in (nh, nkv, nkv))
    ops.rope_strided((q, k, v), outs, cos, sin, inverse=inverse)
    rq, rk = ops.rope(q, k, cos, sin, inverse=inverse)
    assert same_bits(outs[0].contiguous(), rq) and same_bits(outs[1].contiguous(), rk) and same_bits(outs[2].contiguous(), v.contiguous())
    only = torch.empty_like(rk)
    ops.rope_strided((None, k, None), (None, only, None), cos, sin, inverse=inverse)
    assert same_bits(only, rk)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rope_gradient_keeps_the_layout_of_its_input(gpu, dtype):
    from adaptivetrainingsystem_amd import apply_rotary_pos_emb, ops
    g = torch.Generator().manual_seed(8)
    cos, sin = ops.rope_table(33, 64)
    q, k = (torch.randn(2, 33, h, 64, generator=g).to(dtype).to(gpu).requires_grad_() for h in (4, 2))
    dq, dk = (torch.randn(2, h, 33, 64, generator=g).to(dtype).to(gpu) for h in (4, 2))
    torch.autograd.backward(apply_rotary_pos_emb(q.transpose(1, 2), k.transpose(1, 2), cos, sin), (dq, dk))
    rq, rk = ops.rope(dq, dk, cos, sin, inverse=True)
    assert same_bits(q.grad, rq.transpose(1, 2).contiguous()) and same_bits(k.grad, rk.transpose(1, 2).contiguous())
    assert q.grad.is_contiguous()


@pytest.mark.parametrize("rows", [1, 64, 511, 1024, 4000, 8191])
@pytest.mark.parametrize("M,N", [(256, 256), (264, 1032), (1024, 2048)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_weight_gradient_in_slices(gpu, rows, M, N, dtype):
    print("case wgrad", rows, M, N, dtype, flush=True)
    from adaptivetrainingsystem_amd import ops
    g = torch.Generator(device=gpu).manual_seed(9)
    dy, x = (torch.randn(rows, c, generator=g, device=gpu).to(dtype) for c in (M, N))
    start, count = ops._single_group(rows, dy.device)
    dyT, xT = (ops.transpose_grouped_rows(t, start, count, rows) for t in (dy, x))
    ref = dy.double().T.cpu() @ x.double().cpu()
    assert rel_err(ops.wgrad_dense(dyT, xT, rows), ref) <= (F32_TOL if dtype == torch.float32 else BF16_TOL)
    assert 1 <= ops.wgrad_slices(M, N, rows) <= max(1, rows // 512 + 1)


@pytest.mark.parametrize("H,nh,nkv,B,L", [(256, 4, 2, 2, 33), (512, 4, 4, 1, 300)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("frozen", ["", "q", "kv", "x"])
def test_projection_gradients(gpu, H, nh, nkv, B, L, dtype, frozen):
    """Against three linear layers in float64, with parameters that want no gradient."""
    print("case projection", H, nh, nkv, B, L, dtype, frozen, flush=True)
    from adaptivetrainingsystem_amd import autograd as ag
    from adaptivetrainingsystem_amd import ops
    D, g = H // nh, torch.Generator().manual_seed(10)
    cos, sin = ops.rope_table(L, D)
    x = torch.randn(B * L, H, generator=g).to(dtype)
    ws = [(torch.randn(h * D, H, generator=g) * 0.05).to(dtype) for h in (nh, nkv, nkv)]
    ds = [torch.randn(B, h, L, D, generator=g).to(dtype) for h in (nh, nkv, nkv)]
    want = [t not in frozen or not frozen for t in "xqkv"]
    leaf = [t.to(gpu).requires_grad_(w) for t, w in zip([x] + ws, want)]
    outs = ag.QKVRoPEFunction.apply(*leaf, cos, sin, B, L, D)
    torch.autograd.backward(outs, [d.to(gpu) for d in ds])
    ref = [t.double().requires_grad_(w) for t, w in zip([x] + ws, want)]
    c, s = (t.double().cpu()[:L] for t in (cos, sin))
    rot = lambda t: t * c + torch.cat([-t[..., D // 2:], t[..., :D // 2]], -1) * s
    r = [(ref[0] @ w.T).view(B, L, -1, D).transpose(1, 2) for w in ref[1:]]
    r = [rot(r[0]), rot(r[1]), r[2]]
    torch.autograd.backward(r, [d.double() for d in ds])
    # gradients contract over intermediates rounded to the type (dy after the rotation): twice the product's bound
    tol = F32_TOL if dtype == torch.float32 else BF16_TOL
    for a, b in zip(outs, r):
        assert rel_err(a, b) <= 2 * tol
    for a, b, w in zip(leaf, ref, want):
        assert (a.grad is not None) == w
        if w:
            assert rel_err(a.grad, b.grad) <= 2 * tol
