"""The compiled host side of the short calls against the general path, over the forms that it takes and those that it hands
on; its autograd nodes under hooks, checkpointing, threads, transforms and errors."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


class _Nothing:
    """A host side that takes no call: everything goes the general way."""

    def __getattr__(self, name):
        return lambda *a, **k: None


@pytest.fixture
def general(monkeypatch):
    from adaptivetrainingsystem_amd import _lib, layers

    def run(fn):
        with monkeypatch.context() as m:
            m.setattr(_lib, "native", lambda: _Nothing())
            m.setattr(layers, "native", lambda: _Nothing())
            return fn()
    return run


def _same(a, b):
    a, b = (x if isinstance(x, (tuple, list)) else (x,) for x in (a, b))
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert (x is None) == (y is None)
        if x is not None:
            assert x.shape == y.shape and x.dtype == y.dtype and x.stride() == y.stride() and torch.equal(x, y)


@pytest.mark.parametrize("shape,order", [((1, 1, 8), 0), ((3, 5, 1000), 0), ((2, 33, 512), 1), ((7, 72), 0), ((2, 0, 64), 0)])
@pytest.mark.parametrize("dtype,wdtype", [(torch.bfloat16, torch.float32), (torch.bfloat16, torch.bfloat16),
                                          (torch.float32, torch.float32), (torch.float16, torch.float32)])
@pytest.mark.parametrize("needs", [(False, False), (True, True), (True, False), (False, True)])
def test_norm_equals_the_general_path(gpu, general, shape, order, dtype, wdtype, needs):
    from adaptivetrainingsystem_amd import FusedRMSNorm, RMSNorm
    g = torch.Generator().manual_seed(3)
    base = torch.randn(*shape, generator=g).to(dtype).to(gpu)
    if order:                          # rows that are not contiguous
        base = base.transpose(0, 1).contiguous().transpose(0, 1)
    weight = (1 + torch.randn(shape[-1], generator=g) * 0.1).to(wdtype).to(gpu)
    dy = torch.randn(*shape, generator=g).to(dtype).to(gpu)
    for cls in (RMSNorm, FusedRMSNorm):
        def run():
            norm = cls(shape[-1]).to(gpu)
            norm.weight = torch.nn.Parameter(weight.clone(), requires_grad=needs[1])
            x = base.detach().requires_grad_(needs[0])
            y = norm(x)
            if not any(needs):
                assert not y.requires_grad
                return y
            y.backward(dy)
            return y.detach(), x.grad, norm.weight.grad
        _same(run(), general(run))


@pytest.mark.parametrize("layout", ["heads", "positions", "padded", "reversed"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,Hq,Hkv,L,D", [(1, 1, 1, 1, 64), (2, 6, 2, 17, 128), (3, 4, 4, 5, 80)])
@pytest.mark.parametrize("grad", [False, True])
def test_rotation_equals_the_general_path(gpu, general, layout, dtype, B, Hq, Hkv, L, D, grad):
    from adaptivetrainingsystem_amd import FusedRoPE, RotaryEmbedding, apply_rotary_pos_emb
    g = torch.Generator().manual_seed(4)

    def make(h):
        if layout == "heads":
            return torch.randn(B, h, L, D, generator=g).to(dtype).to(gpu)
        if layout == "positions":
            return torch.randn(B, L, h, D, generator=g).to(dtype).to(gpu).transpose(1, 2)
        if layout == "padded":
            return torch.randn(B, h, L, D + 16, generator=g).to(dtype).to(gpu)[..., :D]
        return torch.randn(D, L, h, B, generator=g).to(dtype).to(gpu).permute(3, 2, 1, 0)
    q0, k0 = make(Hq), make(Hkv)
    dq, dk = (torch.randn(B, h, L, D, generator=g).to(dtype).to(gpu) for h in (Hq, Hkv))
    rope, fused = RotaryEmbedding(D, 64), FusedRoPE(D, 64)

    def run():
        out = []
        for fn in (lambda a, b: apply_rotary_pos_emb(a, b, *rope(L, q0.device)), lambda a, b: fused(a, b, 3)):
            q, k = (t.detach().requires_grad_(grad) for t in (q0, k0))
            r = fn(q, k)
            out += [t.detach() for t in r]
            if grad:
                torch.autograd.backward(list(r), [dq, dk])
                out += [q.grad, k.grad]
        return out
    _same(run(), general(run))


@pytest.mark.parametrize("B,L,steps,mask", [(1, 1, 0, False), (3, 33, 2, False), (40, 2, 1, False), (2, 70, 1, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_attention_sub_layer_equals_the_general_path(gpu, general, B, L, steps, mask, dtype):
    from types import SimpleNamespace
    from adaptivetrainingsystem_amd.layers import GroupedQueryAttention
    torch.manual_seed(1)
    att = GroupedQueryAttention(SimpleNamespace(hidden_size=256, num_heads=4, num_kv_heads=2, seq_length=128)).to(gpu).to(dtype).eval()
    x = torch.randn(B, L, 256, device=gpu, dtype=dtype)
    more = [torch.randn(B, 1, 256, device=gpu, dtype=dtype) for _ in range(steps)]
    m = torch.ones(B, L, device=gpu) if mask else None

    def run():
        with torch.no_grad():
            y, cache = att(x, m, use_cache=True)
            out = [y]
            for z in more:
                y, cache = att(z, past_key_value=cache, use_cache=True)
                out.append(y)
        return out + [t.contiguous() for t in cache]
    _same(run(), general(run))


def test_nodes_under_hooks_checkpointing_and_threads(gpu):
    from torch.utils.checkpoint import checkpoint
    from adaptivetrainingsystem_amd import RMSNorm
    norm = RMSNorm(256).to(gpu)
    x = torch.randn(4, 256, device=gpu, requires_grad=True)
    dy = torch.randn(4, 256, device=gpu)
    norm(x).backward(dy)
    want = x.grad.clone(), norm.weight.grad.clone()
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t.cpu())[1], lambda t: t.to(gpu)):
        y = norm(x)
    assert packed == [x.shape, norm.weight.shape]
    x.grad = norm.weight.grad = None
    y.backward(dy)
    _same((x.grad, norm.weight.grad), want)
    x.grad = norm.weight.grad = None
    checkpoint(norm, x, use_reentrant=False).backward(dy)
    _same((x.grad, norm.weight.grad), want)
    results = [None] * 4

    def work(i):
        z = x.detach().clone().requires_grad_()
        with torch.cuda.stream(torch.cuda.Stream()):
            n = RMSNorm(256).to(gpu)
            n(z).backward(dy)
            torch.cuda.current_stream().synchronize()
        results[i] = z.grad
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    torch.cuda.synchronize()
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for r in results:
        _same(r, want[0])
    # in-place changes of a saved input are found, as with any saved tensor
    z = (x * 1.0)
    y = norm(z)
    z.mul_(2.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()


def test_errors_and_transforms_are_those_of_the_general_path(gpu, general):
    from adaptivetrainingsystem_amd import FusedRMSNorm, RotaryEmbedding, apply_rotary_pos_emb
    from adaptivetrainingsystem_amd._lib import AtsError
    norm = FusedRMSNorm(64).to(gpu)
    rope = RotaryEmbedding(64, 16)
    cos, sin = rope(4, torch.device(gpu))
    q = torch.zeros(1, 2, 8, 64, device=gpu)
    calls = [lambda: norm(torch.zeros(2, 72, device=gpu)), lambda: norm(torch.zeros(2, 64)),
             lambda: norm(torch.zeros(2, 64, device=gpu, dtype=torch.float64)),
             lambda: apply_rotary_pos_emb(q, q, cos, sin),                      # more positions than the table has
             lambda: apply_rotary_pos_emb(q[0], q[0], cos, sin), lambda: apply_rotary_pos_emb(q, q[:, :, :4], cos, sin)]
    for call in calls:
        for run in (call, lambda c=call: general(c)):
            with pytest.raises(AtsError):
                run()
    x = torch.randn(3, 64, device=gpu)
    for transform in (lambda: torch.func.vmap(norm)(x), lambda: torch.func.grad(lambda t: norm(t).sum())(x)):
        kinds = []
        for run in (transform, lambda t=transform: general(t)):
            try:
                run()
                kinds.append(None)
            except Exception as e:
                kinds.append(type(e))
        assert kinds[0] == kinds[1]
    with torch.inference_mode():
        _same(norm(x), general(lambda: norm(x)))


class _Marked(torch.Tensor):
    pass


@pytest.mark.filterwarnings("ignore")      # (of the tracer, about Python values)
def test_traces_subclasses_and_tangents_take_the_general_path(gpu, general):
    import torch.autograd.forward_ad as forward
    from adaptivetrainingsystem_amd import RMSNorm, RotaryEmbedding, apply_rotary_pos_emb
    g = torch.Generator().manual_seed(6)
    norm, (cos, sin) = RMSNorm(64).to(gpu), RotaryEmbedding(64, 16)(8, gpu)
    x, other = (torch.randn(1, 2, 8, 64, generator=g).to(gpu) for _ in range(2))
    rotate = lambda t: apply_rotary_pos_emb(t, t, cos, sin)
    for fn in (norm, rotate):
        # a trace made with gradients keeps the autograd function, and with it what it computes
        traced = torch.jit.trace(fn, (x.clone().requires_grad_(),), check_trace=False)
        _same(traced(other), fn(other))
        for grad in (False, True):
            kinds = lambda: [type(t) for t in (lambda r: r if isinstance(r, tuple) else (r,))(fn(x.as_subclass(_Marked).requires_grad_(grad)))]
            assert kinds() == general(kinds)

        def tangent():
            with forward.dual_level(), pytest.raises(Exception) as e:
                fn(forward.make_dual(x.clone().requires_grad_(), torch.ones_like(x)))
            return e.type
        assert tangent() == general(tangent)
    with torch.no_grad():
        assert isinstance(norm(x.as_subclass(_Marked)), _Marked)
    norm.weight = torch.nn.Parameter(norm.weight.detach().as_subclass(_Marked) * 3.0)
    assert type(norm.weight) is not torch.nn.Parameter
    _same(norm(x).as_subclass(torch.Tensor), general(lambda: norm(x).as_subclass(torch.Tensor)))


def test_positions_past_32_bits_are_refused(gpu):
    from adaptivetrainingsystem_amd import ops
    from adaptivetrainingsystem_amd._lib import AtsError
    q = torch.zeros(1, 2, 1, 64, device=gpu)
    cos, sin = ops.rope_table(4, 64, 10000.0, None, half=True)
    caches = [torch.full((1, 2, 8, 64), 7.0, device=gpu) for _ in range(2)]
    for pos in (1 << 32, (1 << 32) + 3, -(1 << 32)):
        with pytest.raises(AtsError, match="do not fit a cache"):
            ops.rope_append(q, q, q, cos, sin, *caches, pos, 0)
    assert all((c == 7.0).all() for c in caches)
