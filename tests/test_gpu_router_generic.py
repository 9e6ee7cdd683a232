"""Router logits of the general kernel at the remainders of its step of 256 columns and 8 experts."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,E,H", [(1, 1, 1), (3, 8, 255), (5, 7, 256), (4, 9, 257), (2, 17, 511), (513, 8, 516), (6, 64, 1023), (2, 3, 63)])
def test_router_logits(gpu, T, E, H, dtype):
    print("case router logits", T, E, H, dtype, flush=True)
    from adaptivetrainingsystem_amd import ops
    g = torch.Generator().manual_seed(T + E + H)
    x, w = torch.randn(T, H, generator=g).to(gpu, dtype), torch.randn(E, H, generator=g).to(gpu, dtype)
    bias = torch.randn(E, generator=g).to(gpu)
    got = ops.router_logits(x, w, bias).cpu().double()
    xd, wd = x.cpu().double(), w.cpu().double()
    want = xd @ wd.T + bias.cpu().double()
    # a lane's chain of ceil(H / 64) products, six steps over the lanes, the bias: each rounds once (a product at most once more)
    bound = (2 * (-(-H // 64)) + 7) * 2.0 ** -24 * (xd.abs() @ wd.abs().T + bias.cpu().double().abs())
    assert bool(((got - want).abs() <= bound).all())
