"""Dense float32 products of more than 256 rows, on both sides of the rule between slices of K and a wave over all of K."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,N,K", [(256, 512, 512), (257, 512, 512), (300, 36, 68), (511, 1024, 516), (700, 1000, 1000), (1500, 2048, 2048),
                                   (2001, 512, 1408), (4100, 516, 512), (257, 4, 8), (276, 6144, 512), (390, 11008, 256)])
def test_linear(gpu, T, N, K):
    print("case dense f32", T, N, K, flush=True)
    from adaptivetrainingsystem_amd import ops
    g = torch.Generator().manual_seed(T + N)
    x, w = torch.randn(T, K, generator=g).to(gpu), torch.randn(N, K, generator=g).to(gpu)
    out = ops.linear_nt(x, w)
    xd, wd = x.double(), w.double()
    # at most K additions in one chain (all of K in a wave), each product in it rounds at most once more
    bound = (K + 4) * 2.0 ** -24 * (xd.abs() @ wd.abs().T)
    assert bool(((out.double() - xd @ wd.T).abs() <= bound).all())
