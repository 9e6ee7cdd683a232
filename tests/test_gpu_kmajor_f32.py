"""Float32 products of training against operands as they lie: data gradients from the forward's weights, weight gradients from
rows with the tokens along them, grouped and gathered.  Against float64 at the ends of tiles, of K and of the groups."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _bound(a, b):      # float32 sums of float32 products: a unit of 6e-8 per product and per addition at the worst end
    return 3e-7 * (a.abs() @ b.abs()) * max(1.0, a.shape[1] ** 0.5 / 4) + 1e-30


@pytest.mark.parametrize("counts,N,K", [([1], 4, 4), ([33, 0, 64, 31], 68, 36), ([65, 129, 1, 2, 0, 40, 7, 200], 512, 264),
                                        ([300, 257], 136, 1032), ([512], 512, 1024)])
def test_data_gradient_from_forward_weights(gpu, counts, N, K):
    print("case f32 nn", counts, N, K, flush=True)
    from adaptivetrainingsystem_amd import ops
    g = torch.Generator().manual_seed(sum(counts))
    E, n, ldb = len(counts), sum(counts), N + 4
    a = torch.randn(n, K, generator=g)
    w = [torch.randn(K, ldb, generator=g) for _ in range(E)]
    cnt = torch.tensor(counts, dtype=torch.int32)
    start = (torch.cumsum(cnt, 0) - cnt).to(torch.int32)
    w_gpu = [t.to(gpu) for t in w]
    out = ops.grouped_gemm_nn_f32(ops.weight_pointer_table(w_gpu), ldb, start.to(gpu), cnt.to(gpu), n, N, K, a.to(gpu)).cpu()
    for e, c in enumerate(counts):
        rows, m = a[start[e]:start[e] + c].double(), w[e][:, :N].double()
        assert ((out[start[e]:start[e] + c].double() - rows @ m).abs() <= _bound(rows, m)).all()


@pytest.mark.parametrize("counts,M,N", [([1], 4, 8), ([0, 31, 33, 64], 36, 68), ([40, 0, 0, 160, 1, 128, 95, 8], 264, 132),
                                        ([257], 512, 1024), ([37] * 8, 2816, 512)])
@pytest.mark.parametrize("gather", [False, True])
def test_weight_gradient_of_rows_as_they_lie(gpu, counts, M, N, gather):
    print("case f32 wgrad", counts, M, N, gather, flush=True)
    from adaptivetrainingsystem_amd import ops
    g = torch.Generator().manual_seed(sum(counts) + M)
    E, n = len(counts), sum(counts)
    a = torch.full((n + 3, M), float("nan"))
    a[:n] = torch.randn(n, M, generator=g)
    src = torch.randint(0, 2 * n, (n + 3,), generator=g)
    b = torch.randn(n + 3, N, generator=g)
    cnt = torch.tensor(counts, dtype=torch.int32)
    start = (torch.cumsum(cnt, 0) - cnt).to(torch.int32)
    args = (a.to(gpu), b.to(gpu), start.to(gpu), cnt.to(gpu))
    assert ops.wgrad_f32_supported(args[0], args[1], E)
    out = ops.wgrad_f32(*args, b_rows=src.int().to(gpu) if gather else None, b_row_div=2 if gather else 1).cpu()
    assert out.shape == (E, M, N)
    for e, c in enumerate(counts):
        r = torch.arange(int(start[e]), int(start[e]) + c)
        x, y = a[r].double().T, b[src[r] // 2 if gather else r].double()
        assert ((out[e].double() - x @ y).abs() <= _bound(x, y)).all()
    if E == 1 and not gather:
        assert torch.equal(ops.wgrad_f32(args[0][:n], args[1][:n]).cpu(), out[0])


def test_large_products_keep_their_copies(gpu):
    from adaptivetrainingsystem_amd import ops
    assert ops.grouped_gemm_nn_f32_supported(1, 512, 512, 1024) and not ops.grouped_gemm_nn_f32_supported(1, 8192, 4096, 4096)
    assert not ops.grouped_gemm_nn_f32_supported(1, 512, 510, 1024)
    t = torch.zeros(8192, 4096, device=gpu)
    assert not ops.wgrad_f32_supported(t, t) and ops.wgrad_f32_supported(t[:512, :512], t[:512, :512])
    assert not ops.wgrad_f32_supported(t[:512, 1:513], t[:512, :512]) and not ops.wgrad_f32_supported(t[:512, :512].T, t[:512, :512])
