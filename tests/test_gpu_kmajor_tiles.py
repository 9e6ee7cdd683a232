"""Float32 products of operands as they lie: 32- and 64-row tiles and the gathered operand give the bits of one group on its own."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _groups(counts, gpu):
    c = torch.tensor(counts, dtype=torch.int32, device=gpu)
    return (torch.cumsum(c, 0) - c).int(), c


@pytest.mark.parametrize("counts", [(0, 1, 31, 32, 33, 129, 200, 5), (500, 470, 530, 512, 640, 33, 700, 615), (7,), (64, 0, 0, 65)])
@pytest.mark.parametrize("M,N", [(2816, 512), (516, 36)])
def test_weight_gradient_gathered(gpu, counts, M, N):
    print("case kmajor wgrad", counts, M, N, flush=True)
    from adaptivetrainingsystem_amd import ops
    g = torch.Generator().manual_seed(sum(counts) + M)
    R = sum(counts)
    a, src = torch.randn(R, M, generator=g).to(gpu), torch.randn((R + 1) // 2, N, generator=g).to(gpu)
    rows = torch.randperm(R, generator=g).int().to(gpu)
    start, count = _groups(counts, gpu)
    if not ops.wgrad_f32_supported(a, src, len(counts)):
        pytest.skip("transposed copies are faster")
    b = src[(rows // 2).long()].contiguous()
    out = ops.wgrad_f32(a, src, start, count, b_rows=rows, b_row_div=2)
    assert torch.equal(out, ops.wgrad_f32(a, b, start, count))
    lo = 0
    for e, n in enumerate(counts):
        ae, be = a[lo:lo + n], b[lo:lo + n]
        lo += n
        want = ae.double().T @ be.double()
        # n products in four chains of ceil(n / 4 + 32) roundings at most, three additions
        bound = (n / 4 + 36) * 2.0 ** -24 * (ae.double().abs().T @ be.double().abs())
        assert bool(((out[e].double() - want).abs() <= bound).all())
        if n and ops.wgrad_f32_supported(ae, be):
            assert torch.equal(out[e], ops.wgrad_f32(ae, be))


@pytest.mark.parametrize("counts", [(0, 1, 31, 32, 33, 129, 200, 5), (500, 470, 530, 512, 640, 33, 700, 615), (7, 64)])
@pytest.mark.parametrize("N,K", [(512, 2816), (1408, 512), (36, 516)])
def test_data_gradient_groups(gpu, counts, N, K):
    print("case kmajor dgrad", counts, N, K, flush=True)
    from adaptivetrainingsystem_amd import ops
    g = torch.Generator().manual_seed(sum(counts) + N)
    R, E = sum(counts), len(counts)
    a = torch.randn(R, K, generator=g).to(gpu)
    ws = [torch.randn(K, N, generator=g).to(gpu) for _ in range(E)]
    start, count = _groups(counts, gpu)
    if not ops.grouped_gemm_nn_f32_supported(E, R, N, K):
        pytest.skip("transposed copies are faster")
    out = ops.grouped_gemm_nn_f32(ops.weight_pointer_table(ws), N, start, count, R, N, K, a)
    lo = 0
    for e, n in enumerate(counts):
        ae = a[lo:lo + n]
        if n:
            bound = (K / 4 + 36) * 2.0 ** -24 * (ae.double().abs() @ ws[e].double().abs())
            assert bool(((out[lo:lo + n].double() - ae.double() @ ws[e].double()).abs() <= bound).all())
            if ops.grouped_gemm_nn_f32_supported(1, n, N, K):
                s1, c1 = _groups((n,), gpu)
                assert torch.equal(out[lo:lo + n], ops.grouped_gemm_nn_f32(ops.weight_pointer_table([ws[e]]), N, s1, c1, n, N, K, ae.contiguous()))
        lo += n
