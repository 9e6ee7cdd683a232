"""Row tiles whose height is an odd number of 16-row fragments (the two wave rows then differ by one fragment)."""
import pytest
import torch

from tests.test_gpu_parity import A, BF16_TOL, gen, ops, rel_err, same_bits  # noqa: F401

pytestmark = pytest.mark.gpu


# 1, 3, 5, .. 15 fragments in one tile and in two or three, last rows at a fragment's first row, an even neighbour beside each
@pytest.mark.parametrize("counts,N,K", [([1, 16, 33, 48, 65, 80, 500, 520], 264, 128), ([193, 208, 209, 225, 240, 200], 136, 64),
                                        ([257, 273, 288, 289, 337, 352, 401, 465], 72, 192), ([529, 600, 625, 721], 520, 320)])
def test_odd_heights(ops, gpu, counts, N, K):  # noqa: F811
    print("case odd heights", counts, N, K, flush=True)
    g = gen(411)
    E, n = len(counts), sum(counts)
    assert n // E > 150
    w = [(torch.randn(2 * N, K, generator=g) * 0.1).bfloat16().to(gpu) for _ in range(E)]
    count = torch.tensor(counts, dtype=torch.int32)
    start = (torch.cumsum(count, 0) - count).to(torch.int32).to(gpu)
    count = count.to(gpu)
    a = torch.randn(n, K, generator=g).bfloat16().to(gpu)
    tab = ops.weight_pointer_table(w)
    out = torch.full((n + 1, 2 * N), 7.0, dtype=torch.bfloat16, device=gpu)
    ops.grouped_gemm_nt(tab, K, 2 * N, start, count, n + 1, n, 2 * N, K, a=a, out=out)
    h = ops.grouped_gateup_swiglu(a, tab, start, count, n, n, K, N)
    nn = None
    if ops.grouped_gemm_nn_supported(E, n, 2 * N, K, 2 * N, torch.bfloat16):
        nn = ops.grouped_gemm_nn(ops.weight_pointer_table([t.t().contiguous() for t in w]), 2 * N, start, count, n, n, 2 * N, K, a)
    off = 0
    for e, c in enumerate(counts):
        r = a[off:off + c].cpu().double() @ w[e].cpu().double().T
        assert rel_err(out[off:off + c], r) <= BF16_TOL
        assert rel_err(h[off:off + c], torch.nn.functional.silu(r[:, :N]) * r[:, N:]) <= BF16_TOL
        if nn is not None:
            assert same_bits(nn[off:off + c], out[off:off + c])
        off += c
    assert torch.all(out[n:] == 7.0)


@pytest.mark.parametrize("rows,N,K", [(1111, 4096, 64), (5331, 4096, 64), (5331, 2048, 128), (333, 6144, 64), (7777, 3072, 64)])
def test_k_major_dense_heights(ops, gpu, rows, N, K):  # noqa: F811
    """One group against weights stored [K, N]: the heights and the bits of the product against [N, K]."""
    print("case k-major heights", rows, N, K, flush=True)
    g = gen(412)
    x = torch.randn(rows, K, generator=g).bfloat16().to(gpu)
    w = (torch.randn(N, K, generator=g) * 0.1).bfloat16().to(gpu)
    start, count = torch.zeros(1, dtype=torch.int32, device=gpu), torch.full((1,), rows, dtype=torch.int32, device=gpu)
    assert ops.grouped_gemm_nn_supported(1, rows, N, K, N, torch.bfloat16)
    out = ops.grouped_gemm_nn(ops.weight_pointer_table([w.t().contiguous()]), N, start, count, rows, rows, N, K, x)
    assert rel_err(out, x.float().cpu().double() @ w.float().cpu().double().T) <= BF16_TOL
    assert same_bits(out, ops.grouped_gemm_nt(ops.weight_pointer_table([w]), K, N, start, count, rows, rows, N, K, a=x))
