"""Grouped bfloat16 products with a few hundred rows per group (tiles of equal height, weights in the deep ring): every
number of 32-row steps a tile can have, tile counts on both sides of a step up, and the ends of K."""
import pytest
import torch

from tests.test_gpu_parity import A, BF16_TOL, gen, ops, rel_err, same_bits  # noqa: F401

pytestmark = pytest.mark.gpu

# heights 32 .. 256 in one tile, two tiles from 257 rows, three from 513, empty groups; K of 1, 2, 3 and 17 slabs
CASES = [([193, 225, 255, 256], 264, 64), ([257, 320, 321, 384], 136, 128), ([385, 448, 449, 512], 72, 192),
         ([513, 0, 600, 1, 33, 97, 161, 767], 264, 1088), ([700, 200, 65], 520, 256)]


def _weights(g, E, N, K, gpu):
    return [(torch.randn(N, K, generator=g) * 0.1).bfloat16().to(gpu) for _ in range(E)]


@pytest.mark.parametrize("counts,N,K", CASES)
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_mid_rows_plain_gathered_and_k_major(ops, gpu, counts, N, K, out_dtype):  # noqa: F811
    print("case mid rows", counts, N, K, out_dtype, flush=True)
    g = gen(311)
    E, n = len(counts), sum(counts)
    w = _weights(g, E, N, K, gpu)
    count = torch.tensor(counts, dtype=torch.int32)
    start = (torch.cumsum(count, 0) - count).to(torch.int32).to(gpu)
    a = torch.randn(n, K, generator=g).bfloat16().to(gpu)
    src = torch.randint(0, 2 * n, (n,), generator=g).to(torch.int32).to(gpu)
    args = (ops.weight_pointer_table(w), K, N, start, count.to(gpu), n, n, N, K)
    out = ops.grouped_gemm_nt(*args, a=a, out_dtype=out_dtype)
    got = ops.grouped_gemm_nt(*args, a=a, a_rows=src, a_row_div=2, out_dtype=out_dtype)
    assert same_bits(got, ops.grouped_gemm_nt(*args, a=a[(src // 2).long()].contiguous(), out_dtype=out_dtype))
    kmajor = [t.t().contiguous() for t in w]
    nn = ops.grouped_gemm_nn(ops.weight_pointer_table(kmajor), N, start, args[4], n, n, N, K, a, out_dtype=out_dtype) \
        if ops.grouped_gemm_nn_supported(E, n, N, K, N, torch.bfloat16) else None
    off = 0
    for e, c in enumerate(counts):
        ref = a[off:off + c].cpu().double() @ w[e].cpu().double().T
        if c:
            assert rel_err(out[off:off + c], ref) <= BF16_TOL
            if nn is not None:
                assert rel_err(nn[off:off + c], ref) <= BF16_TOL
        off += c


@pytest.mark.parametrize("counts,I,H", [(c, n, k) for c, n, k in CASES if n % 8 == 0])
def test_mid_rows_swiglu(ops, gpu, counts, I, H):  # noqa: F811
    print("case mid rows swiglu", counts, I, H, flush=True)
    g = gen(312)
    E, n = len(counts), sum(counts)
    w = _weights(g, E, 2 * I, H, gpu)
    count = torch.tensor(counts, dtype=torch.int32)
    start = (torch.cumsum(count, 0) - count).to(torch.int32).to(gpu)
    a = torch.randn(n, H, generator=g).bfloat16().to(gpu)
    h = ops.grouped_gateup_swiglu(a, ops.weight_pointer_table(w), start, count.to(gpu), n, n, H, I)
    off = 0
    for e, c in enumerate(counts):
        r = a[off:off + c].cpu().double() @ w[e].cpu().double().T
        if c:
            assert rel_err(h[off:off + c], torch.nn.functional.silu(r[:, :I]) * r[:, I:]) <= BF16_TOL
        off += c
