"""Dense bfloat16 products whose launch takes row tiles of 128 to 256 rows, against float64: each height, remainders in the
last tile, a ragged number of columns, the aligned tile list and the plain one; rows behind the last are not written."""
import pytest
import torch

from tests.test_gpu_parity import A, BF16_TOL, gen, ops, rel_err  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,N,K", [
    (193, 4096, 128), (257, 4096, 64), (1000, 6144, 128), (1500, 4096, 256), (1537, 4104, 128), (1409, 2048, 128),       # 128
    (4200, 2048, 192), (2561, 4096, 64),                                                                                # 160
    (3000, 4096, 128), (5331, 4096, 128), (5331, 6144, 64), (2881, 4000, 64),                                           # 192
    (8000, 3072, 128), (7937, 3072, 64),                                                                                # 224
    (2048, 6144, 128), (769, 6144, 64), (4096, 4096, 64)])                                                              # 256
def test_dense_tile_heights(ops, gpu, rows, N, K):  # noqa: F811
    print("case dense tile rows", rows, N, K, flush=True)
    g = gen(77)
    x = torch.randn(rows, K, generator=g).to(torch.bfloat16).to(gpu)
    w = (torch.randn(N, K, generator=g) * 0.1).to(torch.bfloat16).to(gpu)
    out = torch.full((rows + 3, N), 7.0, dtype=torch.bfloat16, device=gpu)
    start, count = torch.zeros(1, dtype=torch.int32, device=gpu), torch.full((1,), rows, dtype=torch.int32, device=gpu)
    ops.grouped_gemm_nt(ops.weight_pointer_table([w]), K, N, start, count, rows + 3, rows, N, K, a=x, out=out)
    ref = x.float() @ w.float().T                       # products of bfloat16 values, at most 256 of them: exact to 2^-16
    assert rel_err(out[:rows], ref.cpu().double()) <= BF16_TOL
    assert torch.all(out[rows:] == 7.0)
    if rows >= 200:      # the last rows by themselves: the same sums over K whatever the height
        tail = ops.grouped_gemm_nt(ops.weight_pointer_table([w]), K, N, start, torch.full_like(count, 200), 200, 200, N, K,
                                   a=x[rows - 200:].contiguous())
        assert torch.equal(tail, out[rows - 200:rows])
