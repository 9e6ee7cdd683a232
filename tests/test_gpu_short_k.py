"""Weight gradients over a few hundred rows per group on the 128 x 128 tile that shares a CU."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# rows per group: none (zeros), one, one slab, its neighbours, several slabs; columns and rows that end inside a tile.  At
# least 2048 tiles and at most eight slabs on average, so that the tile under test is the one that runs
@pytest.mark.parametrize("counts,M,N", [([0, 1, 64, 65], 4104, 2056), ([200, 448, 0, 449, 31, 127], 2600, 2184), ([33] * 64, 264, 1416)])
def test_short_k_weight_gradient(gpu, counts, M, N):
    print("case short K", counts[:6], M, N, flush=True)
    from adaptivetrainingsystem_amd import _lib, ops
    E, rows = len(counts), sum(counts)
    g = torch.Generator().manual_seed(rows)
    cnt = torch.tensor(counts, dtype=torch.int32, device=gpu)
    start = (torch.cumsum(cnt, 0) - cnt).to(torch.int32)
    a = (torch.randn(rows, M, generator=g) * 0.5).bfloat16().to(gpu)
    b = (torch.randn(rows, N, generator=g) * 0.5).bfloat16().to(gpu)
    ks, kc = ops.wgrad_plan(cnt)
    ld = ops.wgrad_padded_rows(rows, E)
    assert (ld // E + 63) // 64 <= 8 and E * -(-M // 128) * -(-N // 128) >= 2048
    lhsT, rhsT = (ops.transpose_grouped_rows(t, start, cnt, rows) for t in (a, b))
    a_ptrs, b_ptrs, rs, rc = ops.wgrad_tables(ks, M, lhsT, rhsT)
    out = ops.grouped_gemm_nt(b_ptrs, ld, N, rs, rc, E * M, E * M, N, ld, a_ptrs=a_ptrs, lda=ld, k_count=kc, dtype=torch.bfloat16,
                              out_dtype=torch.bfloat16).view(E, M, N)
    off = 0
    for e, c in enumerate(counts):
        ref = a[off:off + c].double().T @ b[off:off + c].double()
        if c:      # the bits of the 256 x 256 tile, on the group's rows alone
            one, (first, height) = torch.empty_like(out[e]), ops._single_group(M, gpu)
            assert _lib.load().ats_wgrad_tn(a[off:].data_ptr(), M, b[off:].data_ptr(), N, one.data_ptr(), c, M, N, 1, first.data_ptr(),
                                            height.data_ptr(), _lib.ATS_BF16, _lib.ATS_BF16, torch.cuda.current_stream().cuda_stream) == 0
            assert torch.equal(out[e], one)
        off += c
        # float32 sums of exact products, one rounding to bfloat16
        bound = 2.0 ** -8 * ref.abs() + 4e-7 * max(c, 1) * a.abs().max().double() * b.abs().max().double()
        assert ((out[e].double() - ref).abs() <= bound).all()
