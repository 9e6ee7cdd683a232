"""Grouped products whose large tiles would leave most of the chip idle: the 32 and 64-row tiles with K cut into slices
inside a workgroup, and the float32 2 x 2 tiles above 256 rows per group.  Against float64 at the edges of the tiles, of
the groups and of K."""
import pytest
import torch

from tests.test_gpu_parity import A, BF16_TOL, F32_TOL, gen, ops, rel_err, same_bits  # noqa: F401

pytestmark = pytest.mark.gpu

# rows per group, output columns, K: one row; tile remainders of 1, 31, 33, 63, 65; groups without rows; K of one 16-byte
# piece, of a ragged slab, of fewer slabs than slices; above 256 rows per group (float32: tiles without slices of K)
CASES = [([1], 8, 8), ([33], 24, 40), ([64, 0, 31, 65], 72, 136), ([129, 1, 63], 264, 1000), ([200], 512, 64),
         ([300, 257], 136, 72), ([513], 520, 264), ([600, 0, 400], 64, 1032), ([20, 12], 40, 2048)]


@pytest.mark.parametrize("counts,N,K", CASES)
@pytest.mark.parametrize("dtype,out_dtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16),
                                             (torch.bfloat16, torch.float32)])
def test_small_tiles_plain(ops, gpu, counts, N, K, dtype, out_dtype):  # noqa: F811
    print("case small tiles", counts, N, K, dtype, out_dtype, flush=True)
    g = gen(301)
    E, n = len(counts), sum(counts)
    w = [(torch.randn(N, K, generator=g) * 0.1).to(dtype).to(gpu) for _ in range(E)]
    count = torch.tensor(counts, dtype=torch.int32)
    start = (torch.cumsum(count, 0) - count).to(torch.int32).to(gpu)
    a = torch.randn(n + 3, K, generator=g).to(dtype).to(gpu)
    src = torch.randint(0, 2 * (n + 3), (n,), generator=g).to(torch.int32).to(gpu)
    tab = ops.weight_pointer_table(w)
    args = (tab, K, N, start, count.to(gpu), n + 2, n, N, K)
    out = ops.grouped_gemm_nt(*args, a=a, out_dtype=out_dtype)
    got = ops.grouped_gemm_nt(*args, a=a, a_rows=src, a_row_div=2, out_dtype=out_dtype)
    same = ops.grouped_gemm_nt(*args, a=a[(src // 2).long()].contiguous(), out_dtype=out_dtype)
    assert same_bits(got[:n], same[:n])
    off, tol = 0, F32_TOL if dtype == torch.float32 else BF16_TOL
    for e, c in enumerate(counts):
        if c:
            ref = a[off:off + c].cpu().double() @ w[e].cpu().double().T
            assert rel_err(out[off:off + c], ref) <= tol
        off += c
    # rows outside the groups are not written
    lib = __import__("adaptivetrainingsystem_amd._lib", fromlist=["load"]).load()
    buf = torch.full((n + 2, N), 7.0, dtype=out_dtype, device=gpu)
    tag = lambda t: 0 if t == torch.float32 else 1
    assert lib.ats_grouped_gemm_nt(a.data_ptr(), None, K, n + 3, None, 1, tab.data_ptr(), K, N, buf.data_ptr(), N,
                                   start.data_ptr(), args[4].data_ptr(), None, E, n, N, K, tag(dtype), tag(out_dtype),
                                   None) == 0
    torch.cuda.synchronize()
    assert torch.all(buf[n:] == 7.0) and same_bits(buf[:n], out[:n])


@pytest.mark.parametrize("counts,I,H", [([1], 8, 8), ([33, 0, 40], 40, 136), ([64, 100], 264, 1000), ([300, 257], 136, 72),
                                        ([9, 30], 24, 512)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_small_tiles_swiglu(ops, gpu, counts, I, H, dtype):  # noqa: F811
    print("case small tiles swiglu", counts, I, H, dtype, flush=True)
    g = gen(302)
    E, n = len(counts), sum(counts)
    w = [(torch.randn(2 * I, H, generator=g) * 0.1).to(dtype).to(gpu) for _ in range(E)]
    count = torch.tensor(counts, dtype=torch.int32)
    start = (torch.cumsum(count, 0) - count).to(torch.int32).to(gpu)
    a = torch.randn(n, H, generator=g).to(dtype).to(gpu)
    h = ops.grouped_gateup_swiglu(a, ops.weight_pointer_table(w), start, count.to(gpu), n, n, H, I)
    off = 0
    for e, c in enumerate(counts):
        if c:
            r = a[off:off + c].cpu().double() @ w[e].cpu().double().T
            ref = torch.nn.functional.silu(r[:, :I]) * r[:, I:]
            assert rel_err(h[off:off + c], ref) <= (F32_TOL if dtype == torch.float32 else BF16_TOL)
        off += c


@pytest.mark.parametrize("k_counts,M,N", [([64, 128, 64], 40, 72), ([640, 64], 264, 136), ([192], 520, 264)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_small_tiles_with_a_k_per_group(ops, gpu, k_counts, M, N, dtype):  # noqa: F811
    """Weight gradients: every group has its own K and its own base pointers into two transposed buffers."""
    print("case small tiles k per group", k_counts, M, N, dtype, flush=True)
    g = gen(303)
    E, ld = len(k_counts), sum(k_counts)
    lhs = torch.randn(M, ld, generator=g).to(dtype).to(gpu)
    rhs = torch.randn(N, ld, generator=g).to(dtype).to(gpu)
    kc = torch.tensor(k_counts, dtype=torch.int32)
    ks = torch.cumsum(kc, 0) - kc
    es = lhs.element_size()
    a_ptrs = (ks.long() * es + lhs.data_ptr()).to(gpu)
    b_ptrs = (ks.long() * es + rhs.data_ptr()).to(gpu)
    rs = (torch.arange(E, dtype=torch.int32) * M).to(gpu)
    rc = torch.full((E,), M, dtype=torch.int32, device=gpu)
    out = ops.grouped_gemm_nt(b_ptrs, ld, N, rs, rc, E * M, E * M, N, ld, a_ptrs=a_ptrs, lda=ld, k_count=kc.to(gpu),
                              dtype=dtype, out_dtype=dtype).view(E, M, N)
    for e in range(E):
        sl = slice(int(ks[e]), int(ks[e] + kc[e]))
        ref = lhs[:, sl].cpu().double() @ rhs[:, sl].cpu().double().T
        assert rel_err(out[e], ref) <= (F32_TOL if dtype == torch.float32 else BF16_TOL)
