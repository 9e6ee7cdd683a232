"""Weight gradients of a linear layer from operands as they lie (tokens along the rows), at the ends of tiles and slabs."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# tokens: one, around one slab, an odd number of slabs, enough for slices of K; rows and columns of less than a fragment, of
# tiles of every height, with a remainder of eight; strides wider than the matrix
@pytest.mark.parametrize("T,M,N", [(1, 8, 8), (63, 264, 136), (64, 256, 256), (65, 520, 1000), (200, 1032, 512),
                                   (1777, 264, 520), (4100, 1024, 512), (131, 4096, 264)])
@pytest.mark.parametrize("pad", [0, 24])
def test_wgrad_of_rows_as_they_lie(gpu, T, M, N, pad):
    print("case wgrad tn", T, M, N, pad, flush=True)
    from adaptivetrainingsystem_amd import ops
    g = torch.Generator().manual_seed(T + M)
    # what lies behind the last token and behind a row must not reach the result
    full_a = torch.full((T + 64, M + pad), float("nan"), dtype=torch.bfloat16)
    full_b = torch.full((T + 64, N + pad), float("nan"), dtype=torch.bfloat16)
    full_a[:T, :M] = torch.randn(T, M, generator=g) * 0.5
    full_b[:T, :N] = torch.randn(T, N, generator=g) * 0.5
    a, b = full_a.to(gpu)[:T, :M], full_b.to(gpu)[:T, :N]
    assert ops.wgrad_linear_supported(a, b)
    out = ops.wgrad_linear(a, b)
    ref = a.double().T @ b.double()
    # float32 sums of exact products (a few units of 6e-8 of their sizes), one rounding to bfloat16
    bound = 2.0 ** -8 * ref.abs() + 4e-7 * (a.double().abs().T @ b.double().abs())
    assert ((out.double() - ref).abs() <= bound).all()
    start, count = ops._single_group(T, a.device)
    want = ops.wgrad_dense(*(ops.transpose_grouped_rows(t.contiguous(), start, count, T) for t in (a, b)), T)
    assert torch.equal(out, want)      # the same tiles, slices and order
    if M % 16 == 0:
        parts = ops.wgrad_linear(a, b, (M // 2, M // 2))
        assert torch.equal(torch.cat(parts), out) and all(p.is_contiguous() for p in parts)


def test_operands_that_keep_the_transposed_route(gpu):
    from adaptivetrainingsystem_amd import ops
    t = torch.zeros(128, 64, dtype=torch.bfloat16, device=gpu)
    ok = ops.wgrad_linear_supported
    assert ok(t, t) and ok(t[:, 8:32], t)
    assert not ok(t.float(), t.float()) and not ok(t[:, :60], t) and not ok(t[:, 4:36], t) and not ok(t.t(), t.t())
    assert not ok(t[:0], t[:0])


@pytest.mark.parametrize("T,pitch", [(300, 5_600_000), (3000, 600_000), (100, 12_000_000)])
def test_operands_of_two_to_four_gib(gpu, T, pitch):
    """Rows so far apart that the advance along K passes 2^31 bytes: the bits of contiguous copies."""
    print("case wgrad tn extent", T, pitch, flush=True)
    from adaptivetrainingsystem_amd import ops
    M, N = 72, 264
    g = torch.Generator().manual_seed(T)
    dy, x = (torch.randn(T, n, generator=g).to(gpu, torch.bfloat16) for n in (M, N))
    want = ops.wgrad_linear(dy, x)
    for far in (0, 1):
        pair = [dy, x]
        wide = torch.empty((T - 1) * pitch + N, dtype=torch.bfloat16, device=gpu).as_strided((T, pair[far].shape[1]), (pitch, 1))
        wide.copy_(pair[far])
        assert 2 ** 31 < (T + 63) // 64 * 64 * pitch * 2 < 2 ** 32
        pair[far] = wide
        assert ops.wgrad_linear_supported(*pair)
        assert torch.equal(ops.wgrad_linear(*pair), want)
