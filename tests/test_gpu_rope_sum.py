"""The sum of a projection's K slices, its rotation and the cache append in one launch: the bits of the separate launches."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _tables(rows, D, gpu):
    ang = torch.arange(rows, dtype=torch.float64)[:, None] * torch.arange(1, D // 2 + 1, dtype=torch.float64) * 0.37
    return torch.cos(ang).float().to(gpu), torch.sin(ang).float().to(gpu)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,L,Hq,Hkv,D,parts,pos", [(1, 1, 1, 1, 8, 1, 0), (64, 1, 32, 8, 128, 8, 5), (33, 1, 6, 2, 64, 2, 1),
                                                     (3, 17, 5, 1, 24, 3, 2), (2, 40, 4, 4, 256, 9, 0), (7, 9, 3, 3, 40, 16, 3)])
def test_sum_rotate_append(gpu, B, L, Hq, Hkv, D, parts, pos, dtype):
    print("case rope sum", B, L, Hq, Hkv, D, parts, dtype, flush=True)
    from adaptivetrainingsystem_amd import _lib, ops
    N = (Hq + 2 * Hkv) * D
    p = torch.randn(parts, B * L, N, generator=torch.Generator().manual_seed(B + D)).to(gpu)
    cos, sin = _tables(L + 3, D, gpu)
    caches = lambda: [torch.full((B, Hkv, pos + L + 2, D), 7.0, dtype=dtype, device=gpu) for _ in range(2)]
    (ka, va), (kb, vb) = caches(), caches()
    qkv = ops.sum_partials(p, dtype).view(B, L, Hq + 2 * Hkv, D).transpose(1, 2)
    want = ops.rope_append(qkv[:, :Hq], qkv[:, Hq:Hq + Hkv], qkv[:, Hq + Hkv:], cos, sin, ka, va, pos, 0)
    q = torch.empty(B, Hq, L, D, dtype=dtype, device=gpu)
    tag = _lib.ATS_F32 if dtype == torch.float32 else _lib.ATS_BF16
    call = lambda cache_pos: _lib.load().ats_rope_sum_append(
        p.data_ptr(), parts, B * L * N, q.data_ptr(), kb.data_ptr(), vb.data_ptr(), cos.data_ptr(), sin.data_ptr(), D // 2, L + 3, B,
        Hq, Hkv, L, D, kb.stride(0), kb.stride(1), kb.stride(2), cache_pos, pos + L + 2, tag, torch.cuda.current_stream().cuda_stream)
    assert call(pos) == 0
    for a, b in ((q, want), (kb, ka), (vb, va)):
        assert torch.equal(a, b)
    assert call(pos + 3) != 0        # behind the cache's capacity: refused


@pytest.mark.parametrize("T,seq,fused", [(32, 1, False), (33, 1, True), (64, 1, True), (200, 40, True), (256, 256, True), (260, 1, False)])
def test_linear_rope_append(gpu, T, seq, fused):
    print("case linear rope append", T, seq, flush=True)
    from adaptivetrainingsystem_amd import ops
    Hq, Hkv, D, K = 6, 2, 64, 2304
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, K, generator=g).to(gpu, torch.bfloat16)
    w = (torch.randn((Hq + 2 * Hkv) * D, K, generator=g) * 0.02).to(gpu, torch.bfloat16)
    cos, sin = _tables(seq, D, gpu)
    B = T // seq if T % seq == 0 else 0
    assert B
    caches = lambda: [torch.full((B, Hkv, seq + 3, D), 7.0, dtype=torch.bfloat16, device=gpu) for _ in range(2)]
    (ka, va), (kb, vb) = caches(), caches()
    qkv = ops.linear_nt(x, w).view(B, seq, Hq + 2 * Hkv, D).transpose(1, 2)
    want = ops.rope_append(qkv[:, :Hq], qkv[:, Hq:Hq + Hkv], qkv[:, Hq + Hkv:], cos, sin, ka, va, 3, 0)
    q = ops.linear_rope_append(x, w, cos, sin, kb, vb, 3, seq)
    assert (q is not None) == fused
    if fused:
        for a, b in ((q, want), (kb, ka), (vb, va)):
            assert torch.equal(a, b)
