"""Attention of a prompt whose queries are rotated as they are loaded: the bits of the rotation and the attention apart."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L,Hq,Hkv,D", [(1, 17, 1, 1, 64), (3, 5, 16, 4, 64), (2, 127, 4, 2, 128), (2, 129, 4, 4, 128), (3, 300, 6, 2, 64),
                                          (1, 4097, 2, 1, 128), (1, 4100, 2, 2, 64), (5, 61, 8, 1, 128)])
@pytest.mark.parametrize("keep_values", [False, True])
def test_prompt_attention(gpu, B, L, Hq, Hkv, D, keep_values):
    print("case prompt attention", B, L, Hq, Hkv, D, keep_values, flush=True)
    from adaptivetrainingsystem_amd import _lib, ops
    qkv = torch.randn(B * L, (Hq + 2 * Hkv) * D, generator=torch.Generator().manual_seed(L)).to(gpu, torch.bfloat16)
    ang = torch.arange(L, dtype=torch.float64)[:, None] * torch.arange(1, D // 2 + 1, dtype=torch.float64) * 0.37
    cos, sin = torch.cos(ang).float().to(gpu), torch.sin(ang).float().to(gpu)
    rows = qkv.view(B, L, Hq + 2 * Hkv, D).transpose(1, 2)
    q, k = ops.rope(rows[:, :Hq], rows[:, Hq:Hq + Hkv], cos, sin, 0)
    v = rows[:, Hq + Hkv:]
    want = ops.causal_attention(q, k, v, 0.1, split_keys=False)
    if not _lib.load().ats_attention_fwd_rope_supported(B, Hq, Hkv, L, L, D):
        pytest.skip("keys in ranges")
    out, kk, vv = ops.prompt_attention(qkv, cos, sin, B, Hkv, D, 0.1, keep_values)
    assert torch.equal(out, want) and torch.equal(kk, k) and torch.equal(vv, v)
    assert vv.is_contiguous() == keep_values or Hq + Hkv == 0
    assert ops.prompt_attention(qkv.float(), cos, sin, B, Hkv, D, 0.1, keep_values) is None


# on both sides of the size from which a prompt without a cache has its queries rotated in the attention too (6 M of them)
@pytest.mark.parametrize("B,L", [(2, 241), (1, 6143), (1, 6144), (3, 2049)])
def test_prompt_without_a_cache(gpu, B, L):
    print("case prompt without cache", B, L, flush=True)
    from adaptivetrainingsystem_amd import GroupedQueryAttention
    from adaptivetrainingsystem_amd.workloads import LayerConfig
    torch.manual_seed(L)
    att = GroupedQueryAttention(LayerConfig(1024, 4096, 1, 1, num_heads=8, num_kv_heads=2, seq_length=8192)).to(gpu, torch.bfloat16).eval()
    x = torch.randn(B, L, 1024, generator=torch.Generator().manual_seed(L)).to(gpu, torch.bfloat16)
    with torch.no_grad():
        assert torch.equal(att(x), att(x, use_cache=True)[0])


def test_prompt_attention_refusals(gpu):
    from adaptivetrainingsystem_amd import _lib
    lib = _lib.load()
    ok = lib.ats_attention_fwd_rope_supported
    assert ok(3, 32, 8, 1777, 1777, 128) and not ok(3, 32, 8, 1777, 1777, 96) and not ok(3, 32, 5, 1777, 1777, 128)
    assert not ok(64, 32, 8, 4, 4, 128) and not ok(3, 32, 8, 10, 9, 128)        # 16 rows of a kv head decode; fewer keys than queries
    t = torch.zeros(64 * 64, dtype=torch.bfloat16, device=gpu)
    tab = torch.zeros(64 * 32, device=gpu)
    s = torch.cuda.current_stream().cuda_stream
    call = lambda q=t.data_ptr(), q_sl=64, rows=64, stride=32: lib.ats_attention_fwd_rope(
        q, 4096, 4096, q_sl, tab.data_ptr(), tab.data_ptr(), stride, rows, t.data_ptr(), 4096, 4096, t.data_ptr(), 4096, 64, 4096,
        torch.empty_like(t).data_ptr(), 1, 1, 1, 64, 64, 64, 0.1, s)
    assert call() == 0
    torch.cuda.synchronize()
    assert call(q=t.data_ptr() + 2) != 0 and call(q_sl=63) != 0 and call(rows=63) != 0 and call(stride=30) != 0
