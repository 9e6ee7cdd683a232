"""Attention of up to 16 query rows per kv head (attention_decode_kernel) against float32 on the CPU: one key up to chunks
that end inside a wave's turn, more waves than chunks, several parts, several positions with the causal bound, a padding
bias, strided values, the log-sum-exp."""
import pytest
import torch

from tests.test_gpu_attention import BF16_TOL, gen, ops, rel_err  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,L,Lk,D", [(1, 1, 1, 1, 1, 64), (2, 4, 2, 1, 31, 128), (1, 8, 2, 1, 33, 64), (3, 4, 4, 1, 129, 128),
                                             (1, 16, 1, 1, 257, 128), (2, 4, 1, 4, 300, 64), (1, 6, 2, 5, 5, 128),
                                             (1, 32, 8, 1, 1000, 128), (20, 16, 8, 2, 161, 64), (1, 8, 1, 2, 5000, 128)])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("split", [False, True])
def test_decode_rows(ops, gpu, B, Hq, Hkv, L, Lk, D, masked, split):  # noqa: F811
    print("case decode rows", B, Hq, Hkv, L, Lk, D, masked, split, flush=True)
    g = gen(321)
    q = torch.randn(B, Hq, L, D, generator=g).bfloat16()
    k = torch.randn(B, Hkv, Lk, D, generator=g).bfloat16()
    v = torch.randn(B, Lk, Hkv, D, generator=g).bfloat16().transpose(1, 2)          # strided, as a projection leaves it
    bias = None
    if masked:
        keep = (torch.rand(B, Lk, generator=g) < 0.7).float()
        keep[:, 0] = 1.0
        bias = (1.0 - keep) * -1e4
    rep = Hq // Hkv
    s = q.float() @ k.float().repeat_interleave(rep, 1).transpose(-1, -2) * D ** -0.5
    if bias is not None:
        s = s + bias[:, None, None, :]
    visible = torch.arange(Lk)[None, :] <= torch.arange(L)[:, None] + Lk - L
    s = s.masked_fill(~visible, float("-inf"))
    ref = (torch.softmax(s, -1) @ v.float().repeat_interleave(rep, 1)).transpose(1, 2).reshape(B, L, Hq * D)
    out, lse = ops.causal_attention(q.to(gpu), k.to(gpu), v.to(gpu), return_lse=True,
                                    key_bias=None if bias is None else bias.to(gpu), split_keys=split)
    assert rel_err(out, ref) <= BF16_TOL
    assert (lse.cpu() - torch.logsumexp(s, -1)).abs().max().item() <= 1e-3      # bf16 products: scores to 1e-3 at |s| < 8
    # keys behind the last one, here another tensor's rows, are not read into the result
    big = torch.full((B, Hkv, Lk + 64, D), float("nan"), dtype=torch.bfloat16, device=gpu)
    big[:, :, :Lk] = k.to(gpu)
    again = ops.causal_attention(q.to(gpu), big[:, :, :Lk], v.to(gpu), key_bias=None if bias is None else bias.to(gpu),
                                 split_keys=split)
    assert torch.equal(again, out)
