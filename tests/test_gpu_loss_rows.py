"""Cross-entropy over rows that start at every alignment (head, whole vectors, tail), over more than one register tile, with
masked and not-a-number logits; host arrays sent with a launch."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,V,shift", [(9, 1, 0), (9, 7, 3), (11, 15, 1), (5, 4097, 5), (3, 33001, 2), (2, 70003, 7)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_of_every_alignment(gpu, T, V, shift, dtype):
    print("case loss rows", T, V, shift, dtype, flush=True)
    from adaptivetrainingsystem_amd.training import FusedLoss
    g = torch.Generator().manual_seed(5)
    flat = (torch.randn(T * V + shift, generator=g) * 3).to(dtype).to(gpu)
    z = flat[shift:].view(T, V).detach().requires_grad_()          # gradient buffer and logits differ in alignment
    if V > 8:
        with torch.no_grad():
            z[0, 1:] = float("-inf")                               # whole threads see masked elements only
            z[1, ::3] = float("-inf")
    labels = torch.randint(0, V, (T,), generator=g)
    labels[0], labels[1] = 0, 1 % V
    out = FusedLoss()(z, labels.to(gpu))
    out["loss"].backward()
    ref = z.detach().double().cpu().requires_grad_()
    loss = torch.nn.functional.cross_entropy(ref, labels)
    loss.backward()
    # sums of float32 terms and of float32 token losses: 1e-6 of the largest of them
    assert abs(out["loss"].item() - loss.item()) <= 2e-6 * max(1.0, loss.item())
    assert out["accuracy"].item() == pytest.approx((ref.argmax(-1) == labels).double().mean().item(), abs=1e-6)
    err = (z.grad.double().cpu() - ref.grad).abs().max().item() / ref.grad.abs().max().clamp(min=1e-30).item()
    assert err <= (1e-5 if dtype == torch.float32 else 2 ** -8)    # bfloat16: half an ulp of the stored gradient


@pytest.mark.parametrize("V", [40, 4099, 32000])
def test_nan_is_not_lost_among_masked_logits(gpu, V):
    from adaptivetrainingsystem_amd.training import FusedLoss
    z = torch.full((2, V), float("-inf"), device=gpu)
    z[:, 0] = 1.0
    z[1, V - 1] = float("nan")
    out = FusedLoss()(z, torch.zeros(2, dtype=torch.int64, device=gpu))
    assert out["loss"].item() == 5.0                               # 0 for the first token, the substitute 10 for the second


@pytest.mark.parametrize("V", [40, 1000, 4099, 32000])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_masks_of_the_lowest_value(gpu, V, dtype):
    """Logits masked with the type's lowest value, in part of a row and in all of it, and logits of the highest."""
    from adaptivetrainingsystem_amd.training import FusedLoss
    low, high = torch.finfo(dtype).min, torch.finfo(dtype).max
    z = torch.randn(4, V, generator=torch.Generator().manual_seed(8)).to(dtype)
    z[0, 3:] = low                                                 # whole threads see masked elements only
    z[1, :-2] = low
    z[2] = low
    z[3, ::2] = high
    labels = torch.tensor([1, V - 1, 5, 4])
    ref = torch.nn.functional.log_softmax(z.double(), dim=-1)
    z = z.to(gpu).requires_grad_()
    for t in range(4):
        z.grad = None
        out = FusedLoss()(z[t:t + 1], labels[t:t + 1].to(gpu))
        out["loss"].backward()
        if t < 2:
            want = -ref[t, labels[t]].item()
            assert abs(out["loss"].item() - want) <= 2e-6 * max(1.0, want)
        # at the ends of the range the float32 log-sum-exp has no room for log(V): the loss is 0 and every probability 1
        p = ref[t].exp() if t < 2 else (z[t].detach().double().cpu() == (low if t == 2 else high)).double()
        p[labels[t]] -= 1.0
        err = (z.grad[t].double().cpu() - p).abs().max().item() / p.abs().max().item()
        assert err <= (1e-5 if dtype == torch.float32 else 2 ** -8), (t, err)


def test_upload(gpu):
    from adaptivetrainingsystem_amd import _lib
    lib = _lib.load()
    n = lib.ats_upload_max_bytes()
    host = (ctypes.c_uint8 * n)(*[(7 * i) % 251 for i in range(n)])
    dst = torch.zeros(n + 16, dtype=torch.uint8, device=gpu)
    for bytes_ in (0, 8, 520, n):
        dst.zero_()
        assert lib.ats_upload(dst.data_ptr(), host, bytes_, torch.cuda.current_stream().cuda_stream) == 0
        want = torch.zeros(n + 16, dtype=torch.uint8)
        want[:bytes_] = torch.tensor(list(host[:bytes_]), dtype=torch.uint8)
        assert torch.equal(dst.cpu(), want)
    assert lib.ats_upload(dst.data_ptr(), host, n + 8, None) != 0 and lib.ats_upload(dst.data_ptr(), host, 12, None) != 0
    assert lib.ats_upload(dst.data_ptr() + 4, host, 8, None) != 0


def test_many_gradients(gpu):
    """More tensors than one launch's arguments hold."""
    from adaptivetrainingsystem_amd.training import FusedGradClip
    g = torch.Generator().manual_seed(6)
    grads = [torch.randn(1 + (i * 37) % 500, generator=g) for i in range(700)]
    norm = FusedGradClip().norm_and_clip([x.to(gpu) for x in grads], 1.0)
    ref = torch.cat(grads).double().norm().item()
    assert abs(norm.item() - ref) <= 1e-5 * ref
