"""Normalisation with a workgroup per row: the ends of its ranges of rows and of row lengths, rows that fill no wave evenly."""
import pytest
import torch

from tests.test_gpu_parity import A, gen, ops  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,H", [(torch.bfloat16, 520), (torch.bfloat16, 1024), (torch.bfloat16, 2048), (torch.bfloat16, 2056),
                                     (torch.bfloat16, 4096), (torch.bfloat16, 8192), (torch.float32, 260), (torch.float32, 1024),
                                     (torch.float32, 2048), (torch.float32, 2052), (torch.float32, 4096)])
@pytest.mark.parametrize("rows", [1, 3, 512, 513, 4096, 4097])
@pytest.mark.parametrize("wdtype", [None, torch.float32, torch.bfloat16])
def test_norm_of_long_and_few_rows(ops, gpu, dtype, H, rows, wdtype):  # noqa: F811
    print("case norm rows", dtype, H, rows, wdtype, flush=True)
    if rows > 600 and wdtype != torch.float32:
        rows = 600
    x = (torch.randn(rows, H, generator=gen(H)) * 1.3).to(dtype)
    w = None if wdtype is None else (1 + 0.1 * torch.randn(H, generator=gen(H + 1))).to(wdtype)
    got = ops.rmsnorm(x.to(gpu), None if w is None else w.to(gpu)).cpu().double()
    xd = x.double()
    ref = xd * torch.rsqrt((xd * xd).mean(-1, keepdim=True) + 1e-6) * (1.0 if w is None else w.double())
    # the root is good to some units of 6e-8, the result is rounded once to its type
    assert ((got - ref).abs() <= ref.abs() * (1e-6 + (2.0 ** -8 if dtype == torch.bfloat16 else 0.0))).all()


# both sides of every change of kernel: rows of a wave each, few or long rows of a workgroup each
@pytest.mark.parametrize("dtype,H,wdtype,few,many", [(torch.bfloat16, 1024, torch.float32, 3, 4097), (torch.bfloat16, 2048, torch.bfloat16, 4096, 4097),
                                                     (torch.bfloat16, 4096, torch.float32, 1024, 1025), (torch.float32, 512, None, 512, 513),
                                                     (torch.float32, 1028, torch.float32, 9, 513), (torch.float32, 2048, torch.float32, 512, 2100)])
def test_bits_of_a_row_do_not_depend_on_the_number_of_rows(ops, gpu, dtype, H, wdtype, few, many):  # noqa: F811
    print("case norm row bits", dtype, H, wdtype, few, many, flush=True)
    x = (torch.randn(many, H, generator=gen(H)) * 1.3).to(dtype).to(gpu)
    w = None if wdtype is None else (1 + 0.1 * torch.randn(H, generator=gen(H + 1))).to(wdtype).to(gpu)
    assert torch.equal(ops.rmsnorm(x[:few], w), ops.rmsnorm(x, w)[:few])


@pytest.mark.parametrize("H", [516, 1024, 2048, 2052, 4096])
@pytest.mark.parametrize("rows", [1, 64, 600])
def test_squares_are_added_in_the_order_of_one_wave(ops, gpu, H, rows):  # noqa: F811
    """Lane l of a wave adds up the 16-byte vectors l, l + 64, .. one after another.  One lane's elements are 4096, 1, 1, ..: behind
    2^24 every 1 is rounded away (to even), while in any other grouping the ones meet first and count."""
    print("case norm order", H, rows, flush=True)
    x = torch.zeros(rows, H)
    v = torch.arange(H) // 4
    for r in range(rows):
        lane = r * 7 % min(64, H // 4)
        x[r, v % 64 == lane] = 1.0
        x[r, 4 * lane] = 4096.0
    y = ops.rmsnorm(x.to(gpu), None).cpu().double()
    want = x.double() / (2.0 ** 24 / H + 1e-6) ** 0.5
    # division, root, reciprocal and product: a unit of 2^-23 at most each and half of one
    assert ((y - want).abs() <= want * 2.5 * 2.0 ** -23).all()


# float32 weights: workgroups of one row below 1024 rows (1025 of shorter ones), of two and more from there, of as many as 1024 of them need
@pytest.mark.parametrize("H,many", [(8192, 1024), (5640, 1023), (4104, 1025), (4104, 2049), (5120, 3073)])
def test_rows_that_share_their_weights(ops, gpu, H, many):  # noqa: F811
    print("case norm shared weights", H, many, flush=True)
    x = (torch.randn(many, H, generator=gen(H)) * 1.3).bfloat16().to(gpu)
    w = (1 + 0.1 * torch.randn(H, generator=gen(H + 1))).to(gpu)
    assert torch.equal(ops.rmsnorm(x, w), torch.cat([ops.rmsnorm(part, w) for part in x.split(500)]))
