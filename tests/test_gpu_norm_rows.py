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
