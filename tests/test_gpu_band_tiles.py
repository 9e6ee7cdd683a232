"""Grouped products of groups with some dozens of rows, and of one group with up to a few hundred, on the band tiles (GPU).

Bound: a result is a float32 sum of K products of bfloat16 operands, at most K * 2^-24 * sum |a||w| off (the SwiGLU epilogue's
factor is below 1.1 |u| with unit-sized g), and rounded once to bfloat16 (2^-8 of its value); float32 results only have the first.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")
    return torch.device("cuda")


STREAM, SMALL, BAND, ROWS128, ROWS256, ONCE = range(6)      # ats_grouped_gemm_route


def _route(E, rows, N, K, slices=1, swiglu=0, out=torch.bfloat16):
    from adaptivetrainingsystem_amd import _lib
    return _lib.load().ats_grouped_gemm_route(E, rows, N, K, slices, swiglu, _lib.ATS_F32 if out == torch.float32 else _lib.ATS_BF16)


def _groups(counts, N, K, ldb, seed):
    g = torch.Generator().manual_seed(seed)
    w = [(torch.randn(N, ldb, generator=g) * 0.05).bfloat16() for _ in counts]
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    return g, w, off


def _device(counts, off, gpu):
    return torch.tensor(off[:-1], device=gpu), torch.tensor(counts, dtype=torch.int32, device=gpu)


def _check(got, ref, mag, K, rounded=True):
    bound = K * 2.0 ** -24 * mag + (2.0 ** -8 * ref.abs() if rounded else 0) + 1e-30
    assert ((got.double().cpu() - ref).abs() <= bound).all()


# heights of 32, 64, 96 and 128 rows and their edges, groups of two tiles, without rows; one, two and more slabs; a ragged N
@pytest.mark.parametrize("counts,N,K", [([31, 32, 33, 0, 64, 65] * 7, 1000, 64), ([96, 97, 127, 1] * 16, 1032, 128), ([128, 129, 0, 2] * 16, 1032, 192),
                                        ([1, 2, 0, 3] * 16, 1096, 448), ([40] * 63 + [400], 1024, 320)])
@pytest.mark.parametrize("gather", [False, True])
def test_groups(gpu, counts, N, K, gather):
    from adaptivetrainingsystem_amd import ops
    print("case band groups", len(counts), N, K, gather, flush=True)
    assert _route(len(counts), sum(counts), N, K) == BAND
    ldb = K + 8
    g, w, off = _groups(counts, N, K, ldb, N + K)
    n = int(off[-1])
    a = torch.randn(n, K + 16, generator=g).bfloat16()
    idx = torch.randint(0, 2 * n, (n,), generator=g, dtype=torch.int32) if gather else None
    start, count = _device(counts, off, gpu)
    wd = [t.to(gpu) for t in w]
    ptrs = torch.tensor([t.data_ptr() for t in wd], device=gpu)
    got = ops.grouped_gemm_nt(ptrs, ldb, N, start, count, n, n, N, K, a=a.to(gpu)[:, :K], lda=K + 16, a_rows=None if idx is None else idx.to(gpu),
                              a_row_div=2)
    rows = a[:, :K].double() if idx is None else a[:, :K].double()[(idx // 2).long()]
    for e in range(len(counts)):
        s = slice(off[e], off[e + 1])
        _check(got[s], rows[s] @ w[e][:, :K].double().T, rows[s].abs() @ w[e][:, :K].double().abs().T, K)


# (band tiles of all four heights; the last three on the 256-row tile whose supertiles begin K an eighth apart: one slab, fewer and
# more than eight, groups of two tiles)
@pytest.mark.parametrize("counts,I,K,route", [([31, 33, 64, 0, 65] * 4, 1000, 64, BAND), ([97, 128, 1, 96] * 8, 1032, 192, BAND),
                                              ([12, 129, 0, 20] * 8, 1096, 576, BAND), ([200, 256, 0, 300] * 2, 131080, 64, ONCE),
                                              ([223, 224, 225, 200], 52432, 320, ONCE), ([130, 255, 257, 1, 410], 11048, 1216, ONCE)])
def test_gate_up(gpu, counts, I, K, route):
    from adaptivetrainingsystem_amd import ops
    print("case band gate/up", len(counts), I, K, flush=True)
    assert _route(len(counts), sum(counts), I, K, swiglu=1) == route
    g = torch.Generator(device=gpu).manual_seed(I + K)
    w = [(torch.randn(2 * I, K, generator=g, device=gpu) * 0.05).bfloat16() for _ in counts]
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    n = int(off[-1])
    x = torch.randn(n // 2 + 1, K, generator=g, device=gpu).bfloat16()
    idx = torch.randint(0, n, (n,), generator=g, device=gpu, dtype=torch.int32)
    start, count = _device(counts, off, gpu)
    got = ops.grouped_gateup_swiglu(x, ops.weight_pointer_table(w), start, count, n, n, K, I, a_rows=idx, a_row_div=2)
    rows = x.double()[(idx // 2).long()]
    for e in range(len(counts)):
        s = slice(off[e], off[e + 1])
        gu, mag = rows[s] @ w[e].double().T, rows[s].abs() @ w[e].double().abs().T
        gate, up = gu[:, :I], gu[:, I:]
        ref = gate * torch.sigmoid(gate) * up
        # (the exponential and the division of the sigmoid: 2^-20 of the value)
        bound = 1.1 * mag[:, :I] * up.abs() + gate.abs() * mag[:, I:] + 2.0 ** 4 / K * ref.abs()
        assert ((got[s].double() - ref).abs() <= K * 2.0 ** -24 * bound + 2.0 ** -8 * ref.abs() + 1e-30).all()


@pytest.mark.parametrize("rows,I,K,route", [(60, 1400, 2048, BAND), (200, 1400, 2048, ONCE)])
def test_gate_up_sums_do_not_depend_on_other_groups(gpu, rows, I, K, route):
    """Band tiles and 256-row tiles that begin K out of step: an expert's rows have the same bits whatever the others get."""
    from adaptivetrainingsystem_amd import ops
    E = 24
    assert _route(E, E * rows, I, K, swiglu=1) == route
    g = torch.Generator(device=gpu).manual_seed(9)
    w = [(torch.randn(2 * I, K, generator=g, device=gpu) * 0.05).bfloat16() for _ in range(E)]
    x = torch.randn(E * rows, K, generator=g, device=gpu).bfloat16()
    ptrs = ops.weight_pointer_table(w)
    start = (torch.arange(E, dtype=torch.int32) * rows).to(gpu)
    out = []
    for none in ([], list(range(8)), [1, 9, 10, 11, 20]):
        count = torch.tensor([0 if e in none else rows for e in range(E)], dtype=torch.int32, device=gpu)
        out.append((none, ops.grouped_gateup_swiglu(x, ptrs, start, count, E * rows, E * rows, K, I).view(E, rows, I)))
    for none, one in out[1:]:
        for e in range(E):
            assert e in none or torch.equal(one[e], out[0][1][e]), e


# (33 and 65 rows: tiles of 64 rows with a remainder, 97 and 128 of 128 rows; the others keep the small and the 256-row tiles)
@pytest.mark.parametrize("T,N,K,route", [(33, 1032, 512, SMALL), (33, 14336, 1024, BAND), (64, 4096, 1024, SMALL), (65, 1032, 4096, SMALL), (65, 6144, 512, BAND),
                                         (96, 2056, 2048, SMALL), (97, 6144, 1024, BAND), (128, 6144, 1024, BAND), (129, 4104, 1024, BAND), (200, 2056, 1024, BAND),
                                         (200, 1032, 2048, BAND), (256, 4104, 1024, BAND), (257, 2048, 512, BAND), (300, 2056, 64, BAND), (640, 1032, 1024, BAND),
                                         (1000, 2048, 2048, BAND)])
def test_one_group(gpu, T, N, K, route):
    """A linear layer, plain or in slices of K by the rule; up to 256 rows every slice as well, which run on the band tiles."""
    from adaptivetrainingsystem_amd import ops
    print("case band one group", T, N, K, ops.linear_k_splits(T, N, K, torch.bfloat16), flush=True)
    assert _route(1, T, N, K) == route and (T > 256 or all(_route(1, T, N, K, s, out=torch.float32) == BAND for s in (2, 4)))
    g = torch.Generator().manual_seed(T + N)
    x, w = torch.randn(T, K, generator=g).bfloat16(), (torch.randn(N, K, generator=g) * 0.05).bfloat16()
    ref, mag = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    xd, wd = x.to(gpu), w.to(gpu)
    _check(ops.linear_nt(xd, wd), ref, mag, K)
    if T <= 256:
        start, count = torch.zeros(1, dtype=torch.int32, device=gpu), torch.full((1,), T, dtype=torch.int32, device=gpu)
        for s in (2, 4):
            parts = ops.grouped_down_splitk(xd, ops.weight_pointer_table([wd]), start, count, T, N, K, s)
            for i in range(s):
                k = slice(i * K // s, (i + 1) * K // s)
                _check(parts[i], x[:, k].double() @ w[:, k].double().T, x[:, k].double().abs() @ w[:, k].double().abs().T, K // s, rounded=False)


# one float32 chain of K is 4.7e-7, 7.6e-7 and 4.0e-7 off here (standard normal operands), four of them 2.2e-7, 3.7e-7 and 1.9e-7
@pytest.mark.parametrize("E,rows,N,K,most", [(16, 48, 2048, 5632, 3.2e-7), (8, 32, 4096, 14336, 5.3e-7), (1, 150, 6144, 4096, 2.8e-7)])
def test_float32_results_keep_four_chains(gpu, E, rows, N, K, most):
    from adaptivetrainingsystem_amd import ops
    g = torch.Generator(device=gpu).manual_seed(E)
    w = [torch.randn(N, K, generator=g, device=gpu).bfloat16() for _ in range(E)]
    x = torch.randn(E * rows, K, generator=g, device=gpu).bfloat16()
    start, count = (torch.arange(E, dtype=torch.int32) * rows).to(gpu), torch.full((E,), rows, dtype=torch.int32, device=gpu)
    got = ops.grouped_gemm_nt(ops.weight_pointer_table(w), K, N, start, count, E * rows, E * rows, N, K, a=x, out_dtype=torch.float32)
    ref = torch.cat([x[e * rows:(e + 1) * rows].double() @ w[e].double().T for e in range(E)])
    assert (got.double() - ref).norm() <= most * ref.norm()


@pytest.mark.parametrize("counts,H,I,S", [([40, 30, 33, 0, 96, 1, 70, 128] * 2, 2056, 1024, 2), ([25, 64, 65, 129], 4104, 2048, 4)])
def test_slices_of_groups(gpu, counts, H, I, S):
    from adaptivetrainingsystem_amd import ops
    print("case band slices", len(counts), H, I, S, flush=True)
    assert _route(len(counts), sum(counts), H, I, S, out=torch.float32) == BAND
    g, w, off = _groups(counts, H, I, I, H + I)
    n = int(off[-1])
    h = torch.randn(n, I, generator=g).bfloat16()
    start, count = _device(counts, off, gpu)
    wd = [t.to(gpu) for t in w]
    parts = ops.grouped_down_splitk(h.to(gpu), torch.tensor([t.data_ptr() for t in wd], device=gpu), start, count, n, H, I, S)
    for i in range(S):
        k = slice(i * I // S, (i + 1) * I // S)
        for e in range(len(counts)):
            s = slice(off[e], off[e + 1])
            _check(parts[i][s], h[s, k].double() @ w[e][:, k].double().T, h[s, k].double().abs() @ w[e][:, k].double().abs().T, I // S, rounded=False)
