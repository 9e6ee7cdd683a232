"""Down projections of groups of 21-256 rows cut along K on the direct-to-LDS tile."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# rows per group around 16-row fragments, 32-row steps and one full tile, a group without rows; ragged N; slices of one slab
# and of several; at least 128 tiles, so that the tile under test is the one that runs
@pytest.mark.parametrize("counts,H,I,S", [([33, 1, 0, 200, 256, 17, 64, 127], 2048, 1024, 2), ([257, 30, 31, 32], 2056, 512, 8),
                                          ([40, 40, 41, 39, 500, 1, 1, 12], 4096, 320, 5), ([21, 22], 4104, 256, 4)])
def test_sliced_down_projection(gpu, counts, H, I, S):
    print("case sliced down", counts, H, I, S, flush=True)
    from adaptivetrainingsystem_amd import ops
    g = torch.Generator().manual_seed(sum(counts))
    E, rows = len(counts), sum(counts)
    h = (torch.randn(rows, I, generator=g) * 0.5).bfloat16()
    wd = [(torch.randn(H, I, generator=g) * 0.05).bfloat16() for _ in range(E)]
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    start = torch.tensor(off[:-1], dtype=torch.int32, device=gpu)
    count = torch.tensor(counts, dtype=torch.int32, device=gpu)
    wd_gpu = [w.to(gpu) for w in wd]
    parts = ops.grouped_down_splitk(h.to(gpu), ops.weight_pointer_table(wd_gpu), start, count, rows, H, I, S).cpu()
    K = I // S
    for s in range(S):
        ref = torch.cat([h[off[e]:off[e + 1], s * K:(s + 1) * K].double() @ wd[e][:, s * K:(s + 1) * K].double().T for e in range(E)])
        # float32 sums of K exact products: errors of a few units of 6e-8 of the sum of their sizes
        bound = 4e-7 * (h[:, s * K:(s + 1) * K].double().abs().sum(1).max() * wd[0].abs().max().double())
        assert (parts[s].double() - ref).abs().max() <= bound


# slices of 512 columns and more, where an estimate chooses between that tile and the small ones: a few rows (small, 32-row tiles,
# small), more rows of few (large) and of more groups (large)
@pytest.mark.parametrize("counts,H,I,S", [([40, 56], 1000, 16384, 16), ([21, 24, 0, 33], 1032, 8192, 8), ([100, 156], 1000, 16384, 16),
                                          ([90, 0, 129, 64, 33, 1, 128, 200], 1032, 4096, 8), ([70, 65], 1000, 16384, 8),
                                          ([230, 100, 140, 170], 1032, 8192, 8)])
def test_sliced_down_projection_on_the_estimated_tile(gpu, counts, H, I, S):
    test_sliced_down_projection(gpu, counts, H, I, S)


# 44, 175 and 224 rows per expert; up to 192 the plain launch is the faster one (192 rows 25 us, in four slices 35; 224 rows 48 and 38)
@pytest.mark.parametrize("T", [176, 700, 896])
def test_layer_with_sliced_down_projection(gpu, T):
    """The layer whose rule chooses these slices against the stages in float64."""
    print("case layer sliced", T, flush=True)
    from adaptivetrainingsystem_amd import ops
    from adaptivetrainingsystem_amd import workloads as W
    from oracle import sparse_layer_oracle as O
    ov = {"batch": 1, "seq": T, "hidden": 1024, "num_experts": 8, "top_k": 2, "intermediate": 2048, "dtype": torch.bfloat16}
    w = W.make_moe_workload("c1_cpu_reference", device="cpu", overrides=ov)
    wg = W.make_moe_workload("c1_cpu_reference", device=gpu, overrides=ov)
    layer = W.build_layer(wg, "none")
    assert ops.down_k_splits(8, 2 * T, 1024, 2048, torch.bfloat16) == (4 if T == 896 else 1)
    with torch.no_grad():
        out, _ = layer(wg.x)
    ref = O.moe_forward_nocap(w.x.float(), w.gate.float(), [t.float() for t in w.gate_up], [t.float() for t in w.down], k=2,
                              logits_override=layer.last_plan["logits"].cpu())
    ref = ref["out"] if isinstance(ref, dict) else ref[0]
    err = (out.cpu().double() - ref.double().view(out.shape)).norm() / ref.double().norm()
    assert err <= 1.2e-2      # h and y are rounded to bfloat16 (2^-9 each), measured 3e-3


# the same against weights stored [K][N]: columns that are no multiple of the tile, slices of one slab and of several, groups
# on both sides of a fragment, of one tile and of two, without rows
@pytest.mark.parametrize("counts,N,K,S", [([33, 1, 0, 200, 256, 17, 64, 127], 264, 1024, 2), ([257, 30, 31, 32], 72, 512, 8),
                                          ([40, 500, 1, 12], 1000, 320, 5), ([5], 520, 128, 1), ([190, 16, 0, 15], 8, 192, 1)])
def test_sliced_product_with_k_major_weights(gpu, counts, N, K, S):
    print("case sliced k-major", counts, N, K, S, flush=True)
    from adaptivetrainingsystem_amd import ops
    g = torch.Generator().manual_seed(sum(counts) + N)
    E, rows, ldb = len(counts), sum(counts), N + 8
    a = (torch.randn(rows, K, generator=g) * 0.5).bfloat16()
    w = [(torch.randn(K, ldb, generator=g) * 0.05).bfloat16() for _ in range(E)]
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    start = torch.tensor(off[:-1], dtype=torch.int32, device=gpu)
    count = torch.tensor(counts, dtype=torch.int32, device=gpu)
    w_gpu = [t.to(gpu) for t in w]
    out = ops.grouped_gemm_nn_sliced(ops.weight_pointer_table(w_gpu), ldb, start, count, rows, rows, N, K, a.to(gpu), S).cpu()
    n = K // S
    for s in range(S):
        ref = torch.cat([a[off[e]:off[e + 1], s * n:(s + 1) * n].double() @ w[e][s * n:(s + 1) * n, :N].double() for e in range(E)])
        bound = 4e-7 * (a[:, s * n:(s + 1) * n].double().abs().sum(1).max() * max(t.abs().max().double() for t in w))
        if S == 1:
            bound = bound + 2.0 ** -8 * ref.abs().max()      # one rounding to bfloat16
        assert ((out if S == 1 else out[s]).double() - ref).abs().max() <= bound


def test_rule_of_k_major_slices(gpu):
    from adaptivetrainingsystem_amd import ops
    rule = lambda *a: ops.grouped_gemm_nn_slices(*a, torch.bfloat16)
    assert rule(8, 650, 4096, 28672, 4096) == 2 and rule(8, 650, 14336, 4096, 14336) == 1
    assert rule(8, 8 * 300, 4096, 28672, 4096) == 1 and rule(8, 8 * 200, 4096, 28672, 4096) >= 1
    assert rule(8, 650, 4100, 28672, 4100) == 0 and rule(8, 650, 4096, 28672 + 32, 4096) == 0 and rule(8, 0, 4096, 4096, 4096) == 0
    assert ops.grouped_gemm_nn_slices(8, 650, 4096, 28672, 4096, torch.float32) == 0
