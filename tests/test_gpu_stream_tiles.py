"""Grouped products of a few rows per group (the weight-streaming tiles) against float64: one row up to the last row of a
tile and beyond it, groups without rows, output columns that do not fill a tile, K from one 16-byte piece over ragged
256-byte pieces to several pieces per wave, four and eight waves, panels of 16 and 32 weight rows."""
import pytest
import torch

from tests.test_gpu_parity import A, BF16_TOL, F32_TOL, gen, ops, rel_err, same_bits  # noqa: F401

pytestmark = pytest.mark.gpu

#        rows per group            N     K
CASES = [([1], 32, 8), ([5, 0, 17], 40, 136), ([16, 32, 33, 0, 2], 72, 1000), ([32], 4096, 4160), ([1, 2], 1032, 8200),
         ([20, 15, 40], 264, 8192), ([3] * 20, 2048, 1408), ([31, 1, 29], 136, 16384), ([9], 3000, 2048)]


@pytest.mark.parametrize("counts,N,K", CASES)
@pytest.mark.parametrize("dtype,out_dtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16),
                                             (torch.bfloat16, torch.float32)])
def test_stream_tiles_plain(ops, gpu, counts, N, K, dtype, out_dtype):  # noqa: F811
    print("case stream tiles", counts, N, K, dtype, out_dtype, flush=True)
    g = gen(311)
    E, n = len(counts), sum(counts)
    w = [(torch.randn(N, K, generator=g) * 0.1).to(dtype).to(gpu) for _ in range(E)]
    count = torch.tensor(counts, dtype=torch.int32)
    start = (torch.cumsum(count, 0) - count).to(torch.int32).to(gpu)
    count = count.to(gpu)
    a = torch.randn(n + 3, K, generator=g).to(dtype).to(gpu)
    src = torch.randint(0, 2 * (n + 3), (n,), generator=g).to(torch.int32).to(gpu)
    tab = ops.weight_pointer_table(w)
    out = ops.grouped_gemm_nt(tab, K, N, start, count, n + 2, n, N, K, a=a, out_dtype=out_dtype)
    gathered = ops.grouped_gemm_nt(tab, K, N, start, count, n + 2, n, N, K, a=a, a_rows=src, a_row_div=2, out_dtype=out_dtype)
    copied = ops.grouped_gemm_nt(tab, K, N, start, count, n + 2, n, N, K, a=a[(src // 2).long()].contiguous(),
                                 out_dtype=out_dtype)
    assert same_bits(gathered[:n], copied[:n])
    off, tol = 0, F32_TOL if dtype == torch.float32 else BF16_TOL
    for e, c in enumerate(counts):
        if c:
            assert rel_err(out[off:off + c], a[off:off + c].cpu().double() @ w[e].cpu().double().T) <= tol
        off += c
    # rows outside the groups are not written
    lib = __import__("adaptivetrainingsystem_amd._lib", fromlist=["load"]).load()
    buf = torch.full((n + 2, N), 7.0, dtype=out_dtype, device=gpu)
    tag = lambda t: 0 if t == torch.float32 else 1
    assert lib.ats_grouped_gemm_nt(a.data_ptr(), None, K, n + 3, None, 1, tab.data_ptr(), K, N, buf.data_ptr(), N,
                                   start.data_ptr(), count.data_ptr(), None, E, n, N, K, tag(dtype), tag(out_dtype),
                                   None) == 0
    torch.cuda.synchronize()
    assert torch.all(buf[n:] == 7.0) and same_bits(buf[:n], out[:n])


@pytest.mark.parametrize("counts,I,H", [([1], 32, 8), ([5, 0, 17], 40, 136), ([16, 32, 0, 20], 72, 1000), ([32], 1032, 4096),
                                        ([33, 2, 7], 200, 2048)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_stream_tiles_swiglu(ops, gpu, counts, I, H, dtype):  # noqa: F811
    print("case stream tiles swiglu", counts, I, H, dtype, flush=True)
    g = gen(312)
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


@pytest.mark.parametrize("T,k,mode,onto,I", [(1, 2, "none", False, 136), (3, 6, "none", False, 136), (40, 2, "fcfs", False, 136),
                                             (64, 2, "fcfs", True, 136), (300, 3, "fcfs", True, 136), (700, 2, "none", False, 136),
                                             (100, 4, "none", False, 2048), (300, 3, "fcfs", False, 2048)])
def test_native_layer_call_equals_the_stages(A, gpu, T, k, mode, onto, I):  # noqa: F811
    """The inference pass queued by one native call: bits, routing tensors and auxiliary loss of the stages run one by one
    (which a stage timer selects), with the down projection whole and in slices of K."""
    from adaptivetrainingsystem_amd import ops as O
    from adaptivetrainingsystem_amd import profiling
    from adaptivetrainingsystem_amd import workloads as W
    print("case native layer", T, k, mode, onto, I, flush=True)
    ov = {"batch": 1, "seq": T, "hidden": 256, "num_experts": 8, "top_k": k, "intermediate": I, "dtype": torch.bfloat16}
    w = W.make_moe_workload("c1_cpu_reference", device=gpu, overrides=ov)
    layer = W.build_layer(w, mode)
    base = torch.randn(2 * T, 256, generator=gen(313)).bfloat16().to(gpu)
    rows_to = torch.randperm(2 * T, generator=gen(314))[:T].to(torch.int32).to(gpu)
    run = lambda: layer(w.x, add_onto=(base.clone(), rows_to)) if onto else layer(w.x)
    got, got_aux = run()
    plan = layer.last_plan
    rows = min(T * k, 8 * plan["capacity"])
    assert (O.down_k_splits(8, rows, 256, I, torch.bfloat16) > 1) == (I == 2048)
    layer.stage_timer = profiling.StageTimer()
    want, want_aux = run()
    assert same_bits(got, want) and torch.equal(got_aux, want_aux)
    ref = layer.last_plan
    assert plan["capacity"] == ref["capacity"] and set(ref) <= set(plan)
    for name in ("logits", "indices", "weights", "hist", "prob_colsum", "slot", "token_map", "kept", "offsets", "row_of", "aux"):
        assert torch.equal(plan[name], ref[name].view(plan[name].shape)), name
    n = int(ref["kept"].sum())
    assert torch.equal(plan["row_src"][:n], ref["row_src"][:n])


# panels dealt to the XCDs in one piece each (32 groups and more) or in chunks; more than 64 groups; tiles of 16 rows (up to 4 rows per
# group on average) with groups that need several
@pytest.mark.parametrize("counts,N,K", [([1] * 31, 40, 136), ([1] * 32, 40, 136), ([40] + [0] * 29 + [1] * 5, 72, 520), ([17, 16, 0, 1] + [0] * 6, 1032, 264),
                                        ([2, 0, 1] * 24, 264, 136), ([0] * 129 + [33], 72, 264), ([3, 0, 19] * 45, 40, 136)])
def test_stream_panels_of_many_groups(ops, gpu, counts, N, K):  # noqa: F811
    print("case stream panels", len(counts), sum(counts), N, K, flush=True)
    g = gen(313)
    E, n = len(counts), sum(counts)
    w = [(torch.randn(N, K, generator=g) * 0.1).bfloat16().to(gpu) for _ in range(E)]
    count = torch.tensor(counts, dtype=torch.int32)
    start = (torch.cumsum(count, 0) - count).to(torch.int32).to(gpu)
    a = torch.randn(n, K, generator=g).bfloat16().to(gpu)
    # (n + 5 rows at most: the launch may have more blocks than panels)
    out = ops.grouped_gemm_nt(ops.weight_pointer_table(w), K, N, start, count.to(gpu), n + 5, n + 5, N, K, a=a, out_dtype=torch.float32)
    off = 0
    for e, c in enumerate(counts):
        if c:
            assert rel_err(out[off:off + c], a[off:off + c].cpu().double() @ w[e].cpu().double().T) <= F32_TOL
        off += c
