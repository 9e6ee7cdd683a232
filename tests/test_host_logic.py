"""CPU-side checks: the C-ABI library loads and exports every declared symbol, the tile
schedule covers every tile exactly once, host-side integer logic, error behaviour without a GPU."""
import ctypes
import os
import re

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "ats_gfx950.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(ats_[a-z0-9_]+|[a-z_]+_launcher)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from adaptivetrainingsystem_amd import _lib
    assert _lib.is_built(), "build the library first: python -m adaptivetrainingsystem_amd.build"
    lib = _lib.load()
    names = _declared_symbols()
    assert len(names) >= 20
    for n in names:
        assert hasattr(lib, n), n
        assert n in _lib._SIGNATURES, f"{n} has no ctypes signature"
    assert lib.ats_version() >= 100
    assert set(_lib._SIGNATURES) == set(names)


def test_reference_launcher_names_are_exported_and_never_exit():
    """The four launcher names the reference's ctypes loader binds (cuda_opt_wrapper.py:98-108, 156-169,
    219-228, 337-344) exist with void returns; a bad argument leaves a status and a text, not an exit()."""
    from adaptivetrainingsystem_amd import _lib
    lib = _lib.load()
    raw = ctypes.CDLL(_lib.LIB_PATH)        # as the reference binds it: no argtypes, explicit ctypes wrappers
    for n in ("rms_norm_launcher", "rope_precompute_launcher", "rope_apply_launcher", "swiglu_launcher", "swiglu_fused_launcher",
              "fused_cross_entropy_accuracy_launcher", "fused_grad_clip_launcher"):      # training/cuda_kernels.py:60-78
        assert hasattr(raw, n), n
    raw.rms_norm_launcher(ctypes.c_void_p(0), ctypes.c_void_p(0), ctypes.c_void_p(0), ctypes.c_int(4), ctypes.c_int(0),
                          ctypes.c_float(1e-6), ctypes.c_void_p(0))
    assert lib.ats_legacy_last_status() == -1 and b"hidden" in lib.ats_last_error_string()
    raw.rope_apply_launcher(ctypes.c_void_p(0), ctypes.c_void_p(0), ctypes.c_void_p(0), ctypes.c_void_p(0),
                            ctypes.c_int(1), ctypes.c_int(1), ctypes.c_int(4), ctypes.c_int(7), ctypes.c_int(0),
                            ctypes.c_void_p(0))
    assert lib.ats_legacy_last_status() == -1           # odd head_dim
    raw.swiglu_launcher(ctypes.c_void_p(0), ctypes.c_void_p(0), ctypes.c_void_p(0), ctypes.c_int(0), ctypes.c_int(16),
                        ctypes.c_void_p(0))
    assert lib.ats_legacy_last_status() == 0            # nothing to do is not an error
    raw.rope_precompute_launcher(ctypes.c_void_p(0), ctypes.c_void_p(0), ctypes.c_int(8), ctypes.c_int(16),
                                 ctypes.c_float(10000.0), ctypes.c_void_p(0))
    assert lib.ats_legacy_last_status() == -1 and b"null" in lib.ats_last_error_string()


def test_argument_errors_return_codes_not_exits():
    from adaptivetrainingsystem_amd import _lib
    lib = _lib.load()
    # invalid arguments are rejected on the host before any device work
    assert lib.ats_rmsnorm_fwd(None, None, None, 4, 0, 1e-6, 0, 0, None) == -1
    assert b"hidden" in lib.ats_last_error_string()
    assert lib.ats_rmsnorm_fwd(None, None, None, 4, 8, 1e-6, 7, 0, None) != 0
    assert lib.ats_route_topk(None, 4, 8, 9, 1.0, 0, None, None, None, None, None, 0.01, None, 0, None) == -1
    assert lib.ats_dispatch_plan(None, 0, 4, 2, 5000, 3, None, None, None, None, None, None, None, None, None, 0,
                                 None) == -1
    assert lib.ats_rope_fwd(None, None, None, None, None, None, 4, 4, 1, 1, 1, 4, 7, 0, 0, 0, 0, 0, 0, 0, 0,
                            None) == -1       # odd head_dim
    assert lib.ats_select_topk_per_sequence(None, 1, 10000, 5, None, None) == -1
    # attention: head_dim outside {64, 128}, fewer keys than queries, query heads not a multiple of kv heads
    assert lib.ats_attention_fwd(None, None, 0, 0, None, 0, 96, 0, None, None, None, 1, 4, 2, 16, 16, 96, 0.1, None, 0, None) == -2
    assert b"head_dim" in lib.ats_last_error_string()
    assert lib.ats_attention_fwd(None, None, 0, 0, None, 0, 128, 0, None, None, None, 1, 4, 2, 16, 8, 128, 0.1, None, 0, None) == -1
    assert lib.ats_attention_fwd(None, None, 0, 0, None, 0, 128, 0, None, None, None, 1, 3, 2, 16, 16, 128, 0.1, None, 0, None) == -1
    assert lib.ats_attention_fwd(None, None, 0, 0, None, 0, 128, 0, None, None, None, 1, 4, 2, 16, 16, 128, 0.1, None, 0, None) == -1     # null pointers
    assert lib.ats_attention_fwd(None, None, 0, 0, None, 0, 128, 0, None, None, None, 0, 4, 2, 16, 16, 128, 0.1, None, 0, None) == 0      # empty batch
    assert lib.ats_attention_bwd(*([None] * 10), 1, 4, 2, 16, 8, 128, 0.1, None, 0, None) == -1
    assert lib.ats_attention_bwd(*([None] * 10), 1, 4, 2, 16, 16, 32, 0.1, None) == -2
    assert lib.ats_attention_delta(None, None, None, 1, 4, 16, 80, None) == -2
    assert lib.ats_attention_bwd_out(*([None] * 9), 0, 0, 0.0, 0, None, None, None, 1, 4, 2, 16, 16, 128, 0.1, None) == -1
    assert lib.ats_attention_bwd_out(*([None] * 9), 0, 0, 0.0, 0, None, None, None, 0, 4, 2, 16, 16, 128, 0.1, None) == 0
    # K slices: I must be k_splits whole slabs, and only weight-streaming sizes (<= 48 rows per expert)
    one = ctypes.c_void_p(16)
    assert lib.ats_grouped_down_splitk(one, one, one, one, one, 8, 128, 128, 4096, 14336, 3, 1, None) == -2
    assert b"slices" in lib.ats_last_error_string()
    assert lib.ats_grouped_down_splitk(one, one, one, one, one, 8, 4096, 4096, 4096, 14336, 2, 1, None) == -2   # 512 rows per expert
    assert lib.ats_grouped_down_splitk(one, one, one, one, one, 8, 128, 128, 4096, 14336, 0, 1, None) == -1
    assert lib.ats_sum_partials(one, 2, 10, one, 8, 1, None) == -1          # stride not a multiple of 4
    assert lib.ats_sum_partials(None, 2, 16, None, 0, 1, None) == 0         # nothing to add
    assert lib.ats_combine_partials(one, 2, 64, one, one, None, one, 4, 9, 64, 1, None) == -1   # k > 8
    assert lib.ats_route_topk_workspace(16384, 8) > 0
    assert lib.ats_dispatch_plan_workspace(16384, 2, 8) == (32768 // 256) * 8 * 4


@pytest.mark.parametrize("aligned", [0, 1])
@pytest.mark.parametrize("counts,BM,n_tiles,SM,SN,slices", [
    ([5120, 4000, 300, 0, 1, 256, 257, 77], 256, 112, 4, 8, 1),
    ([20, 16, 0, 3], 32, 112, 1, 32, 1),
    ([130, 90, 576, 1], 128, 11, 8, 4, 1),
    ([0, 0, 0], 128, 5, 4, 8, 1),
    ([1000] * 64, 128, 11, 4, 8, 1),
    ([384] * 70, 256, 11, 8, 4, 1),
    ([20, 16, 0, 3], 32, 32, 1, 32, 3),
    ([64, 33, 1], 64, 40, 1, 32, 2),
])
def test_tile_schedule_covers_each_tile_once(counts, BM, n_tiles, SM, SN, slices, aligned):
    from adaptivetrainingsystem_amd import _lib
    lib = _lib.load()
    rc = np.asarray(counts, dtype=np.int32)
    E = len(counts)
    blocks = lib.ats_debug_grid_blocks(int(rc.sum()) * slices, E * slices, BM, n_tiles, SM, SN, aligned)
    assert blocks % 256 == 0
    seen = {}
    out = np.zeros(4, dtype=np.int32)
    for b in range(blocks):
        if lib.ats_debug_decode_tile(b, rc.ctypes.data, E, BM, n_tiles, SM, SN, aligned, slices, out.ctypes.data):
            key = tuple(out.tolist())
            assert key not in seen, f"tile {key} given to blocks {seen[key]} and {b}"
            seen[key] = b
    expect = {(e, mt, nt, ks) for ks in range(slices) for e in range(E) for mt in range(-(-counts[e] // BM))
              for nt in range(n_tiles)}
    assert set(seen) == expect
    # blocks of one supertile land on one XCD (ids congruent mod 8) and cover SN neighbouring n-tiles of one band:
    # SM consecutive entries of the m-tile list (group 0's tiles, then group 1's, ...; a group is an expert or one
    # K slice of it; with `aligned` every group's tile count is rounded up to a multiple of SM)
    if expect:
        per = [-(-c // BM) for c in counts] * slices
        if aligned:
            per = [-(-t // SM) * SM for t in per]
        first = np.concatenate([[0], np.cumsum(per)])
        by_xcd = {}
        for key, b in seen.items():
            by_xcd.setdefault((b % 8, (b // 8) // 32), []).append(key)
        order = []
        for (xcd, li), keys in sorted(by_xcd.items(), key=lambda kv: kv[0][1] * 8 + kv[0][0]):
            pos = {int(first[ks * E + e]) + mt for e, mt, _, ks in keys}
            assert len({q // SM for q in pos}) == 1
            assert len({k[2] // SN for k in keys}) == 1
            if aligned:
                assert len({(k[0], k[3]) for k in keys}) == 1      # one expert's weight panels per supertile
            order.append((min(pos) // SM, keys[0][2] // SN))
        # supertiles go group by group (by the group a band starts in), n-group by n-group, band by band
        owner = lambda band: int(np.searchsorted(first, band * SM, side="right") - 1)
        assert order == sorted(order, key=lambda t: (owner(t[0]), t[1], t[0]))


def test_capacity_is_python_double_arithmetic():
    from adaptivetrainingsystem_amd import ops
    assert ops.expert_capacity(512, 2, 8, 1.25) == 160
    assert ops.expert_capacity(64, 2, 8, 1.25) == 20
    assert ops.expert_capacity(16384, 2, 8, 1.25) == 5120
    assert ops.expert_capacity(4096, 6, 64, 1.5) == 576
    assert ops.expert_capacity(512, 2, 8, 1.1) == 140


def test_no_cpu_fallback_and_module_surface():
    import adaptivetrainingsystem_amd as A
    from adaptivetrainingsystem_amd.workloads import LayerConfig
    with pytest.raises(A.AtsError):
        A.RMSNorm(16)(torch.randn(2, 16))
    with pytest.raises(A.AtsError):
        A.apply_rotary_pos_emb(torch.randn(1, 1, 4, 8), torch.randn(1, 1, 4, 8), torch.ones(4, 8), torch.zeros(4, 8))
    layer = A.MoEFFNLayer(LayerConfig(32, 64, 4, 2))
    with pytest.raises(A.AtsError):
        layer(torch.randn(1, 3, 32))
    # parameter names and shapes that checkpoints of the reference model carry
    sd = layer.state_dict()
    assert sd["gate.weight"].shape == (4, 32)
    assert sd["experts.0.gate_up_proj.weight"].shape == (128, 32)
    assert sd["experts.3.down_proj.weight"].shape == (32, 64)
    assert set(sd) == {"gate.weight"} | {f"experts.{i}.{n}.weight" for i in range(4)
                                         for n in ("gate_up_proj", "down_proj")}
    for attr in ("num_experts", "top_k", "capacity_factor", "routing_temperature", "noise_std",
                 "load_balancing_weight", "use_cuda_ops", "get_routing_stats", "reset_routing_stats"):
        assert hasattr(layer, attr)
    assert layer.get_routing_stats() == {"error": "No routing statistics available"}
    assert A.RMSNorm(8).state_dict()["weight"].shape == (8,)
    assert list(A.RotaryEmbedding(8).state_dict()) == []           # buffers are non-persistent
    assert A.MoECUDAOps.should_use_cuda(1, 1, 1, True, False) is False
    # attention sub-layer and block: the reference's parameter names; CPU tensors are refused
    cfg = LayerConfig(64, 128, 4, 2, num_heads=4, num_kv_heads=2, seq_length=32, use_moe=True)
    att = A.GroupedQueryAttention(cfg)
    assert {k: tuple(v.shape) for k, v in att.state_dict().items()} == {
        "q_proj.weight": (64, 64), "k_proj.weight": (32, 64), "v_proj.weight": (32, 64), "o_proj.weight": (64, 64)}
    with pytest.raises(A.AtsError):
        att(torch.randn(1, 4, 64).bfloat16())
    # attention dropout (model.py:831-833) is part of the kernel path: with or without it a CPU tensor is refused
    drop = A.GroupedQueryAttention(LayerConfig(64, 128, 4, 2, num_heads=4, num_kv_heads=2, seq_length=32, dropout=0.1))
    assert drop.dropout_p == pytest.approx(0.1)
    for mode in (drop.train(), drop.eval()):
        with pytest.raises(A.AtsError, match="GPU"):
            mode(torch.randn(1, 4, 64).bfloat16())
    blk = A.TransformerBlock(cfg, layer_idx=0)
    names = set(blk.state_dict())
    assert {"input_norm.weight", "post_attn_norm.weight", "self_attn.o_proj.weight", "ffn.gate.weight",
            "ffn.experts.3.down_proj.weight"} <= names
    dense = A.TransformerBlock(LayerConfig(64, 128, 1, 1, num_heads=4, num_kv_heads=2, seq_length=32), layer_idx=0)
    assert {"ffn.gate_up_proj.weight", "ffn.down_proj.weight"} <= set(dense.state_dict())
    assert A.DenseGroupedQueryAttention is A.GroupedQueryAttention


def test_workloads_are_reproducible():
    from adaptivetrainingsystem_amd import workloads as W
    a = W.make_moe_workload("c1_cpu_reference", device="cpu")
    b = W.make_moe_workload("c1_cpu_reference", device="cpu")
    assert torch.equal(a.x, b.x) and torch.equal(a.down[7], b.down[7])
    assert a.x.shape == (2, 256, 512) and a.gate_up[0].shape == (2816, 512) and a.gate.shape == (8, 512)
    c = W.make_moe_workload("c4_prefill", device="cpu", scale_tokens=16, overrides={"hidden": 64, "intermediate": 64})
    assert torch.allclose(c.logit_bias, 1.5 * torch.log(1.0 / torch.arange(1, 9).float()))
    n = W.make_norm_rope_workload(device="cpu", batch=1, seq=8)
    assert n.q.shape == (1, 16, 8, 128) and n.k.shape == (1, 4, 8, 128) and n.norm_weight.dtype == torch.float32


def test_bench_refuses_more_than_one_gpu():
    """The path runs on one GPU: asking the benchmark for more exits with a message instead of measuring."""
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    for argv, env in ((["--gpus", "2"], {}), ([], {"WORLD_SIZE": "2"})):
        r = subprocess.run([sys.executable, os.path.join(root, "bench.py"), *argv], capture_output=True, text=True,
                           env={**os.environ, **env}, timeout=300)
        assert r.returncode == 2 and "one GPU" in r.stderr and r.stdout.strip() == ""


def test_layer_is_pickled_with_the_plan_of_its_last_pass():
    """What an inference pass leaves in the layer (here on the CPU: a buffer and the offsets of its parts) goes through
    pickle; a layer pickled with the plan as a plain attribute is read as well."""
    import io
    import pickle
    from adaptivetrainingsystem_amd import ops
    from adaptivetrainingsystem_amd.layers import MoEFFNLayer
    from adaptivetrainingsystem_amd.workloads import LayerConfig
    layer = MoEFFNLayer(LayerConfig(16, 32, 4, 2, num_heads=2, num_kv_heads=1, seq_length=8))
    T, E, k, C = 5, 4, 2, 3
    layout = ops._moe_layout(T, 16, 32, E, k, C, 1, 0)[1]
    plan = torch.arange(layout[15], dtype=torch.int64).to(torch.uint8)
    layer._last_plan = ((plan, layout, T, E, k, C), torch.tensor(0.5))
    again = pickle.loads(pickle.dumps(layer))
    buf = io.BytesIO()
    torch.save(layer, buf)
    buf.seek(0)
    saved = torch.load(buf, weights_only=False)
    want = layer.last_plan
    for got in (again.last_plan, saved.last_plan):
        assert set(got) == set(want) and got["capacity"] == C
        assert all(torch.equal(got[n].view(torch.uint8), want[n].view(torch.uint8)) for n in ("weights", "row_of", "token_map"))
    state = {n: v for n, v in layer.__dict__.items() if n != "_last_plan"}
    old = MoEFFNLayer.__new__(MoEFFNLayer)
    old.__setstate__({**state, "last_plan": {"capacity": 7}})
    assert old.last_plan == {"capacity": 7} and "last_plan" not in old.__dict__


@pytest.mark.parametrize("B,Lk,D,parts", [(32, 2048, 128, 1), (33, 512, 128, 1), (33, 1024, 128, 4), (40, 2048, 128, 4),
                                          (48, 4096, 128, 1), (54, 2048, 128, 1), (64, 4096, 128, 1), (33, 4096, 64, 1)])
def test_key_ranges_of_a_decoding_step(B, Lk, D, parts):
    """32 / 8 heads, one new token: more than one range between one and one and a half workgroups per CU only."""
    from adaptivetrainingsystem_amd import _lib
    want = B * 32 * parts * (D + 4) * 4 if parts > 1 else 0
    assert _lib.load().ats_attention_fwd_workspace(B, 32, 8, 1, Lk, D) == want


@pytest.mark.parametrize("rows,M,N,slices", [(16384, 4096, 4096, 1), (16384, 2048, 4096, 2), (16384, 2048, 2048, 4),
                                             (16384, 1024, 2048, 8), (8192, 2048, 4096, 1), (4096, 2048, 4096, 1),
                                             (4096, 1024, 2048, 8), (2048, 2048, 2048, 1), (2048, 1024, 4096, 1),
                                             (1024, 512, 2048, 1), (1, 2048, 2048, 1)])
def test_slices_of_a_weight_gradient(rows, M, N, slices):
    """The choice at the measured sizes (the fastest or within 2 % of it)."""
    from adaptivetrainingsystem_amd import ops
    assert ops.wgrad_slices(M, N, rows) == slices


@pytest.mark.parametrize("E,rows,N,K,slices", [(2, 22, 1024, 16384, 16), (2, 48, 1024, 16384, 16), (4, 48, 1024, 8192, 8),
                                               (2, 64, 4096, 14336, 4), (2, 192, 4096, 14336, 8), (4, 96, 4096, 14336, 4), (8, 22, 4096, 14336, 2),
                                               (8, 96, 4096, 14336, 2), (16, 22, 2048, 8192, 2), (16, 48, 2048, 8192, 2), (16, 96, 2048, 8192, 2),
                                               (16, 48, 2048, 5632, 2), (16, 128, 2048, 5632, 2), (8, 48, 1024, 4096, 4), (8, 96, 1024, 4096, 1),
                                               (8, 96, 2048, 2048, 1), (8, 128, 2048, 2048, 4), (8, 192, 1024, 2048, 1), (64, 128, 2048, 1408, 1),
                                               (3, 32, 4096, 14336, 8), (6, 48, 4096, 14336, 4), (7, 48, 4096, 14336, 2), (10, 48, 4096, 11008, 4),
                                               (12, 56, 3072, 8192, 4), (16, 64, 768, 4096, 4), (4, 32, 1024, 8192, 8), (32, 64, 2048, 2816, 1)])
def test_slices_of_a_down_projection(E, rows, N, K, slices):
    """The choice at measured sizes: the fastest, or within 10 % of it.  (2 x 64 rows of [4096, 14336]: 53 us in four slices on the band tiles,
    58 in eight; 16 x 22 rows of [2048, 8192] 102 plain, 105 in two, with sizes that fall as rank^-1.5 124 and 101.)"""
    from adaptivetrainingsystem_amd import ops
    assert ops.down_k_splits(E, E * rows, N, K, torch.bfloat16) == slices


# a few rows against a long K: the stream of a copy's weights is the faster one; short sums, more rows and groups of them: not
@pytest.mark.parametrize("E,rows,N,K,direct", [(1, 13, 1408, 8192, False), (1, 5, 1408, 6144, False), (1, 8, 256, 8192, False), (1, 4, 2560, 8192, False),
                                               (2, 11, 1408, 8192, False), (1, 8, 2048, 2048, True), (1, 13, 1408, 256, True), (1, 512, 512, 1024, True),
                                               (8, 1024, 512, 2816, True), (8, 2000, 1408, 512, True), (1, 4096, 4096, 4096, False)])
def test_float32_data_gradient_reads_weights_as_they_lie(E, rows, N, K, direct):
    """The choice at measured sizes: the faster way."""
    from adaptivetrainingsystem_amd import ops
    assert ops.grouped_gemm_nn_f32_supported(E, rows, N, K) == direct


# bfloat16, a smaller head_dim, fewer values than keys, fewer keys than queries, heads that do not divide, 3-D, more pairs than served
@pytest.mark.parametrize("q,k,v,dtype", [((1, 4, 8, 64), (1, 2, 8, 64), (1, 2, 8, 64), torch.bfloat16), ((1, 4, 8, 64), (1, 2, 8, 32), (1, 2, 8, 32), None),
                                         ((1, 4, 8, 64), (1, 2, 8, 64), (1, 2, 7, 64), None), ((1, 4, 8, 64), (1, 2, 7, 64), (1, 2, 7, 64), None),
                                         ((1, 4, 8, 64), (1, 3, 8, 64), (1, 3, 8, 64), None), ((4, 8, 64), (4, 8, 64), (4, 8, 64), None),
                                         ((2, 4, 8, 64), (1, 2, 8, 64), (1, 2, 8, 64), None), ((1, 4097, 1, 64), (1, 4097, 1, 64), (1, 4097, 1, 64), None)])
def test_float32_attention_checks_its_operands_on_every_route(q, k, v, dtype):
    from adaptivetrainingsystem_amd import autograd, ops
    from adaptivetrainingsystem_amd._lib import AtsError
    q, k, v = (torch.zeros(s, dtype=dtype or torch.float32) for s in (q, k, v))
    out = torch.zeros(1)
    for call in (lambda: ops.attention_f32(q, k, v), lambda: ops.attention_f32_fused(q, k, v, 0.125, None),
                 lambda: autograd.AttentionF32Function.apply(q, k, v, 0.125), lambda: ops.attention_f32_fused_bwd(q, k, v, out, out, out, 0.125, None)):
        with pytest.raises(AtsError, match="attention_f32: (shapes|q, k, v must be 4-D float32)"):
            call()


def test_float32_attention_gradient_checks_what_it_is_given():
    from adaptivetrainingsystem_amd import ops
    from adaptivetrainingsystem_amd._lib import AtsError
    q, kv, out, stats = torch.zeros(1, 4, 8, 64), torch.zeros(1, 2, 8, 64), torch.zeros(1, 8, 256), torch.zeros(4, 8, 2)
    for bad in ((out[:, :7], stats, out), (out, stats[:3], out), (out, stats, out[..., :64]), (out, stats, out.bfloat16())):
        with pytest.raises(AtsError, match="as handed out"):
            ops.attention_f32_fused_bwd(q, kv, kv, *bad, 0.125, None)


def test_native_calls_let_other_threads_run():
    """With a switch interval of minutes another thread runs only where this one gives the interpreter lock up."""
    import sys
    import threading
    import time
    from adaptivetrainingsystem_amd import _lib
    native, x = _lib.native(), torch.zeros(2, 3, 4, 8)
    cache, table = torch.zeros(2, 3, 4, 8), torch.zeros(4, 8)
    calls = {"rmsnorm": (x, None, 1e-6), "rope": (x, x, table, table, 0), "rope_append": (x, x, x, table, table, cache, cache, 0, 0),
             "linear": (x, x, x, x, 8, 1), "linear_rope_append": (x, x, x, x, 2, table, table, cache, cache, 0, 1, 1),
             "attention": (x, x, x, 1.0, True), "prompt_attention": (x, table, table, 2, 1, 8, 1.0, True)}
    assert set(calls) == {n for n in dir(native) if not n.startswith("_")} - {"set_error"}
    seen, stop = [0], threading.Event()

    def other():
        while not stop.is_set():
            seen[0] += 1
            time.sleep(0)
    before, thread = sys.getswitchinterval(), threading.Thread(target=other)
    sys.setswitchinterval(300.0)
    try:
        thread.start()
        for name, args in calls.items():
            call, count = getattr(native, name), seen[0]
            for _ in range(1000000):
                assert call(*args) is None      # (not on the GPU: handed on to the general path)
                if seen[0] > count + 3:
                    break
            assert seen[0] > count + 3, name
    finally:
        stop.set()
        sys.setswitchinterval(before)
        thread.join()


def test_joined_attention_launches_check_their_shapes():
    from adaptivetrainingsystem_amd import ops
    from adaptivetrainingsystem_amd._lib import AtsError
    x, w, table, cache = torch.zeros(6, 4096), torch.zeros(512, 4096), torch.zeros(8, 64), torch.zeros(2, 2, 9, 64)
    good = {"x": x, "weight": w, "cos": table, "sin": table, "k_cache": cache, "v_cache": cache, "cache_pos": 0, "seq": 3}
    assert ops.linear_rope_append(**good) is None       # (not on the GPU)
    for bad in ({"x": torch.zeros(6, 4104)}, {"x": x[0]}, {"x": x[:5]}, {"seq": 2}, {"weight": w[:500]}, {"weight": w[:256]},
                {"weight": w[:, :4088]}, {"v_cache": cache[:, :1]}, {"k_cache": cache[0], "v_cache": cache[0]}):
        with pytest.raises(AtsError, match="linear_rope_append: x"):
            ops.linear_rope_append(**{**good, **bad})
    qkv = torch.zeros(6, 512, dtype=torch.bfloat16)
    assert ops.prompt_attention(qkv, table, table, 2, 2, 64, 0.125, True) is None
    for args in ((qkv, 4, 2, 64), (qkv, 0, 2, 64), (qkv, 2, 4, 64), (qkv, 2, 2, 96), (qkv[0], 2, 2, 64), (qkv, 2, 0, 64)):
        with pytest.raises(AtsError, match="prompt_attention: qkv"):
            ops.prompt_attention(args[0], table, table, *args[1:], 0.125, True)


def test_products_of_operands_as_they_lie_check_their_rows():
    from adaptivetrainingsystem_amd import ops
    from adaptivetrainingsystem_amd._lib import AtsError
    a, b, two = torch.zeros(64, 512), torch.zeros(64, 512), torch.zeros(2, dtype=torch.int32)
    rows = torch.zeros(64, dtype=torch.int32)
    for bad in ({"b": b[:60]}, {"b": b[:60], "k_start": two, "k_count": two}, {"b_rows": rows[:60]}, {"b_rows": rows.long()},
                {"b_rows": rows, "b_row_div": 0}):
        with pytest.raises(AtsError, match="wgrad_f32: a and b must have the same number of rows, or"):
            ops.wgrad_f32(**{"a": a, "b": b, **bad})
    with pytest.raises(AtsError, match="than K columns"):
        ops.grouped_gemm_nn_sliced(two, 512, two, two, 64, 64, 512, 1024, a.bfloat16(), 2)


def test_joined_rotation_refuses_more_threads_than_its_numbers_hold():
    """The last workgroup's thread numbers run up to 255 past the pieces."""
    from adaptivetrainingsystem_amd import _lib
    lib, p = _lib.load(), 4096
    call = lambda rows: lib.ats_rope_sum_append(p, 2, 1 << 40, p, p, p, p, p, 4, 1, rows, 1, 1, 1, 8, 8, 8, 8, 0, 1, _lib.ATS_F32, None)
    for pieces in (2 ** 31 - 2, 2 ** 31 - 252):
        rows = pieces // 3
        assert 2 ** 31 - 1 - 255 < 3 * rows < 2 ** 31 - 1
        assert call(rows) == -1, lib.ats_last_error_string()       # an argument that is not served, not a failed launch


def test_routing_statistics_are_pickled_as_a_plain_dictionary():
    import copy
    import pickle
    import adaptivetrainingsystem_amd as A
    from adaptivetrainingsystem_amd.workloads import LayerConfig
    layer = A.MoEFFNLayer(LayerConfig(32, 64, 4, 2))
    store = layer._routing_store
    counts = torch.tensor([3, 0, 1, 4, 2, 5])          # what a device would have counted: 4 experts, 2 dropped, 5 tokens
    store._counters[torch.device("cpu")] = [counts, torch.tensor([1, 0, 1, 0, 2, 1]), 0]
    assert layer._routing_stats["total_routed"] == 4 and layer._routing_stats["dropped_tokens"] == 0
    assert layer.__getstate__()["_routing_stats"] is layer._routing_stats and "_routing_store" not in layer.__getstate__()
    for twin in (copy.deepcopy(layer), pickle.loads(pickle.dumps(layer))):
        assert twin._routing_stats["expert_usage"].tolist() == [2, 0, 0, 4] and twin._routing_stats["total_routed"] == 4
        twin._routing_stats["total_routed"] = 7
        assert layer._routing_stats["total_routed"] == 4
        twin.reset_routing_stats()
        assert twin.get_routing_stats() == {"error": "No routing statistics available"}
    counts += 1
    assert layer._routing_stats["expert_usage"].tolist() == [3, 1, 1, 5] and layer._routing_stats["total_routed"] == 5
    layer.num_experts = 5                              # an expert was added
    store._counters[torch.device("cpu")] = [torch.ones(7, dtype=torch.int64), torch.zeros(7, dtype=torch.int64), 0]
    assert layer._routing_stats["expert_usage"].tolist() == [4, 2, 2, 6, 1]
    # a layer pickled when the dictionary was an attribute of its own
    state = layer.__getstate__()
    old = A.MoEFFNLayer.__new__(A.MoEFFNLayer)
    old.__setstate__({**state, "_routing_stats": {"expert_usage": torch.ones(5), "total_routed": 3, "dropped_tokens": 1}})
    assert old._routing_stats["total_routed"] == 3


def test_slices_weights_go_past_the_caches_only_where_they_are_larger():
    """8 x [1024, 2816] in four slices, 200 rows on average that fall as rank^-1.5: 31.3 us kept in the caches, 35.1 past them."""
    from adaptivetrainingsystem_amd import _lib
    route = _lib.load().ats_grouped_gemm_route
    rows256, once = 4, 5
    for E, N, K, slices, swiglu, want in ((8, 1024, 2816, 4, 0, rows256), (8, 2048, 5632, 4, 0, rows256), (8, 2816, 1024, 1, 1, once),
                                          (8, 4096, 14336, 2, 0, once), (16, 2048, 5632, 2, 0, once), (64, 1408, 2048, 1, 1, once),
                                          (8, 14336, 4096, 1, 1, once)):
        for avg in (200, 224):
            assert route(E, E * avg, N, K, slices, swiglu, _lib.ATS_F32 if slices > 1 else _lib.ATS_BF16) == want, (E, N, K, avg)
        assert route(E, E * 225, N, K, slices, swiglu, _lib.ATS_F32 if slices > 1 else _lib.ATS_BF16) == rows256


@pytest.mark.parametrize("rows,N,K,slices,route", [
    (200, 512, 512, 1, "band"), (512, 512, 512, 1, "band"), (400, 1024, 1024, 1, "band"), (300, 1000, 1536, 1, "band"), (512, 1024, 4096, 1, "band"),
    (100, 32000, 4096, 1, "band"), (200, 1536, 512, 1, "band"), (300, 12288, 4096, 1, "band"), (160, 3072, 1024, 1, "small"), (64, 2048, 2048, 1, "small"),
    (100, 1024, 1024, 1, "small"), (128, 2048, 1408, 1, "small"), (200, 1024, 1024, 1, "band"), (200, 1000, 1536, 4, None), (256, 2048, 1408, 2, None), (200, 2048, 2048, 4, None),
    (256, 2048, 2048, 4, None), (64, 6144, 4096, 4, None), (64, 4096, 4096, 8, None), (100, 4096, 14336, 8, None), (64, 3072, 2048, 1, "small")])
def test_route_of_one_weight(rows, N, K, slices, route):
    """The fastest of every route measured alone, or within 10 % of it (band tiles, slices of K, other tiles; weights from HBM)."""
    from adaptivetrainingsystem_amd import _lib, ops
    assert ops.linear_k_splits(rows, N, K, torch.bfloat16) == slices
    if route:
        assert _lib.load().ats_grouped_gemm_route(1, rows, N, K, 1, 0, _lib.ATS_BF16) == {"small": 1, "band": 2, "256": 4}[route]


@pytest.mark.parametrize("E,rows,N,K,slices,route", [(8, 32, 4096, 14336, 2, 2), (8, 48, 4096, 14336, 2, 5), (8, 72, 4096, 14336, 2, 5), (16, 64, 2048, 5632, 2, 2),
                                                     (12, 64, 2048, 5632, 4, 2), (4, 64, 4096, 14336, 2, 2), (8, 48, 2048, 5632, 2, 2)])
def test_tiles_of_a_sliced_down_projection(E, rows, N, K, slices, route):
    """Band tiles (2) or 256-row tiles (5) for the slices that the rule chooses, as measured with equal and with unequal groups."""
    from adaptivetrainingsystem_amd import _lib, ops
    assert ops.down_k_splits(E, E * rows, N, K, torch.bfloat16) == slices
    assert _lib.load().ats_grouped_gemm_route(E, E * rows, N, K, slices, 0, _lib.ATS_F32) == route
