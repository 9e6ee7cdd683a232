"""Routing and dispatch plan of a decoding step in one launch: the bits of the two launches."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,k,C", [(1, 1, 1, 1), (1, 64, 6, 1), (3, 64, 6, 3), (64, 8, 2, 20), (64, 64, 6, 9), (170, 8, 6, 64),
                                     (512, 8, 2, 160), (5, 70, 3, 5), (2, 1024, 16, 2), (33, 5, 5, 7)])
@pytest.mark.parametrize("variant,temperature", [(0, 1.0), (1, 0.7)])
def test_route_plan(gpu, T, E, k, C, variant, temperature):
    print("case route plan", T, E, k, C, variant, flush=True)
    from adaptivetrainingsystem_amd import _lib, ops
    lib = _lib.load()
    if T * k > 1024:
        pytest.skip("more than one workgroup's assignments")
    assert lib.ats_route_plan_supported(T, E, k)
    logits = (torch.randn(T, E, generator=torch.Generator().manual_seed(T + E)) * 2).to(gpu)
    route = ops.route_topk(logits, k, temperature, variant)
    plan = ops.dispatch_plan(route["indices"], E, C)
    i32 = lambda *s: torch.full(s, 77, dtype=torch.int32, device=gpu)
    f32 = lambda *s: torch.full(s, 7.0, device=gpu)
    idx, w, routed, col, aux = i32(T, k), f32(T, k), i32(E), f32(E), f32(1)
    out = {n: torch.full_like(t, 77) for n, t in plan.items()}
    ws1 = i32(2 * E)
    args = [logits.data_ptr(), T, E, k, temperature, variant, idx.data_ptr(), w.data_ptr(), routed.data_ptr(), col.data_ptr(),
            aux.data_ptr(), 0.01, ws1.data_ptr(), 8 * E, C] + \
        [out[n].data_ptr() for n in ("slot", "token_map", "hist", "kept", "offsets", "row_src", "row_of", "status")] + \
        [torch.cuda.current_stream().cuda_stream]
    assert lib.ats_route_plan(*args) == 0, lib.ats_last_error_string()
    for a, b in ((idx, route["indices"]), (w, route["weights"]), (routed, route["hist"]), (col, route["prob_colsum"]),
                 (aux, route["aux"])):
        assert torch.equal(a, b)
    for n in plan:
        assert torch.equal(out[n], plan[n]), n
    args[13] = 8 * E - 1
    assert lib.ats_route_plan(*args) != 0


def test_route_plan_sizes(gpu):
    from adaptivetrainingsystem_amd import _lib
    lib = _lib.load()
    assert not lib.ats_route_plan_supported(0, 8, 2) and not lib.ats_route_plan_supported(4, 8, 9)
    assert not lib.ats_route_plan_supported(513, 8, 2) and not lib.ats_route_plan_supported(65, 64, 1)
