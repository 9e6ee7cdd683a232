// The inference pass of the MoE layer as one call: the launches of its stages, issued from native code.
//
// At decode sizes the layer is six short launches, and issuing them one by one from Python (a wrapper, an allocation or
// two and a foreign call each, about 20 us a stage) took longer than the kernels run: 64 experts, 3 tokens: 120-150 us of
// host work around 85 us of kernels.  The stages and their results are those of the separate entry points.
#include "ats_common.hpp"

namespace ats {
namespace {

constexpr int64_t kAlign = 256;
int64_t padded(int64_t bytes) { return (bytes + kAlign - 1) / kAlign * kAlign; }

}  // namespace
}  // namespace ats

extern "C" int ats_moe_forward_layout(int64_t T, int H, int I, int E, int k, int C, int k_splits, int dtype,
                                      int64_t* layout) {
    using namespace ats;
    ATS_REQUIRE(layout && T > 0 && H > 0 && I > 0 && E > 0 && k > 0 && C > 0 && k_splits >= 1, ATS_ERR_INVALID_ARG,
                "ats_moe_forward_layout: T=%lld H=%d I=%d E=%d k=%d C=%d k_splits=%d", (long long)T, H, I, E, k, C, k_splits);
    ATS_REQUIRE(dtype == ATS_F32 || dtype == ATS_BF16, ATS_ERR_UNSUPPORTED, "ats_moe_forward_layout: dtype tag %d", dtype);
    const int64_t n = T * k, cap = (int64_t)E * C, rows = n < cap ? n : cap;
    int64_t plan_ws = (int64_t)ats_dispatch_plan_workspace(T, k, E);
    if (plan_ws < 4 * E) plan_ws = 4 * E;
    const int64_t bytes[ATS_MOE_LAYOUT_PLAN_BYTES] = {
        4 * T * E, 4 * n, 4 * n, 4 * E, 4 * E, 4 * n, 4 * cap, 4 * E, 4 * E, 4 * (E + 1), 4 * rows, 4 * n, 4,
        (int64_t)ats_route_topk_workspace(T, E), plan_ws};
    int64_t at = 0;
    for (int i = 0; i < ATS_MOE_LAYOUT_PLAN_BYTES; ++i) {
        layout[i] = at;
        at += padded(bytes[i] > 0 ? bytes[i] : 1);
    }
    layout[ATS_MOE_LAYOUT_PLAN_BYTES] = at;
    const int64_t es = dtype == ATS_F32 ? 4 : 2;
    layout[ATS_MOE_LAYOUT_Y] = padded(rows * I * es);
    layout[ATS_MOE_LAYOUT_SCRATCH_BYTES] = layout[ATS_MOE_LAYOUT_Y] + padded(rows * H * (k_splits > 1 ? 4 * k_splits : es));
    return ATS_OK;
}

extern "C" int ats_moe_forward(const void* x, const void* gate, const float* gate_bias, const void* const* w_gu,
                               const void* const* w_d, void* out, const int32_t* out_rows, float* aux, void* plan,
                               void* scratch, const int64_t* layout, int64_t T, int H, int I, int E, int k, int C,
                               int k_splits, float temperature, int variant, float load_balancing_weight, int dtype,
                               ats_stream_t stream) {
    using namespace ats;
    ATS_REQUIRE(x && gate && w_gu && w_d && out && aux && plan && scratch && layout, ATS_ERR_INVALID_ARG,
                "ats_moe_forward: null pointer");
    ATS_REQUIRE(T > 0 && E > 0 && k > 0 && C > 0 && k_splits >= 1, ATS_ERR_INVALID_ARG,
                "ats_moe_forward: T=%lld E=%d k=%d C=%d k_splits=%d", (long long)T, E, k, C, k_splits);
    ATS_REQUIRE(!(out_rows && k_splits > 1), ATS_ERR_UNSUPPORTED,
                "ats_moe_forward: adding onto rows of a target needs an unsliced down projection");
    const int64_t n = T * k, cap = (int64_t)E * C, rows = n < cap ? n : cap;
    char* const base = static_cast<char*>(plan);
    auto at = [&](int field) { return static_cast<void*>(base + layout[field]); };
    auto i32 = [&](int field) { return static_cast<int32_t*>(at(field)); };
    float* const logits = static_cast<float*>(at(ATS_MOE_LAYOUT_LOGITS));
    float* const w = static_cast<float*>(at(ATS_MOE_LAYOUT_WEIGHTS));
    const size_t route_ws = (size_t)(layout[ATS_MOE_LAYOUT_PLAN_WS] - layout[ATS_MOE_LAYOUT_ROUTE_WS]);
    const size_t plan_ws = (size_t)(layout[ATS_MOE_LAYOUT_PLAN_BYTES] - layout[ATS_MOE_LAYOUT_PLAN_WS]);
    void* const h = scratch;
    void* const y = static_cast<char*>(scratch) + layout[ATS_MOE_LAYOUT_Y];

    int rc = ats_router_logits(x, gate, gate_bias, logits, T, H, E, dtype, stream);
    if (rc != ATS_OK) return rc;
    if (ats_route_plan_supported(T, E, k)) {
        rc = ats_route_plan(logits, T, E, k, temperature, variant, i32(ATS_MOE_LAYOUT_INDICES), w, i32(ATS_MOE_LAYOUT_ROUTED),
                            static_cast<float*>(at(ATS_MOE_LAYOUT_PROB_COLSUM)), aux, load_balancing_weight,
                            at(ATS_MOE_LAYOUT_ROUTE_WS), route_ws, C, i32(ATS_MOE_LAYOUT_SLOT), i32(ATS_MOE_LAYOUT_TOKEN_MAP),
                            i32(ATS_MOE_LAYOUT_HIST), i32(ATS_MOE_LAYOUT_KEPT), i32(ATS_MOE_LAYOUT_OFFSETS),
                            i32(ATS_MOE_LAYOUT_ROW_SRC), i32(ATS_MOE_LAYOUT_ROW_OF), i32(ATS_MOE_LAYOUT_STATUS), stream);
        if (rc != ATS_OK) return rc;
    } else {
        rc = ats_route_topk(logits, T, E, k, temperature, variant, i32(ATS_MOE_LAYOUT_INDICES), w, i32(ATS_MOE_LAYOUT_ROUTED),
                            static_cast<float*>(at(ATS_MOE_LAYOUT_PROB_COLSUM)), aux, load_balancing_weight,
                            at(ATS_MOE_LAYOUT_ROUTE_WS), route_ws, stream);
        if (rc != ATS_OK) return rc;
        rc = ats_dispatch_plan(i32(ATS_MOE_LAYOUT_INDICES), ATS_IDX_I32, T, k, E, C, i32(ATS_MOE_LAYOUT_SLOT),
                               i32(ATS_MOE_LAYOUT_TOKEN_MAP), i32(ATS_MOE_LAYOUT_HIST), i32(ATS_MOE_LAYOUT_KEPT),
                               i32(ATS_MOE_LAYOUT_OFFSETS), i32(ATS_MOE_LAYOUT_ROW_SRC), i32(ATS_MOE_LAYOUT_ROW_OF),
                               i32(ATS_MOE_LAYOUT_STATUS), at(ATS_MOE_LAYOUT_PLAN_WS), plan_ws, stream);
        if (rc != ATS_OK) return rc;
    }
    const int32_t* const offsets = i32(ATS_MOE_LAYOUT_OFFSETS);
    const int32_t* const kept = i32(ATS_MOE_LAYOUT_KEPT);
    rc = ats_grouped_gateup_swiglu(x, T, i32(ATS_MOE_LAYOUT_ROW_SRC), k, w_gu, h, offsets, kept, E, rows, H, I, dtype, stream);
    if (rc != ATS_OK) return rc;
    if (k_splits > 1) {
        rc = ats_grouped_down_splitk(h, w_d, static_cast<float*>(y), offsets, kept, E, rows, rows, H, I, k_splits, dtype, stream);
        if (rc != ATS_OK) return rc;
        return ats_combine_partials(static_cast<float*>(y), k_splits, rows * H, i32(ATS_MOE_LAYOUT_ROW_OF), w, nullptr, out, T,
                                    k, H, dtype, stream);
    }
    rc = ats_grouped_down(h, w_d, y, offsets, kept, E, rows, H, I, dtype, dtype, stream);
    if (rc != ATS_OK) return rc;
    if (out_rows)
        return ats_combine_scatter_add(y, i32(ATS_MOE_LAYOUT_ROW_OF), w, out_rows, out, T, k, H, dtype, dtype, stream);
    return ats_combine(y, i32(ATS_MOE_LAYOUT_ROW_OF), w, nullptr, out, T, k, H, dtype, dtype, stream);
}
