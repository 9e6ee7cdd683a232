// Address and row tables of grouped products, several per launch.
//
// The grouped kernels read their groups' base addresses and row ranges from device memory.  All of these tables are
// affine in an index that follows from the group number (the group itself, the key/value matrix of a query head, the
// slot of a head in a reduction buffer, an int32 read on the device), so one launch of one small workgroup per table
// writes every table that a step needs.  Bound: the launch itself (about 5 us on the timeline of a stream).  Built from
// torch expressions, each table was two or three launches and as many host calls of 4-6 us: a float32 transformer block
// made 107 of its 250 launches for them.
#include <string.h>

#include "ats_common.hpp"

namespace ats {

constexpr int kMaxTables = 20;
struct TableArgs {
    ats_table t[kMaxTables];
    int Hq, Hkv, BHkv;
};

__global__ __launch_bounds__(64) void fill_tables_kernel(TableArgs a) {
    const ats_table t = a.t[blockIdx.x];
    for (int i = threadIdx.x; i < t.n; i += 64) {
        int64_t x = 0;
        switch (t.kind) {
            case ATS_TABLE_INDEX: x = i; break;
            case ATS_TABLE_KV_OF_HEAD: x = (i / a.Hq) * a.Hkv + (i % a.Hq) / (a.Hq / a.Hkv); break;
            case ATS_TABLE_SLOT_OF_HEAD:
                x = (i % a.Hq % (a.Hq / a.Hkv)) * a.BHkv + (i / a.Hq) * a.Hkv + (i % a.Hq) / (a.Hq / a.Hkv);
                break;
            case ATS_TABLE_HEAD_OF_SLOT: {
                const int kv = i % a.BHkv;
                x = (kv / a.Hkv) * a.Hq + (kv % a.Hkv) * (a.Hq / a.Hkv) + i / a.BHkv;
                break;
            }
            case ATS_TABLE_FROM_ARRAY: x = t.index[i]; break;
            default: break;      // ATS_TABLE_CONSTANT
        }
        const int64_t v = t.base + x * t.stride;
        if (t.wide) static_cast<int64_t*>(t.out)[i] = v;
        else static_cast<int32_t*>(t.out)[i] = (int32_t)v;
    }
}

// Small host arrays (a list of tensor addresses and sizes) as launch arguments: a copy from pageable memory waits until
// the queue has drained, which left the GPU idle between the backward of the loss and the gradient norm.
constexpr int kUploadBytes = 3584;           // of the 4 KiB that the arguments of a launch can have
struct UploadArgs {
    uint64_t w[kUploadBytes / 8];
};
__global__ __launch_bounds__(64) void upload_kernel(UploadArgs a, uint64_t* __restrict__ dst, int words) {
    for (int i = threadIdx.x; i < words; i += 64) dst[i] = a.w[i];
}

// Several matrices of one width below each other, and the address of the result where a grouped product reads it.  Bound by the
// bytes: a workgroup moves 16 KB at a time, four 16-byte loads per lane in flight, with ordinary stores (the product behind it
// reads them).  Projections of hidden 4096, 32 + 16 heads (50 MB): 18.5 us against 39.5 for torch's concatenation and 4.7 for the
// launch that wrote the address.
constexpr int kMaxStack = 8;
struct StackArgs {
    const uint4* src[kMaxStack];
    int64_t first[kMaxStack], n[kMaxStack];      // 16-byte units
};
__global__ __launch_bounds__(256) void stack_rows_kernel(StackArgs a, uint4* __restrict__ out, int64_t* __restrict__ address) {
    const uint4* __restrict__ const src = a.src[blockIdx.y];
    uint4* const dst = out + a.first[blockIdx.y];
    const int64_t n = a.n[blockIdx.y];
    if (address && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *address = (int64_t)reinterpret_cast<uintptr_t>(out);
    for (int64_t i = (int64_t)blockIdx.x * 1024 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 1024) {
        uint4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = src[min(i + 256 * u, n - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i + 256 * u < n) dst[i + 256 * u] = v[u];
    }
}

}  // namespace ats

extern "C" int ats_stack_rows(const void* const* src, const int64_t* bytes, int n, void* out, int64_t* address, ats_stream_t stream) {
    using namespace ats;
    const char* name = "ats_stack_rows";
    ATS_REQUIRE(src && bytes && n >= 1 && n <= kMaxStack && out && aligned16(out), ATS_ERR_INVALID_ARG,
                "%s: %d matrices (at most %d), null or misaligned pointer", name, n, kMaxStack);
    StackArgs a{};
    int64_t first = 0, most = 0;
    for (int i = 0; i < n; ++i) {
        ATS_REQUIRE(src[i] && aligned16(src[i]) && bytes[i] > 0 && bytes[i] % 16 == 0, ATS_ERR_INVALID_ARG,
                    "%s: matrix %d of %lld bytes (16-byte aligned, a multiple of 16)", name, i, (long long)bytes[i]);
        a.src[i] = static_cast<const uint4*>(src[i]);
        a.first[i] = first;
        a.n[i] = bytes[i] / 16;
        first += a.n[i];
        most = a.n[i] > most ? a.n[i] : most;
    }
    int64_t blocks = (most + 1023) / 1024;
    if (blocks > 2048) blocks = 2048;
    hipLaunchKernelGGL(stack_rows_kernel, dim3((unsigned)blocks, (unsigned)n), dim3(256), 0, as_stream(stream), a,
                       static_cast<uint4*>(out), address);
    ATS_CHECK_LAUNCH(name);
    return ATS_OK;
}

extern "C" int ats_upload_max_bytes(void) { return ats::kUploadBytes; }

extern "C" int ats_upload(void* dst, const void* src, int bytes, ats_stream_t stream) {
    using namespace ats;
    ATS_REQUIRE(bytes >= 0 && bytes <= kUploadBytes && bytes % 8 == 0, ATS_ERR_INVALID_ARG,
                "ats_upload: %d bytes (a multiple of 8, at most %d)", bytes, kUploadBytes);
    if (bytes == 0) return ATS_OK;
    ATS_REQUIRE(dst && src && (reinterpret_cast<uintptr_t>(dst) & 7u) == 0, ATS_ERR_INVALID_ARG,
                "ats_upload: null pointer or unaligned destination");
    UploadArgs a;
    memcpy(a.w, src, (size_t)bytes);
    memset(reinterpret_cast<char*>(a.w) + bytes, 0, sizeof(a.w) - (size_t)bytes);
    hipLaunchKernelGGL(upload_kernel, dim3(1), dim3(64), 0, as_stream(stream), a, static_cast<uint64_t*>(dst), bytes / 8);
    ATS_CHECK_LAUNCH("ats_upload");
    return ATS_OK;
}

extern "C" int ats_fill_tables(const ats_table* tables, int n_tables, int batch, int q_heads, int kv_heads,
                               ats_stream_t stream) {
    using namespace ats;
    ATS_REQUIRE(tables && n_tables >= 0 && n_tables <= kMaxTables, ATS_ERR_INVALID_ARG, "ats_fill_tables: %d tables (at most %d)",
                n_tables, kMaxTables);
    if (n_tables == 0) return ATS_OK;
    TableArgs a{};
    for (int i = 0; i < n_tables; ++i) {
        const ats_table& t = tables[i];
        const bool heads = t.kind == ATS_TABLE_KV_OF_HEAD || t.kind == ATS_TABLE_SLOT_OF_HEAD || t.kind == ATS_TABLE_HEAD_OF_SLOT;
        ATS_REQUIRE(t.out && t.n >= 0 && t.kind >= ATS_TABLE_INDEX && t.kind <= ATS_TABLE_CONSTANT, ATS_ERR_INVALID_ARG,
                    "ats_fill_tables: table %d: n=%d kind=%d or null output", i, t.n, t.kind);
        ATS_REQUIRE(t.kind != ATS_TABLE_FROM_ARRAY || t.index, ATS_ERR_INVALID_ARG, "ats_fill_tables: table %d has no index array", i);
        ATS_REQUIRE(!heads || (batch > 0 && kv_heads > 0 && q_heads > 0 && q_heads % kv_heads == 0 && t.n <= (int64_t)batch * q_heads),
                    ATS_ERR_INVALID_ARG, "ats_fill_tables: table %d: %d entries of %d x %d heads (%d key/value heads)", i, t.n, batch,
                    q_heads, kv_heads);
        a.t[i] = t;
    }
    a.Hq = q_heads > 0 ? q_heads : 1;
    a.Hkv = kv_heads > 0 ? kv_heads : 1;
    a.BHkv = batch > 0 ? batch * a.Hkv : 1;
    hipLaunchKernelGGL(fill_tables_kernel, dim3((unsigned)n_tables), dim3(64), 0, as_stream(stream), a);
    ATS_CHECK_LAUNCH("ats_fill_tables");
    return ATS_OK;
}
