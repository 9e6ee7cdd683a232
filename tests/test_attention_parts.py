"""The query tiles that a workgroup of the causal attention kernels takes (csrc/attention_parts.hpp): every tile once, on the host,
and results that do not depend on how a launch is cut."""
import ctypes
import os
import random
import subprocess
import time

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "attention_parts.hpp"
extern "C" int parts(int n, long heads, int cus, int two, int per_tile, int off, unsigned* tiles) {
    const ats::AttnParts p = ats::attn_parts(n, heads, cus, two, [&](int t) { return (t + 1) * per_tile + off; });
    for (int i = 0; i < p.count; ++i) tiles[i] = p.tiles[i];
    return p.count;
}
"""


def _host_rule(tmp_path):
    src, lib = tmp_path / "parts.cpp", tmp_path / "parts.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I" + os.path.join(ROOT, "adaptivetrainingsystem_amd", "csrc"),
                    str(src), "-o", str(lib)], check=True)
    return ctypes.CDLL(str(lib)).parts


def test_long_tiles_are_dealt_in_bounded_time(tmp_path):
    """2081 new positions, 32 heads, up to a million cached keys: each room by itself took 0.19 ms at 34 000 keys and 6 ms at a million."""
    f = _host_rule(tmp_path)
    tiles = (ctypes.c_uint * 16)()
    for heads, cached in ((4, 34000), (4, 1000000), (16, 1000000), (128, 1000000)):
        times = []
        for _ in range(5):
            t0 = time.perf_counter()
            f(17, ctypes.c_long(heads), 32, 1, 2, cached // 64, tiles)
            times.append(time.perf_counter() - t0)
        assert min(times) < 1e-4, (heads, cached, min(times))


def _least_room(w, parts, rooms):
    for room in rooms:
        left, used = [room] * parts, set()
        for t in reversed(range(len(w))):
            p = next((p for p in range(parts) if left[p] >= w[t]), None)
            if p is None:
                break
            left[p] -= w[t]
            used.add(p)
        else:
            return room, len(used)
    return None


def test_the_least_estimate_of_all_rooms_is_taken(tmp_path):
    """Against trying every room of every number of parts (tile starts count 6 key tiles; 5 quarters a pair of parts on a unit)."""
    f = _host_rule(tmp_path)
    tiles = (ctypes.c_uint * 16)()
    rng = random.Random(4)
    for case in range(60):
        n, heads, cus, two = rng.randint(2, 20), rng.randint(1, 120), rng.choice((32, 256)), rng.randint(0, 1)
        per, off = rng.choice((1, 2, 4, 9)), rng.choice((0, 0, 7, 200))
        w = [(t + 1) * per + off + 6 for t in range(n)]

        def cost(parts, most):
            cu = -(-heads * parts // cus)
            return most * (5 * (cu // 2) + 4 * (cu % 2) if two else 4 * cu)

        pairs = [w[p] + w[n - 1 - p] for p in range(n // 2)] + ([w[n // 2]] if n % 2 else [])
        least, best = cost((n + 1) // 2, max(pairs)) * 19 // 20, 0
        for parts in range(min(n, 16), 0, -1):
            lo = max(w[-1], -(-sum(w) // parts))
            found = _least_room(w, parts, range(lo, (least - 1) // cost(parts, 1) + 1))
            if found and found[1] == parts:
                least, best = cost(parts, found[0]), parts
        assert f(n, ctypes.c_long(heads), cus, two, per, off, tiles) == best, (n, heads, cus, two, per, off)


def test_every_tile_belongs_to_one_part(tmp_path):
    f = _host_rule(tmp_path)
    f.argtypes = [ctypes.c_int, ctypes.c_long, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.POINTER(ctypes.c_uint)]
    seen = set()
    for n in list(range(1, 34)) + [64]:
        for heads in (1, 4, 12, 16, 20, 32, 33, 96, 256, 100000):
            for cus, two, per_tile, off in ((32, 1, 2, 0), (256, 1, 2, 0), (32, 0, 4, 0), (256, 1, 2, 40), (32, 1, 0, 3)):
                tiles = (ctypes.c_uint * 16)()
                count = f(n, heads, cus, two, per_tile, off, tiles)
                seen.add(count)
                assert 0 <= count <= min(n, 16) and (count == 0 or 2 <= n <= 32)
                if count:
                    assert all(tiles[i] for i in range(count))
                    assert sum(bin(tiles[i]).count("1") for i in range(count)) == n
                    assert sum(tiles[i] for i in range(count)) == (1 << n) - 1
    assert {0, 1, 2, 3, 5} <= seen


def test_scratch_of_the_backward_is_bounded():
    from adaptivetrainingsystem_amd import _lib
    f = _lib.load().ats_attention_bwd_workspace
    for B, Hq, Hkv in ((1, 32, 8), (4, 32, 8), (1, 8, 8), (1, 128, 1), (3, 16, 4), (8, 32, 32)):
        for D in (64, 128):
            for L in (1, 300, 1777, 4100, 6144, 12000, 50000, 84340, 100000, 1000000):
                for Lk in (L, L + 5000):
                    size = f(B, Hq, Hkv, L, Lk, D)
                    assert size <= 512 * 10 ** 6 and size % (2 * B * Hkv * Lk * D * 4) == 0, (B, Hq, Hkv, L, Lk, D, size)
    # 8, 3 and 4 ranges of one, three and four sequences' queries, as before
    assert [f(B, 32, 8, L, L, 128) // (2 * B * 8 * L * 128 * 4) for B, L in ((1, 1777), (3, 1777), (8, 2048), (1, 12000))] == [8, 3, 0, 4]


@pytest.mark.gpu
def test_without_memory_for_the_scratch(gpu, monkeypatch):
    from adaptivetrainingsystem_amd import ops
    q, k, v, do = (torch.randn(*s, device=gpu).bfloat16() for s in ((1, 4, 300, 64), (1, 2, 300, 64), (1, 2, 300, 64), (1, 300, 256)))
    out, lse = ops.causal_attention(q, k, v, return_lse=True)
    want = ops.causal_attention_bwd(q, k, v, out, lse, do)
    empty = torch.empty

    def full(*shape, dtype=None, **more):
        if dtype == torch.uint8:
            raise torch.OutOfMemoryError("no room")
        return empty(*shape, dtype=dtype, **more)

    monkeypatch.setattr(torch, "empty", full)
    got = ops.causal_attention_bwd(q, k, v, out, lse, do)
    monkeypatch.undo()
    assert torch.equal(got[0], want[0])
    # the same float32 sums in another order, then one rounding to bfloat16 (8 bits: neighbours lie up to 2^-7 of their value apart)
    for a, b in zip(got[1:], want[1:]):
        assert ((a.float() - b.float()).abs() <= 2 ** -7 * b.float().abs() + 1e-5 * b.float().abs().max()).all()


# keys of a tile whose queries are cut into ranges, some of them empty (the last tile sees 2 queries, 1 of 4 heads' steps each)
@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hkv,L,Lk,D", [(1, 4, 1, 130, 130, 128), (1, 8, 1, 33, 33, 64), (1, 4, 4, 1500, 1500, 64), (1, 8, 2, 700, 900, 64), (2, 32, 2, 2, 300, 128)])
@pytest.mark.parametrize("dropout", [0.0, 0.2])
def test_ranges_of_queries_add_up(gpu, B, Hq, Hkv, L, Lk, D, dropout):
    from adaptivetrainingsystem_amd import _lib, ops
    print("case", B, Hq, Hkv, L, Lk, D, dropout, flush=True)
    lib = _lib.load()
    g = torch.Generator(device=gpu).manual_seed(5)
    q, k, v, do = (torch.randn(*s, generator=g, device=gpu).bfloat16()
                   for s in ((B, Hq, L, D), (B, Hkv, Lk, D), (B, Hkv, Lk, D), (B, L, Hq * D)))
    out, lse = ops.causal_attention(q, k, v, return_lse=True, dropout_p=dropout, dropout_seed=3)
    assert lib.ats_attention_bwd_workspace(B, Hq, Hkv, L, Lk, D) > 0
    dq, dk, dv = ops.causal_attention_bwd(q, k, v, out, lse, do, dropout_p=dropout, dropout_seed=3)
    q1, k1, v1, delta = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v), torch.empty_like(lse)
    assert lib.ats_attention_bwd_out(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), do.data_ptr(), lse.data_ptr(),
                                     delta.data_ptr(), None, None, 0, 0, dropout, 3, q1.data_ptr(), k1.data_ptr(), v1.data_ptr(), B, Hq,
                                     Hkv, L, Lk, D, D ** -0.5, torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(dq, q1)
    # the same float32 sums in another order, then one rounding to bfloat16 (8 bits: neighbours lie up to 2^-7 of their value apart)
    for a, b in ((dk, k1), (dv, v1)):
        assert ((a.float() - b.float()).abs() <= 2 ** -7 * b.float().abs() + 1e-5 * b.float().abs().max()).all()


# tiles of 128 rows in 2, 3, 5, 7, 14 and 32 (33: pairs again), of 256 rows in 17; cached keys; packed heads of a short chunk
@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hkv,L,Lk,D", [(5, 32, 8, 225, 225, 128), (5, 32, 8, 372, 372, 64), (3, 12, 4, 640, 640, 128),
                                             (3, 32, 8, 897, 1100, 128), (3, 32, 8, 1777, 1777, 128), (1, 8, 8, 4090, 4090, 64),
                                             (1, 8, 2, 4200, 4200, 64), (7, 16, 8, 100, 900, 128)])
def test_results_do_not_depend_on_the_parts(gpu, B, Hq, Hkv, L, Lk, D):
    from adaptivetrainingsystem_amd import ops
    print("case", B, Hq, Hkv, L, Lk, D, flush=True)
    g = torch.Generator(device=gpu).manual_seed(11)
    q, k, v, do = (torch.randn(*s, generator=g, device=gpu).bfloat16()
                   for s in ((B, Hq, L, D), (B, Hkv, Lk, D), (B, Hkv, Lk, D), (B, L, Hq * D)))
    out, lse = ops.causal_attention(q, k, v, return_lse=True)
    dq, dk, dv = ops.causal_attention_bwd(q, k, v, out, lse, do)
    # one sequence by itself, with one kv head's queries, is cut otherwise: the same rows, the same bits
    rep = Hq // Hkv
    for b, h in {(0, 0), (B - 1, Hkv - 1)}:
        hq = slice(h * rep, (h + 1) * rep)
        q1, k1, v1 = q[b:b + 1, hq].contiguous(), k[b:b + 1, h:h + 1].contiguous(), v[b:b + 1, h:h + 1].contiguous()
        o1, l1 = ops.causal_attention(q1, k1, v1, return_lse=True)
        cols = slice(h * rep * D, (h + 1) * rep * D)
        if L * rep >= 128 * rep:     # (fewer rows against many keys: ranges of keys, whose sums have another order)
            assert torch.equal(o1[0], out[b, :, cols]) and torch.equal(l1[0], lse[b, hq])
        d1 = ops.causal_attention_bwd(q1, k1, v1, out[b:b + 1, :, cols].contiguous(), lse[b:b + 1, hq].contiguous(), do[b:b + 1, :, cols].contiguous())
        assert torch.equal(d1[0][0], dq[b, hq])
        # against float32 of the same values (bfloat16 bar of the attention tests: 2e-2 of the largest value, gradients 3e-2)
        s = torch.einsum("hld,kd->hlk", q1[0].float(), k1[0, 0].float()) * D ** -0.5
        s = s.masked_fill(torch.ones(L, Lk, dtype=torch.bool, device=gpu).triu(Lk - L + 1), float("-inf"))
        p = s.softmax(-1)
        ref = torch.matmul(p, v1[0, 0].float())
        got = out[b, :, cols].view(L, rep, D).transpose(0, 1).float()
        assert (got - ref).abs().max() <= 2e-2 * ref.abs().max()
        do1 = do[b, :, cols].view(L, rep, D).transpose(0, 1).float()
        dp = torch.matmul(do1, v1[0, 0].float().t())
        ds = p * (dp - (do1 * ref).sum(-1, keepdim=True)) * D ** -0.5
        for have, want in ((dq[b, hq].float(), torch.matmul(ds, k1[0, 0].float())),
                           (dk[b, h].float(), torch.matmul(ds.transpose(1, 2), q1[0].float()).sum(0)),
                           (dv[b, h].float(), torch.matmul(p.transpose(1, 2), do1).sum(0))):
            assert (have - want).abs().max() <= 3e-2 * want.abs().max()
