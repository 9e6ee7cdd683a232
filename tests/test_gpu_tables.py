"""ats_fill_tables: every kind of table against the expressions they stand for."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv", [(1, 1, 1), (2, 4, 2), (3, 32, 8), (5, 70, 10)])
def test_fill_tables(gpu, B, Hq, Hkv):
    from adaptivetrainingsystem_amd import ops
    E, rep = B * Hq, Hq // Hkv
    e = torch.arange(E)
    kv = (e // Hq) * Hkv + (e % Hq) // rep
    slot = (e % Hq % rep) * (B * Hkv) + kv
    order = torch.empty(E, dtype=torch.int64)
    order[slot] = e
    index = torch.randint(0, 1 << 20, (E,), dtype=torch.int32)
    base, step = 1 << 40, 3 << 33
    got = ops.fill_tables(gpu, [(ops.TABLE_INDEX, E, base, step, True), (ops.TABLE_KV_OF_HEAD, E, base, step, True),
                                (ops.TABLE_SLOT_OF_HEAD, E, base, step, True), (ops.TABLE_HEAD_OF_SLOT, E, base, step, True),
                                (ops.TABLE_FROM_ARRAY, E, base, 2, True, index.to(gpu)), (ops.TABLE_INDEX, B * Hkv, 7, 5, True),
                                (ops.TABLE_INDEX, E, 0, 64, False), (ops.TABLE_CONSTANT, E, 9, 0, False)], (B, Hq, Hkv))
    want = [base + v * step for v in (e, kv, slot, order)] + [base + 2 * index.long(), 7 + 5 * torch.arange(B * Hkv),
                                                              (64 * e).int(), torch.full((E,), 9, dtype=torch.int32)]
    for g, w in zip(got, want):
        assert g.dtype == w.dtype and torch.equal(g.cpu(), w)


def test_fill_tables_refuses(gpu):
    from adaptivetrainingsystem_amd import _lib, ops
    with pytest.raises(_lib.AtsError):
        ops.fill_tables(gpu, [(ops.TABLE_KV_OF_HEAD, 5, 0, 1, True)], (1, 4, 2))       # more entries than heads
    with pytest.raises(_lib.AtsError):
        ops.fill_tables(gpu, [(ops.TABLE_KV_OF_HEAD, 4, 0, 1, True)], (1, 4, 3))
    with pytest.raises(_lib.AtsError):
        ops.fill_tables(gpu, [(9, 4, 0, 1, True)])
    assert _lib.load().ats_fill_tables((_lib.Table * 21)(), 21, 0, 0, 0, None) != 0
    assert ctypes.sizeof(_lib.Table) == 48
