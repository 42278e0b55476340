"""The shape of a prefill launch, on the host: every piece of a unit has a slot of
its own within the workspace, and the merge asks the workgroups that have them."""
import ctypes as C
import random

import pytest

from kvmem_amd import _lib as L

lib = L.load()
lib.kvm_fa_prefill_slot.restype = lib.kvm_fa_prefill_slots.restype = C.c_uint32


def prefill_shape(k_type, head_dim, n_head_kv, n_cells, n_tokens, n_head, n_cu):
    """(source, rows of a unit, row tiles, segments, units, workgroups, slots) of a launch."""
    out = (C.c_uint32 * 7)()
    assert lib.kvm_fa_prefill_shape(k_type, head_dim, n_head_kv, n_cells, n_tokens, n_head, n_cu, out) == 0
    return list(out)


def _pieces(U, P):
    """(workgroup, unit, whole) of every piece: workgroup p has [p U, (p + 1) U) of U P, unit u [u P, (u + 1) P)."""
    for p in range(P):
        for u in range(p * U // P, ((p + 1) * U - 1) // P + 1):
            yield p, u, p * U <= u * P and (u + 1) * P <= (p + 1) * U


def _check(U, P, n_seg):
    slots = lib.kvm_fa_prefill_slots(U, P, n_seg)
    of, has = {}, {}
    for p, u, whole in _pieces(U, P):
        if whole and n_seg == 1:
            continue
        s = lib.kvm_fa_prefill_slot(U, P, n_seg, p, u)
        assert s < slots and s not in of, (U, P, n_seg, p, u, of.get(s))
        of[s] = (p, u)
        has.setdefault(u, []).append(p)
    for u, ps in has.items():
        assert ps == list(range(u * P // U, ((u + 1) * P - 1) // U + 1)), (U, P, u)


@pytest.mark.parametrize("n_seg", [1, 2, 3])
def test_pieces_have_slots_of_their_own(n_seg):
    rng = random.Random(n_seg)
    for U in [1, 2, 3, 7, 64, 255, 256, 257, 304, 400, 511, 512, 513, 768, 1000] + [rng.randint(1, 3000) for _ in range(30)]:
        for P in {256, U, 2 * U, 3 * U + 1, max(1, U // 3), rng.randint(1, 700)}:
            if U % n_seg == 0:
                _check(U, P, n_seg)


@pytest.mark.parametrize("n_cells,H,G,D,T", [(525312, 4, 6, 256, 2100), (525312, 8, 4, 128, 1160), (1048640, 4, 6, 256, 2048)])
def test_segmented_windows_with_more_units_than_workgroups(n_cells, H, G, D, T):
    src, rows, n_row_tiles, n_seg, U, P, slots = prefill_shape(L.T_Q8_0, D, H, n_cells, T, H * G, 256)
    assert n_seg > 1 and U > P and U % P and U == n_row_tiles * H * n_seg
    assert slots == lib.kvm_fa_prefill_slots(U, P, n_seg)
    _check(U, P, n_seg)


@pytest.mark.parametrize("n_cells,T,want", [(2048, 1500, 376), (4096, 1500, 376), (8192, 1500, 256), (2048, 2048, 256)])
def test_units_that_outnumber_the_cus(n_cells, T, want):
    """Whole units over few tiles (376 of 256 rows), equal shares over many and where
    the units fill every round (512)."""
    _, _, _, _, U, P, slots = prefill_shape(L.T_F16, 128, 8, n_cells, T, 64, 256)
    assert P == want and U == (376 if T == 1500 else 512)
    assert slots == (512 if U % P else 0)
    _check(U, P, 1)


@pytest.mark.parametrize("kt,D,H,G,n_cells,T,rows", [
    (L.T_Q8_0, 128, 8, 4, 4096, 1024, 128), (L.T_Q8_0, 128, 8, 4, 8192, 1024, 256),      # two workgroups a unit
    (L.T_F16, 128, 8, 4, 2048, 2048, 128), (L.T_F16, 128, 8, 4, 8192, 2048, 256),        # one
    (L.T_Q4_0, 256, 4, 6, 32768, 170, 128), (L.T_Q4_0, 256, 4, 6, 32768, 171, 256),      # four row tiles of 256 rows, five
    (L.T_F16, 256, 4, 6, 32768, 170, 256),
])
def test_rows_of_a_unit(kt, D, H, G, n_cells, T, rows):
    """Both sides of the rules that choose between 128- and 256-row units."""
    src, got, *_ = prefill_shape(kt, D, H, n_cells, T, H * G, 256)
    assert got == rows
    assert src == (1 if kt == L.T_F16 else 0 if rows == 256 else 2)       # f16 window, converted ahead, by the attention
