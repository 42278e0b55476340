"""The shape of a prefill launch, on the host: every piece of a unit has a slot of
its own within the workspace, and the merge asks the workgroups that have them."""
import ctypes as C
import random

import pytest

from kvmem_amd import _lib as L

lib = L.load()
lib.kvm_fa_prefill_slot.restype = lib.kvm_fa_prefill_slots.restype = C.c_uint32


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
    out = (C.c_uint32 * 7)()
    assert lib.kvm_fa_prefill_shape(L.T_Q8_0, D, H, n_cells, T, H * G, 256, out) == 0
    src, rows, n_row_tiles, n_seg, U, P, slots = out
    assert n_seg > 1 and U > P and U % P and U == n_row_tiles * H * n_seg
    assert slots == lib.kvm_fa_prefill_slots(U, P, n_seg)
    _check(U, P, n_seg)
