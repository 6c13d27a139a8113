"""The split plan of the prefill attention over the row blocks the engine
launches (pf_flash_split, host code in csrc/prefill.hip, through
chk_pf_flash_split_rows; no device call): 16 rows for 8 query heads a kv
head, up to 128 for one.  Every step once, pieces in consecutive slots, and
no more slots than the engine keeps for chunks of that size."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from cherenkov_amd import abi

MAXSEG, NONE = 6, 0xFFFFFFFF


def split(T, pos0, max_wg, rows):
    if not abi.LIB_PATH.exists():
        pytest.skip("libcherenkov.so not built (run __graft_entry__.build())")
    n = max(max_wg, (T + rows - 1) // rows)
    seg, merge = np.zeros(n * MAXSEG * 4, np.uint32), np.zeros(4 * n, np.uint32)
    W, nslots, nmerge = C.c_uint32(), C.c_uint32(), C.c_uint32()
    abi.check(abi.lib().chk_pf_flash_split_rows(T, pos0, max_wg, rows, C.byref(W), C.byref(nslots), seg.ctypes.data, seg.size,
                                                merge.ctypes.data, merge.size, C.byref(nmerge)))
    return (W.value, nslots.value, seg[: W.value * MAXSEG * 4].reshape(W.value, MAXSEG, 4),
            merge[: 4 * nmerge.value].reshape(-1, 4))


def slots_kept(T, ctx, max_wg, rows):
    n = C.c_uint32()
    abi.check(abi.lib().chk_pf_flash_slots(T, ctx, max_wg, rows, C.byref(n)))
    return n.value


@pytest.mark.parametrize("rows", [16, 32, 64, 128])
@pytest.mark.parametrize("max_wg", [1, 4, 32, 128, 256])
def test_split_covers_every_step_once(rows, max_wg):
    for T in (1, rows - 1, rows, rows + 1, 70, 333, 1001, 4096):
        for pos0 in (1, 31, 97, 700, 6500, 250000):
            W, nslots, seg, merge = split(T, pos0, max_wg, rows)
            R = (T + rows - 1) // rows
            tl = [(pos0 + min(rows * rb + rows - 1, T - 1)) // 32 + 1 for rb in range(R)]
            cover = [np.zeros(n, int) for n in tl]
            pieces: dict[int, list[int]] = {}
            for k in range(W):
                for rb, ta, tb, slot in seg[k].tolist():
                    if rb == NONE:
                        break
                    assert rb < R and ta < tb <= tl[rb]
                    cover[rb][ta:tb] += 1
                    assert (ta == 0 and tb == tl[rb]) == (slot == NONE)
                    if slot != NONE:
                        pieces.setdefault(rb, []).append(slot)
            assert all((c == 1).all() for c in cover), (T, pos0)
            assert sorted(s for p in pieces.values() for s in p) == list(range(nslots))
            assert {int(m[0]): (int(m[1]), int(m[2])) for m in merge} == {rb: (min(s), len(s)) for rb, s in pieces.items()}
            for s in pieces.values():
                assert sorted(s) == list(range(min(s), min(s) + len(s))) and len(s) <= 256
            # engines whose context ends with the chunk, and larger ones
            for cap, ctx in ((T, pos0 + T), (T + 5, pos0 + T), (max(T, 1000), pos0 + T + 5000)):
                assert nslots <= slots_kept(cap, ctx, max_wg, rows), (T, pos0, cap, ctx)


def test_slots_kept_bound_every_chunk_of_a_small_engine():
    """Each chunk of up to 96 rows within 400 tokens, any start."""
    for rows in (16, 64):
        for max_wg in (3, 128):
            kept = slots_kept(96, 400, max_wg, rows)
            took = max(split(T, pos0, max_wg, rows)[1] for T in range(1, 97) for pos0 in range(1, 401 - T, 7))
            assert took <= kept <= 2 * max(took, 1) + 8
