"""The split plan of the prefill attention (pf_flash_split, host code in
csrc/prefill.hip, through chk_pf_flash_split; no device call): a chunk with
fewer 16-row blocks than workgroups has its (row block, tile) steps cut
into near-equal ranges.  Every step must be covered once, pieces flagged
and listed in consecutive slots, and the plan stay within the buffers the
engine sizes for max_wg workgroups."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from cherenkov_amd import abi

MAXSEG, NONE = 6, 0xFFFFFFFF


def split(T, pos0, max_wg):
    L = abi.lib()
    n = max(max_wg, (T + 15) // 16)
    seg, merge = np.zeros(n * MAXSEG * 4, np.uint32), np.zeros(4 * n, np.uint32)
    W, nslots, nmerge = C.c_uint32(), C.c_uint32(), C.c_uint32()
    abi.check(L.chk_pf_flash_split(T, pos0, max_wg, C.byref(W), C.byref(nslots), seg.ctypes.data, seg.size,
                                   merge.ctypes.data, merge.size, C.byref(nmerge)))
    return W.value, nslots.value, seg[: W.value * MAXSEG * 4].reshape(W.value, MAXSEG, 4), merge[: 4 * nmerge.value].reshape(-1, 4)


@pytest.mark.parametrize("T", [1, 15, 16, 17, 70, 333, 1001, 2047, 4096])
@pytest.mark.parametrize("pos0", [0, 1, 31, 1500, 5001, 250000])
@pytest.mark.parametrize("max_wg", [1, 7, 128, 256])
def test_split_covers_every_step_once(T, pos0, max_wg):
    if not abi.LIB_PATH.exists():
        pytest.skip("libcherenkov.so not built (run __graft_entry__.build())")
    W, nslots, seg, merge = split(T, pos0, max_wg)
    R = (T + 15) // 16
    tl = [(pos0 + min(16 * rb + 15, T - 1)) // 32 + 1 for rb in range(R)]
    assert W <= max(R, max_wg) and nslots <= 2 * max(W, 1)
    cover = [np.zeros(n, int) for n in tl]
    pieces: dict[int, list[int]] = {}
    shares = []
    for k in range(W):
        live = [tuple(int(v) for v in g) for g in seg[k]]
        live = live[: [g[0] for g in live].index(NONE)] if NONE in [g[0] for g in live] else live
        for rb, ta, tb, slot in live:
            assert rb < R and ta < tb <= tl[rb]
            cover[rb][ta:tb] += 1
            assert (ta == 0 and tb == tl[rb]) == (slot == NONE)
            if slot != NONE:
                pieces.setdefault(rb, []).append(slot)
        shares.append(sum(g[2] - g[1] for g in live))
    assert all((c == 1).all() for c in cover)
    assert {int(m[0]): (int(m[1]), int(m[2])) for m in merge} == {rb: (min(s), len(s)) for rb, s in pieces.items()}
    for s in pieces.values():
        assert sorted(s) == list(range(min(s), min(s) + len(s))) and len(s) <= 256
    if R < W:  # split: equal shares, none below the least
        assert max(shares) - min(shares) <= 1 and min(shares) >= 3
