"""The launch rules of the dense prefill GEMMs (pf_ksplit, pf_dense_tile_rows
in csrc/prefill.hip, through chk_pf_gemm_form; no device call): K chunks
and 32-row tiles fill the compute units the device has, and no more."""

from __future__ import annotations

import ctypes as C

import pytest

from cherenkov_amd import abi


def form(N, K, M, least, most, cus, per_cu=1):
    if not abi.LIB_PATH.exists():
        pytest.skip("libcherenkov.so not built (run __graft_entry__.build())")
    ks, rows = C.c_uint32(), C.c_uint32()
    abi.check(abi.lib().chk_pf_gemm_form(N, K, M, least, most, cus, per_cu, C.byref(ks), C.byref(rows)))
    return ks.value, rows.value


@pytest.mark.parametrize("M,whole,eighth", [(70, (16, 32), (8, 64)), (256, (16, 32), (4, 64)), (512, (16, 32), (4, 64)),
                                            (2048, (4, 64), (4, 64))])
def test_down_inject_of_8192_inputs(M, whole, eighth):
    # a whole device, and one of eight partitions of it
    assert form(324, 8192, M, 4, 16, 256) == whole
    assert form(324, 8192, M, 4, 16, 32) == eighth


@pytest.mark.parametrize("N,K", [(256, 512), (324, 8192), (2048, 4096), (12288, 2048), (333, 960)])
@pytest.mark.parametrize("M", [1, 32, 33, 64, 65, 333, 1000, 4096])
@pytest.mark.parametrize("cus", [32, 64, 128, 256])
@pytest.mark.parametrize("least,most,per_cu", [(1, 1, 1), (1, 4, 2), (2, 8, 1)])
def test_launches_stay_within_the_device(N, K, M, cus, least, most, per_cu):
    ks, rows = form(N, K, M, least, most, cus, per_cu)
    wg64 = (N + 255) // 256 * ((M + 63) // 64)
    assert least <= ks <= max(least, most) and (ks == least or (K // 64 // ks % 8 == 0 and wg64 * ks <= per_cu * cus))
    wg32 = (N + 255) // 256 * ((M + 31) // 32) * ks
    assert rows == (32 if wg32 <= cus or (K // 64 // ks <= 8 and wg32 <= 3 * cus) else 64)
