"""Device scratch of the primitive calls (CallScratch in csrc/engine.cpp):
one allocation while the parts' sum is small or a part is large, one each
where only the sum is large."""

from __future__ import annotations

import time

import numpy as np
import pytest

from cherenkov_amd.abi import check, lib
from tests.gpu_util import assert_close, empty_dev, to_dev, to_host
from tests.numerics import bf16_bits

pytestmark = pytest.mark.gpu

# (outputs, inputs): planes of rows x inputs fp16 around the 2 MB line
OUT, IN = 768, 960


def make(rows, shift=0):
    rng = np.random.default_rng(rows)
    w = rng.integers(0, 2**32, size=(OUT, IN // 8), dtype=np.uint64).astype(np.uint32)
    s = bf16_bits(rng.normal(0, 0.02, size=(OUT, IN // 64)))
    b = bf16_bits(rng.normal(0, 0.01, size=(OUT, IN // 64)))
    words = np.concatenate([np.zeros(shift, np.uint32), w.ravel()])
    x = rng.normal(0, 1, (rows, IN)).astype(np.float32)
    dev = to_dev(words), to_dev(s), to_dev(b), to_dev(x), empty_dev((rows, OUT))
    dw, ds, db, dx, dy = dev
    return dev, x, (w, s, b), lambda: check(lib().chk_q4_gemm(
        dw.data_ptr() + 4 * shift, ds.data_ptr(), db.data_ptr(), OUT, IN, dx.data_ptr(), rows, dy.data_ptr(), None))


# parts' sum below the line, only the sum above it, one part above it
@pytest.mark.parametrize("rows", [500, 551, 600, 1092, 1093, 1200])
def test_gemm_is_one_result_for_any_split_of_its_scratch(have_gpu, rows):
    (_, _, _, _, y), x, (w, s, b), call = make(rows)
    call()
    got = to_host(y)
    (_, _, _, _, y1), _, _, call1 = make(rows, shift=1)  # codes copied: a larger part
    call1()
    assert np.array_equal(got, to_host(y1))
    sc = np.repeat((s.astype(np.uint32) << 16).view(np.float32), 64, 1).astype(np.float64)
    bi = np.repeat((b.astype(np.uint32) << 16).view(np.float32), 64, 1).astype(np.float64)
    code = (w[:, :, None] >> (4 * np.arange(8, dtype=np.uint32))) & 15
    ref = x.astype(np.float64) @ (code.reshape(OUT, IN) * sc + bi).T
    # operands of 22 bits, f32 sums over 960 inputs
    assert_close(got, ref, f"{rows} rows", abs_frac=1e-4, min_cos=0.999999)


def test_call_does_not_jump_where_the_sum_passes_the_line(have_gpu):
    """600 rows hold a fifth more than 500 and take the same launches: 56 us
    against 53, where one mapping of the 2.3 MB sum took 86."""
    (keep_a, _, _, a), (keep_b, _, _, b) = make(500), make(600)

    def best(f):
        for _ in range(5):
            f()
        ts = []
        for _ in range(60):
            t = time.perf_counter()
            f()
            ts.append(time.perf_counter() - t)
        return sorted(ts)[20]

    t500, t600 = min(best(a), best(a)), min(best(b), best(b))
    print(f"500 rows {t500 * 1e6:.1f} us, 600 rows {t600 * 1e6:.1f} us")
    assert t600 < 1.3 * t500
