"""The prefill GEMMs' forms for few rows: 32-row tiles, K chunks of the
hyper-connection, input and out projections (their partials summed by the
next pass), expert tiles of 32 rows.  One layer of the 80B shape at row
counts around the tiles and around each rule's bound, as a prompt's first
chunk (which keeps its K chunks) and behind a context, in engines of two
capacities, against the row path; and the bits at any capacity."""

from __future__ import annotations

import numpy as np
import pytest

from cherenkov_amd import presets
from cherenkov_amd.engine import Engine
from tests.gpu_util import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,interval", [(4, 4), (4, 1), (3, 4), (2, 4)])
def test_few_rows_match_row_path(have_gpu, bits, interval):
    cfg = presets.qwen3next_80b_shape(layers=1, mtp=0)
    cfg.full_attention_interval = interval
    toks = np.random.default_rng(bits * 10 + interval).integers(0, cfg.vocab_size, size=455).tolist()
    rows = [1, 15, 16, 17, 33, 65, 128, 129, 161, 300] + ([410, 450] if bits == 4 and interval == 4 else [])
    b = Engine(cfg, experts=bits, drafts=0, max_t=512)
    ref = {}
    try:
        for i, t in enumerate(toks[:max(rows) + 5]):
            b.step(t)
            if i + 1 in rows or i - 4 in rows:
                ref[i + 1] = b.logits()
    finally:
        b.close()
    for max_t in (2048, 512):
        a = Engine(cfg, experts=bits, drafts=0, max_t=max_t)
        try:
            for n, ctx in [(n, ctx) for n in rows for ctx in (0, 5)]:
                a.reset()
                if ctx:
                    a.prefill_chunk(toks[:ctx])
                a.prefill_chunk(toks[ctx:ctx + n])
                # one layer: only the last row's own routing matters; f32-grade
                # sums in another order
                assert_close(a.logits(), ref[ctx + n], f"{bits} bits, {n} rows behind {ctx}, max_t {max_t}", abs_frac=1e-3, min_cos=0.99999)
        finally:
            a.close()


def small(nh, nkv, hd):
    c = presets.tiny(mtp=0, layers=1)
    c.full_attention_interval = 1
    c.num_attention_heads, c.num_key_value_heads, c.head_dim = nh, nkv, hd
    return c


@pytest.mark.parametrize("make", [lambda: presets.qwen3next_80b_shape(layers=1, mtp=0), lambda: small(16, 2, 256),
                                  lambda: small(2, 2, 128)], ids=["80b", "16x256", "2x128"])
@pytest.mark.parametrize("interval", [4, 1])
def test_a_chunk_is_the_same_at_any_capacity(have_gpu, make, interval):
    """K chunks, attention shares and their partials follow the chunk, the
    shape and the device: the same rows behind the same context give the
    same bits in engines of any max_t that hold them."""
    cfg = make()
    cfg.full_attention_interval = interval
    toks = np.random.default_rng(interval).integers(0, cfg.vocab_size, size=420).tolist()
    got = {}
    for max_t in (424, 1200, 5000):
        e = Engine(cfg, experts=4, drafts=0, max_t=max_t)
        try:
            e.prefill_chunk(toks[:120])
            cp = e.save_prefix()
            for n in (1, 5, 17, 70, 128, 129, 300):
                e.restore_prefix(cp)
                e.prefill_chunk(toks[120:120 + n])
                got[max_t, n] = e.logits().copy()
                assert np.array_equal(got[max_t, n], got[424, n]), (max_t, n)
        finally:
            e.close()
