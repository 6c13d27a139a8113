"""The prefill attention kernel in each of its forms (1, 2, 4 or 8 query
heads a kv head, head dims 128 and 256, dense and under a QSA selection,
row blocks whole and split) at row counts around its blocks (16 rows a
wave, 16 to 128 a workgroup): a chunk behind a context against the row
path, which the model tests pin to the oracle."""

from __future__ import annotations

import numpy as np
import pytest

from cherenkov_amd import presets
from cherenkov_amd.engine import Engine
from tests.gpu_util import assert_close

pytestmark = pytest.mark.gpu


def config(nh, nkv, hd, budget=0, ratio=4):
    # one layer: the last row's logits depend on every row's keys and
    # values, but on no other row's routing (a near-tie there parts two
    # correct paths)
    c = presets.tiny(mtp=0, layers=1)
    c.full_attention_interval = 1
    c.num_attention_heads, c.num_key_value_heads, c.head_dim = nh, nkv, hd
    if budget:
        c.indexer_budget, c.indexer_compress_ratio = budget, ratio
    return c


@pytest.mark.parametrize("nh,nkv,hd,budget,ratio", [(2, 2, 128, 0, 4), (4, 2, 256, 0, 4), (8, 2, 128, 0, 4), (16, 2, 256, 0, 4),
                                                    (2, 2, 256, 64, 4), (4, 2, 128, 63, 3), (8, 2, 256, 32, 1),
                                                    (16, 2, 128, 96, 32)])
@pytest.mark.parametrize("ctx,rows", [(0, 17), (200, 1), (130, 33), (97, 130)])
def test_chunk_attention_matches_row_path(have_gpu, nh, nkv, hd, budget, ratio, ctx, rows):
    cfg = config(nh, nkv, hd, budget, ratio)
    toks = np.random.default_rng(nh * 31 + ctx + rows).integers(0, cfg.vocab_size, size=ctx + rows).tolist()
    a = Engine(cfg, experts=4, drafts=0, max_t=512)
    b = Engine(cfg, experts=4, drafts=0, max_t=512)
    try:
        if ctx:
            a.prefill_chunk(toks[:ctx])
        a.prefill_chunk(toks[ctx:], all_logits=True)
        for t in toks:
            b.step(t)
        # f32-grade both ways (22-bit operands, f32 sums); int8 cache codes
        # may fall on either side of a rounding boundary
        assert_close(a.pf_logits_row(rows - 1), b.logits(), "last row", abs_frac=1e-3, min_cos=0.99999)
        a.reset()
        if ctx + rows > 64:  # the same rows in one chunk: other blocks, other pieces
            a.prefill_chunk(toks)
            assert_close(a.logits(), b.logits(), "one chunk", abs_frac=1e-3, min_cos=0.99999)
    finally:
        a.close()
        b.close()
