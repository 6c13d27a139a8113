"""Prefill attention behind contexts of thousands of tokens, on one layer of
a small model: row blocks joined from dozens of pieces, block scores of more
than one workgroup and row group, and chunks of a few rows past the QSA
budget in the decode step's kernels and in the flash kernel, at the rule's
line and with partials in each of their buffers.  Chunk and row path start
from the same checkpoint."""

from __future__ import annotations

import time

import numpy as np
import pytest

from cherenkov_amd.engine import Engine
from tests.gpu_util import assert_close, torch_dev
from tests.test_flash_split_rows import split
from tests.test_gpu_flash import config

pytestmark = pytest.mark.gpu


def check_chunks(cfg, ctx, rows):
    toks = np.random.default_rng(ctx).integers(0, cfg.vocab_size, size=ctx + max(rows)).tolist()
    e = Engine(cfg, experts=4, drafts=0, max_t=ctx + max(rows) + 8)
    try:
        e.prefill_chunk(toks[:ctx])
        cp = e.save_prefix()
        ref = []
        for t in toks[ctx:]:
            e.step(t)
            ref.append(e.logits())
        for n in rows:
            e.restore_prefix(cp)
            e.prefill_chunk(toks[ctx:ctx + n], all_logits=True)
            for r in {0, n // 2, n - 1}:
                # f32-grade both ways; int8 cache codes may fall on either
                # side of a rounding boundary
                assert_close(e.pf_logits_row(r), ref[r], f"{n} rows behind {ctx}: row {r}", abs_frac=1e-3, min_cos=0.99999)
    finally:
        e.close()


# k_pf_flash_join: more pieces than the four it loads at once, and than the 64
# lanes of a wave hold
@pytest.mark.parametrize("nh,nkv,hd", [(16, 2, 256), (8, 2, 128), (4, 2, 256), (2, 2, 128)])
@pytest.mark.parametrize("ctx,rows,more_than", [(700, (1, 16, 17, 40), 4), (6500, (1, 16, 17), 64)])
def test_blocks_of_many_pieces(have_gpu, nh, nkv, hd, ctx, rows, more_than):
    block = 16 * (8 // (nh // nkv))
    _, _, _, merge = split(min(rows[-1], block), ctx, 256 // nkv, block)
    assert merge[0][2] > more_than
    check_chunks(config(nh, nkv, hd), ctx, rows)


# the scores of rows past the budget stand in a buffer of 64 rows' attention
# partials: 9 MB here, 325 rows of 6908 blocks, so 400 rows take two groups
def test_scores_of_two_row_groups(have_gpu):
    check_chunks(config(2, 2, 128, 64, 1), 6500, (400,))


# the step form holds up to 16 rows behind 700 tokens, 9 (16 heads over 2)
# and 16 (2 over 2) behind 6500
@pytest.mark.parametrize("nh,nkv,hd,budget,ratio", [(16, 2, 256, 64, 4), (2, 2, 256, 64, 4), (8, 8, 128, 63, 3)])
@pytest.mark.parametrize("ctx,rows", [(700, (1, 4, 5, 16, 17)), (6500, (1, 9, 10, 16, 17))])
def test_few_rows_past_the_budget(have_gpu, nh, nkv, hd, budget, ratio, ctx, rows):
    check_chunks(config(nh, nkv, hd, budget, ratio), ctx, rows)


# 64 heads of 128 over 64: the expert output buffer holds partials of five
# rows behind 12000 tokens (six rows: two launches), of three behind 16400
# (then a step batch's buffer, four rows a launch)
@pytest.mark.parametrize("ctx,rows", [(12000, (5, 6)), (16400, (1, 4, 5))])
def test_step_form_partials_in_each_buffer(have_gpu, ctx, rows):
    cfg = config(64, 64, 128, 63, 3)
    cfg.hidden_size, cfg.num_experts_per_tok = 256, 1
    check_chunks(cfg, ctx, rows)


def test_one_row_past_the_budget_costs_what_a_step_does(have_gpu):
    """One row of 8 heads of 128 over 8 behind 64000 tokens against one behind
    1100: 1.6 times in the step's kernels, 2.1 in the flash kernel."""
    cfg = config(8, 8, 128, 1024, 2)
    best = {}
    for ctx in (1100, 64000):
        toks = np.random.default_rng(ctx).integers(0, cfg.vocab_size, size=ctx + 1).tolist()
        e = Engine(cfg, experts=4, drafts=0, max_t=ctx + 8)
        try:
            e.prefill_chunk(toks[:ctx])
            cp = e.save_prefix()
            ts = []
            for _ in range(30):
                e.restore_prefix(cp)
                torch_dev().cuda.synchronize()
                t = time.perf_counter()
                e.prefill_chunk(toks[ctx:])
                ts.append(time.perf_counter() - t)
            best[ctx] = sorted(ts)[5]
        finally:
            e.close()
    print({k: f"{v * 1e6:.0f} us" for k, v in best.items()})
    assert best[64000] < 1.85 * best[1100]
