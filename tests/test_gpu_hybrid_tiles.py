"""Products of more than 16 rows on the hybrid engine's bf16 path: every tile form at its edges.

The tile forms add an output's products in the same order, so the logits of a row have to be the same bits whichever form the number of
rows and columns picks; the smallest form is held to the float64 restatement by the design's own tests.  Gate and up products with their
activation behind them, dense and routed, are held to the restatement at sizes that pick each form."""
import pytest
import torch

from oracle import kazozen_ref as KR
from tests import hybrid_util as U
from tests import kazozen_util as P
from vox_serve_amd.engine_hybrid import HybridEngine
from vox_serve_amd.model import kazozen

pytestmark = pytest.mark.gpu

BF16_BAR = 4e-2     # relative RMS over the vocabulary, as in the design's tests


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


# (rows, vocabulary): 192 x 128 (remainders of 2 rows and 1 column), 128 x 64 twice, 192 x 128 of one k-tile, against the 64 x 64 that 17 rows take
@pytest.mark.parametrize("rows,vocab,width", [(130, 16769, 128), (255, 14400, 192), (65, 19201, 128), (129, 28673, 64)])
def test_a_row_has_the_same_logits_in_every_tile_form(rows, vocab, width):
    cfg = P.config([P.attention(heads=2, kv_heads=1, dim=32, vdim=32, size=50, keep=2)], width=width, vocab=vocab, bigram=None)
    d = kazozen.config_from_dict(cfg)
    eng = HybridEngine(d, kazozen.pack_weights(P.random_checkpoint(cfg, seed=rows), d), dtype=torch.bfloat16, max_batch=1, page_size=16, max_pages=20,
                       max_seq_len=320, max_prefill_rows=rows, max_out=rows)
    toks = torch.randint(0, vocab, (rows,), generator=torch.Generator().manual_seed(7), dtype=torch.int32)
    eng.row_ids[:rows, 0] = toks.cuda()

    def logits(out):
        npg = (rows + 15) // 16
        eng.upload_plan(pos=range(rows), kvlen=range(1, rows + 1), page=[t // 16 for t in range(rows)], slot=[t % 16 for t in range(rows)], q_req=[0] * rows,
                        last_rows=out, indptr=[0, npg], indices=range(npg), req_rows=[0, rows], state=[0])
        eng.step(rows, 1, len(out), sample=False, max_kvlen=rows)
        return eng.out_logits[: len(out)].clone()
    try:
        whole = logits(list(range(rows)))
        for a in range(0, rows, 17):
            part = list(range(min(a, rows - 17), min(a, rows - 17) + 17))      # 17 rows: tiles of 64
            assert torch.equal(logits(part), whole[part]), (rows, vocab, a)
    finally:
        eng.close()


@pytest.mark.parametrize("rows,mlp", [(130, P.dense(8384)), (129, P.dense(7424)), (65, P.dense(9600)), (17, P.dense(64)), (70, P.moe(4, 4, 3840, 0, 0)),
                                      (131, P.moe(4, 4, 2176, 2, 2)), (67, P.moe(6, 2, 2560, 3, 2)), (33, P.moe(3, 1, 64, 0, 0))])
def test_activation_behind_both_products(rows, mlp):
    cfg = P.config([P.attention(heads=2, kv_heads=1, dim=32, vdim=32, size=50, keep=2, mlp=mlp)], width=64, vocab=50)
    S = P.random_checkpoint(cfg, seed=3)
    toks = torch.randint(0, 50, (rows,), generator=torch.Generator().manual_seed(rows)).tolist()
    d = U.Driver(cfg, S, dtype=torch.bfloat16, page_size=16, pages=20, max_rows=rows)
    try:
        got = d.run_cut("r", toks, [rows])
    finally:
        d.close()
    # (a routed layer: a choice that bf16 rounding flips moves a whole row, so the bar holds for nine rows of ten)
    err = U.rel_err(got, KR.forward(cfg, S, toks), None if mlp["kind"] == "dense" else 0.9)
    assert err < BF16_BAR, err


# K of the second product = the layer's inner width: one step into the second round of requests, two whole rounds, one step into the third,
# three whole rounds and one step into a fourth; up to eight rows the unit's own launch, more the general one, which zeroes early
@pytest.mark.parametrize("rows,inner", [(2, 2080), (16, 4096), (7, 4128), (8, 6144), (16, 6176)])
def test_rounds_of_a_few_row_product(rows, inner):
    cfg = P.config([P.attention(heads=2, kv_heads=1, dim=32, vdim=32, size=50, keep=2, mlp=P.dense(inner))], width=64, vocab=50)
    S = P.random_checkpoint(cfg, seed=5)
    toks = torch.randint(0, 50, (rows,), generator=torch.Generator().manual_seed(rows)).tolist()
    d = U.Driver(cfg, S, dtype=torch.bfloat16, page_size=16, pages=20, max_rows=rows)
    try:
        got = d.run_cut("r", toks, [rows])
    finally:
        d.close()
    assert U.rel_err(got, KR.forward(cfg, S, toks)) < BF16_BAR


# The general few-row product where it zeroes late: up to eight rows of few columns, K = heads x 32 (a whole round of requests, a step into the second, two
# whole rounds, a step into the fourth) ...
@pytest.mark.parametrize("rows,heads", [(2, 64), (8, 65), (7, 128), (8, 193)])
def test_rounds_of_a_few_row_product_of_few_columns(rows, heads):
    cfg = P.config([P.attention(heads=heads, kv_heads=1, dim=8, vdim=32, size=50, keep=2)], width=64, vocab=50)
    S = P.random_checkpoint(cfg, seed=heads)
    toks = torch.randint(0, 50, (rows,), generator=torch.Generator().manual_seed(rows)).tolist()
    d = U.Driver(cfg, S, dtype=torch.bfloat16, page_size=16, pages=20, max_rows=rows)
    try:
        got = d.run_cut("r", toks, [rows])
    finally:
        d.close()
    assert U.rel_err(got, KR.forward(cfg, S, toks)) < BF16_BAR


# ... and of many columns, K = width: a few steps, a whole round
@pytest.mark.parametrize("rows,width", [(2, 96), (7, 2048)])
def test_few_row_product_of_many_columns(rows, width):
    cfg = P.config([P.attention(heads=2, kv_heads=1, dim=32, vdim=32, size=50, keep=2)], width=width, vocab=8200)
    S = P.random_checkpoint(cfg, seed=width)
    toks = torch.randint(0, 8200, (rows,), generator=torch.Generator().manual_seed(rows)).tolist()
    d = U.Driver(cfg, S, dtype=torch.bfloat16, page_size=16, pages=20, max_rows=rows)
    try:
        got = d.run_cut("r", toks, [rows])
    finally:
        d.close()
    assert U.rel_err(got, KR.forward(cfg, S, toks)) < BF16_BAR


# the other tiles: 32 x 32, 64 x 32, 128 x 64, 128 x 128, 192 x 128, 256 x 128, 256 x 192, 256 x 160 (whose columns do not divide among the waves), rows
# and columns with remainders; most with fewer k-tiles than stages (a stage that is filled again: test_gpu_hybrid_order.py)
@pytest.mark.parametrize("rows,vocab,width", [(33, 515, 192), (63, 6145, 512), (65, 8193, 64), (65, 16769, 256), (129, 24001, 64), (255, 28673, 128),
                                              (257, 16769, 192), (257, 16769, 512)])
def test_a_row_has_the_same_logits_in_every_tile(rows, vocab, width):
    test_a_row_has_the_same_logits_in_every_tile_form(rows, vocab, width)


# gate and up products in 64 x 64, 192 x 128 and 256 x 192, columns that are no multiple of a block's, one k-tile
@pytest.mark.parametrize("rows,mlp", [(300, P.dense(1088)), (129, P.dense(8384)), (300, P.dense(11328)), (257, P.dense(16448)), (131, P.moe(4, 4, 5632, 0, 0))])
def test_activation_behind_both_products_in_every_tile(rows, mlp):
    test_activation_behind_both_products(rows, mlp)


# Window attention of 64 and 128 dims, steps of more rows than the few-row form takes: 1, 2, 8, 16 and 32 query heads to a key head (a block's 64
# columns are 64 to 2 rows), pages that are no power of two, kept tokens before the window, portions that start inside and behind it
@pytest.mark.parametrize("heads,kv,dim,page,window,keep,cuts", [(2, 2, 64, 16, 70, 3, [65, 66, 70]), (4, 2, 128, 24, 40, 5, [130, 67]), (8, 1, 64, 8, 300, 0, [129, 90]),
                                                                (16, 1, 128, 32, 64, 70, [200, 65]), (32, 1, 64, 40, 33, 1, [67, 66]), (3, 1, 64, 16, 50, 2, [70, 66])])
def test_window_attention_heads_of_a_key_head_together(heads, kv, dim, page, window, keep, cuts):
    cfg = P.config([P.attention(heads=heads, kv_heads=kv, dim=dim, vdim=dim, size=window, keep=keep, mlp=P.dense(64))], width=64, vocab=50)
    S = P.random_checkpoint(cfg, seed=heads, gain=1.3)
    n = sum(cuts)
    toks = torch.randint(0, 50, (n,), generator=torch.Generator().manual_seed(dim + n)).tolist()
    d = U.Driver(cfg, S, dtype=torch.bfloat16, page_size=page, pages=(n + page - 1) // page + 1, max_rows=max(cuts))
    try:
        got = d.run_cut("r", toks, cuts)
    finally:
        d.close()
    assert U.rel_err(got, KR.forward(cfg, S, toks)) < BF16_BAR


# 2 to 16 rows: units of a dense layer in one launch each (an inner width of one round of requests, of one step into the second; nine rows
# and an inner width that is no multiple of 32 go on in the general product), routed layers whose experts have one entry, several and all rows, rows of
# one piece and of several
@pytest.mark.parametrize("rows,mlp", [(2, P.dense(64)), (8, P.dense(4096)), (7, P.dense(4224)), (9, P.dense(4224)), (5, P.dense(104)), (16, P.dense(2080)),
                                      (2, P.moe(2, 2, 64, 0, 0)), (8, P.moe(3, 1, 2048, 0, 0)), (7, P.moe(5, 5, 2112, 0, 0)), (8, P.moe(48, 6, 128, 4, 2)),
                                      (3, P.moe(48, 16, 64, 0, 0)), (6, P.moe(8, 2, 96, 0, 0))])
def test_few_row_units(rows, mlp):
    test_activation_behind_both_products(rows, mlp)


# ... beside a layer whose choices include outputs without an expert, and one whose weights multiply an expert's input
@pytest.mark.parametrize("rows", [2, 8])
@pytest.mark.parametrize("over", [dict(identity=5), dict(scale_input=True)])
def test_few_row_routed_forms(rows, over):
    import dataclasses
    cfg = P.config([P.attention(heads=2, kv_heads=1, dim=32, vdim=32, size=50, keep=2, mlp=P.moe(6, 3, 64, 0, 0))], width=64, vocab=50)
    base = kazozen.config_from_dict(cfg)
    layer = base.layers[-1]
    d = dataclasses.replace(base, layers=[*base.layers[:-1], dataclasses.replace(layer, moe=dataclasses.replace(layer.moe, **over))])
    W = kazozen.pack_weights(P.random_checkpoint(cfg, seed=3), base)
    n_out = layer.moe.experts + d.layers[-1].moe.identity
    g = torch.Generator().manual_seed(1)
    W["layers"][-1]["moe"].update(router=torch.randn(n_out, d.width, generator=g), correction=torch.zeros(n_out))
    toks = torch.randint(0, 50, (9,), generator=g, dtype=torch.int32)

    def logits(cuts):
        eng = HybridEngine(d, W, dtype=torch.bfloat16, max_batch=1, page_size=16, max_pages=2, max_seq_len=32, max_prefill_rows=16, max_out=16)
        out, at = [], 0
        try:
            for n in cuts:
                eng.row_ids[:n, 0] = toks[at: at + n].cuda()
                eng.upload_plan(pos=range(at, at + n), kvlen=range(at + 1, at + n + 1), page=[0] * n, slot=range(at, at + n), q_req=[0] * n, last_rows=list(range(n)),
                                indptr=[0, 1], indices=[0], req_rows=[0, n], state=[0])
                eng.step(n, 1, n, sample=False, max_kvlen=at + n)
                out.append(eng.out_logits[:n].float().cpu().clone())
                at += n
        finally:
            eng.close()
        return torch.cat(out)
    # one row at a time takes each entry's vectors apart; the bar is that of the other bf16 comparisons
    err = U.rel_err(logits([rows]), logits([1] * rows))
    assert err < BF16_BAR, err


# Steps of up to 32 rows, four heads of a key head at 128 dims: one and three of 16-key groups, a chunk's last key, kept tokens before the window, two
# key heads, groups of eight heads, and (4170 keys) two chunks to a block
@pytest.mark.parametrize("heads,kv,page,window,keep,cuts", [(4, 1, 16, 300, 0, [17, 31, 16, 1, 2]), (8, 2, 24, 70, 5, [130, 3, 32]), (8, 1, 40, 64, 70, [140, 1, 5]),
                                                            (4, 1, 128, 5000, 0, [2080, 2080, 10])])
def test_window_attention_of_few_rows(heads, kv, page, window, keep, cuts):
    test_window_attention_heads_of_a_key_head_together(heads, kv, 128, page, window, keep, cuts)


# Stacks of post-normed layers, more than 16 rows: the rows that every product reads are left as bf16 by the norm before it (rows of one, two and four
# pieces of 1024 columns, and of a width that it takes element by element); up to 6300 entries, listed in one round of 1024 and in several.  (All experts
# are chosen: no choice that bf16 rounding could flip, so every row counts.)
@pytest.mark.parametrize("rows,width", [(17, 64), (40, 1088), (33, 2112), (20, 70), (700, 128)])
def test_stack_of_post_normed_layers(rows, width):
    a = dict(heads=2, kv_heads=1, dim=32, vdim=32, size=50, keep=2)
    cfg = P.config([P.attention(mlp=P.dense(128), **a), P.attention(mlp=P.moe(4, 4, 64, 0, 0), kv_from=0, **a), P.attention(mlp=P.moe(9, 9, 64, 3, 3), **a)], width=width,
                   vocab=50)
    S = P.random_checkpoint(cfg, seed=width)
    toks = torch.randint(0, 50, (rows,), generator=torch.Generator().manual_seed(rows)).tolist()
    d = U.Driver(cfg, S, dtype=torch.bfloat16, page_size=16, pages=(rows + 15) // 16, max_rows=rows)
    try:
        got = d.run_cut("r", toks, [rows])
    finally:
        d.close()
    err = U.rel_err(got, KR.forward(cfg, S, toks))
    assert err < BF16_BAR, err
