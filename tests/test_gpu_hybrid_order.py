"""GPU: the hybrid engine's launches for some sizes against the ones that serve any size, on the same weights and tokens: the same bits.

A choice of experts turns on the last bit of what the router reads, so a form that adds in another order moves a row by an expert now and
then.  `vox_hybrid_set_general` sends every step of an engine to the general launches."""
import dataclasses

import pytest
import torch

from tests import dipivik_util as DU
from tests import fusanex_util as FU
from tests import gaparax_util as GU
from tests import hybrid_util as U
from tests import kazozen_util as P
from tests import sizitar_util as ZU
from vox_serve_amd.engine_hybrid import HybridEngine
from vox_serve_amd.model import kazozen

pytestmark = pytest.mark.gpu

PLAIN, GATED, JOIN = 0, 1, 2


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def tokens(n, vocab, seed):
    return torch.randint(0, vocab, (n,), generator=torch.Generator().manual_seed(seed)).tolist()


def check(cfg, S, n, cuts, tiles=(), page=16, requests=1):
    """The logits of n tokens fed in portions of the given sizes, then one by one (by several requests beside each other), in both modes.
    tiles: (kind, rows, n, k, groups, rows and columns of the tile) that the sized mode takes on the way."""
    out = []
    for general in (0, 1):
        d = U.Driver(cfg, S, dtype=torch.bfloat16, page_size=page, pages=requests * ((n + page - 1) // page + 1), max_rows=max(max(cuts), 17) * requests, max_batch=requests,
                     slots=requests)
        eng = d.model.engine
        for kind, rows, cols, k, groups, bm, bn in tiles:
            t = eng.L.vox_hybrid_tile(kind, rows, cols, k, groups)
            assert (t >> 16, t & 0xffff) == (bm, bn), (kind, rows, cols, k, t >> 16, t & 0xffff)
        eng.L.vox_hybrid_set_general(eng.h, general)
        toks = {f"r{i}": tokens(n, cfg["vocab"], 3 + i) for i in range(requests)}
        got, at = [], 0
        try:
            for c in list(cuts) + [1] * n:
                if at >= n:
                    break
                fed = d.feed([(r, t[at: at + c]) for r, t in toks.items()])
                got += [fed[r] for r in toks]
                at += c
        finally:
            d.close()
        out.append(torch.cat(got))
    assert torch.isfinite(out[0]).all() and out[0].std() > 0
    assert torch.equal(out[0], out[1]), (out[0] != out[1]).any(1).nonzero().flatten().tolist()[:8]


ATT = dict(heads=2, kv_heads=1, dim=32, vdim=32, size=50, keep=2)


# The head in every tile of a plain product: more k-tiles than stages and one more round of them, rows and columns with remainders (a step's
# output rows are its tokens and one per request)
@pytest.mark.parametrize("rows,vocab,bm,bn", [(17, 1025, 32, 32), (33, 5013, 64, 32), (17, 9001, 64, 64), (65, 9001, 128, 64), (65, 16977, 128, 128), (129, 16977, 192, 128),
                                              (193, 16977, 256, 128), (257, 20965, 256, 192), (65, 32929, 256, 160)])
def test_plain_products(rows, vocab, bm, bn):
    cfg = P.config([P.attention(**ATT)], width=768, vocab=vocab, bigram=None)
    check(cfg, P.random_checkpoint(cfg, seed=rows), rows - 1, [rows - 1], [(PLAIN, rows, vocab, 768, 1, bm, bn)])


# Gate and up products with their activation in every tile of theirs, dense, against products and activation apart
@pytest.mark.parametrize("rows,ff,bm,bn", [(17, 64, 32, 64), (33, 4160, 64, 64), (65, 4160, 128, 64), (65, 8256, 128, 128), (129, 8256, 192, 128), (193, 8256, 256, 128),
                                           (129, 16448, 256, 192)])
def test_gated_products(rows, ff, bm, bn):
    cfg = P.config([P.attention(mlp=P.dense(ff), **ATT)], width=512, vocab=50)
    check(cfg, P.random_checkpoint(cfg, seed=ff), rows, [rows], [(GATED, rows, ff, 512, 1, bm, bn)])


# ... and of eight experts, whose rows are gathered: the first column of tiles is that of the gate and up products, the second that of the down products.
# All experts take all rows; in the last two lines two and three of eight are chosen, so the experts have unequal numbers of rows
@pytest.mark.parametrize("rows,width,ff,top,up,down", [(17, 64, 640, 8, None, (32, 32)), (33, 576, 576, 8, (64, 64), (64, 32)), (17, 1088, 512, 8, (32, 64), (64, 64)),
                                                       (65, 512, 576, 8, (128, 64), None), (65, 1088, 1088, 8, (128, 128), (128, 64)), (65, 2112, 512, 8, (64, 64), (128, 128)),
                                                       (129, 2112, 1088, 8, (192, 128), (192, 128)), (193, 2112, 1088, 8, (256, 128), (256, 128)),
                                                       (257, 2112, 512, 8, None, (256, 160)), (257, 2624, 512, 8, None, (256, 192)), (129, 512, 2112, 8, (256, 192), None),
                                                       (700, 512, 576, 2, None, None), (1030, 320, 128, 3, None, None)])
def test_routed_products(rows, width, ff, top, up, down):
    cfg = P.config([P.attention(mlp=P.moe(8, top, ff, 0, 0), **ATT)], width=width, vocab=50)
    each = -(-rows * top // 8)
    tiles = ([(GATED, each, ff, width, 8, *up)] if up else []) + ([(PLAIN, each, width, ff, 8, *down)] if down else [])
    check(cfg, P.random_checkpoint(cfg, seed=ff), rows, [rows], tiles, page=64)


# Sums that join two gated residual streams (closing products of the mixer and of the dense unit), and routed ones
@pytest.mark.parametrize("rows,width,k,tile", [(33, 512, 640, (32, 32)), (520, 2432, 640, (64, 32)), (850, 1856, 640, (64, 64)), (850, 2368, 1280, (128, 128))])
def test_products_that_join_streams(rows, width, k, tile):
    cfg = GU.config([GU.attention(heads=k // 64, kv_heads=k // 128, dim=32, vdim=64, size=64, bias_max=40, rows=16, mlp=GU.dense(k))], width=width, vocab=50)
    check(cfg, GU.random_checkpoint(cfg, seed=rows), rows, [rows], [(JOIN, rows, width, k, 1, *tile)], page=64)


@pytest.mark.parametrize("streams,width", [(2, 512), (2, 70), (3, 96), (4, 128)])
def test_routed_sums_that_join_streams(streams, width):
    cfg = GU.config([GU.attention(mlp=GU.moe(experts=8, top=2, ff=64, count=4, keep=2)), GU.latent(mlp=GU.moe(experts=6, top=3, ff=64))], width=width, vocab=50, streams=streams)
    check(cfg, GU.random_checkpoint(cfg, seed=streams), 120, [100, 5, 8])


# 2 to 16 rows, dense units: K of the gate and up products up to one round of requests, of two whole rounds, one step into the second and the
# third; inner widths of one and several rounds, and none (no multiple of 32); nine rows and more and a width above 2048 leave the down product to
# the general launch
@pytest.mark.parametrize("width,ff,cuts", [(64, 64, [2, 3, 8, 16]), (512, 4224, [8, 7, 9, 16]), (2048, 5632, [8, 2, 9]), (2080, 96, [2, 16, 5]), (4096, 64, [8, 3, 12]),
                                           (4128, 104, [7, 9]), (1024, 2080, [8, 4, 16]), (256, 6176, [8, 5])])
def test_dense_units_of_few_rows(width, ff, cuts):
    cfg = P.config([P.attention(mlp=P.dense(ff), **ATT), P.attention(mlp=P.dense(ff, limit=7.0), kv_from=0, **ATT)], width=width, vocab=50)
    check(cfg, P.random_checkpoint(cfg, seed=width), sum(cuts) + 2, cuts)


# Products of 2 to 16 rows whose columns make more tiles than there are CUs (a head's, and gate and up): one tile more, whole rounds, a last round of one block,
# a last tile of one column; every K that a wave's registers hold, with the rows' requests of several requests a step
@pytest.mark.parametrize("width,vocab,ff,cuts", [(512, 4097, 2056, [8, 16, 2]), (1024, 8192, 4096, [3, 9]), (1536, 8193, 64, [16, 5]), (2048, 12305, 2064, [7, 2, 16])])
def test_more_column_tiles_than_cus(width, vocab, ff, cuts):
    cfg = P.config([P.attention(mlp=P.dense(ff), **ATT)], width=width, vocab=vocab, bigram=None)
    check(cfg, P.random_checkpoint(cfg, seed=width), sum(cuts) + 2, cuts)


# 2 to 8 rows, routed layers of wide experts (inner widths of 2048 and more, or many weights in all): rows of one piece, of a few columns into the next, of
# two whole rounds; one to 64 entries, an odd one at the end; inner widths of one round, a few columns into the next, two rounds, and less than one piece
@pytest.mark.parametrize("width,moe,cuts", [(64, (2, 2, 2048, 0, 0), [2, 8, 3]), (512, (3, 1, 4096, 0, 0), [8, 7]), (2048, (8, 2, 2048, 4, 2), [8, 2, 5]),
                                            (2056, (4, 2, 2048, 0, 0), [8, 3]), (4096, (5, 5, 2056, 0, 0), [7, 8, 2]), (3080, (4, 3, 2120, 0, 0), [4, 6]),
                                            (256, (48, 6, 2048, 4, 2), [8, 6]), (64, (48, 16, 2048, 0, 0), [3, 4]), (128, (16, 8, 4104, 0, 0), [8, 8]),
                                            (4096, (8, 8, 168, 0, 0), [8]), (4096, (4, 1, 2048, 0, 0), [8, 3]), (4096, (4, 2, 1032, 0, 0), [8, 5]), (2052, (8, 2, 2048, 0, 0), [6, 8])])
def test_routed_layers_of_few_rows(width, moe, cuts):
    cfg = P.config([P.attention(mlp=P.moe(*moe), **ATT), P.attention(mlp=P.moe(*moe), kv_from=0, **ATT)], width=width, vocab=50)
    check(cfg, P.random_checkpoint(cfg, seed=width), sum(cuts) + 2, cuts)


# ... with outputs that have no expert, and with weights that multiply an expert's input; two choices and 8192 sums and more take the walk of the down rows
@pytest.mark.parametrize("rows", [2, 5, 8, 40])
@pytest.mark.parametrize("over", [dict(identity=5), dict(scale_input=True), dict(identity=5, scale_input=True)])
@pytest.mark.parametrize("width,top,ff", [(64, 3, 2048), (2056, 2, 2048), (64, 2, 2048)])
def test_routed_forms(rows, over, width, top, ff):
    cfg = P.config([P.attention(heads=2, kv_heads=1, dim=32, vdim=32, size=50, keep=2, mlp=P.moe(6, top, ff, 0, 0))], width=width, vocab=50)
    base = kazozen.config_from_dict(cfg)
    layer = base.layers[-1]
    d = dataclasses.replace(base, layers=[*base.layers[:-1], dataclasses.replace(layer, moe=dataclasses.replace(layer.moe, **over))])
    W = kazozen.pack_weights(P.random_checkpoint(cfg, seed=3), base)
    n_out = layer.moe.experts + d.layers[-1].moe.identity
    g = torch.Generator().manual_seed(1)
    W["layers"][-1]["moe"].update(router=torch.randn(n_out, d.width, generator=g), correction=torch.zeros(n_out))
    toks = torch.randint(0, 50, (rows,), generator=g, dtype=torch.int32)
    out = []
    for general in (0, 1):
        eng = HybridEngine(d, W, dtype=torch.bfloat16, max_batch=1, page_size=64, max_pages=2, max_seq_len=128, max_prefill_rows=64, max_out=64)
        eng.L.vox_hybrid_set_general(eng.h, general)
        try:
            eng.row_ids[:rows, 0] = toks.cuda()
            eng.upload_plan(pos=range(rows), kvlen=range(1, rows + 1), page=[0] * rows, slot=range(rows), q_req=[0] * rows, last_rows=list(range(rows)), indptr=[0, 1],
                            indices=[0], req_rows=[0, rows], state=[0])
            eng.step(rows, 1, rows, sample=False, max_kvlen=rows)
            out.append(eng.out_logits[:rows].float().cpu().clone())
        finally:
            eng.close()
    assert torch.isfinite(out[0]).all() and torch.equal(out[0], out[1])


# Window attention, prompts and then few rows: 1, 2, 4, 8, 16 and 32 query heads to a key head, pages that are no power of two, kept tokens before the
# window, portions that start inside and behind it, (4170 keys) two chunks to a block of the few-row form
@pytest.mark.parametrize("heads,kv,dim,page,window,keep,cuts", [(2, 2, 64, 16, 70, 3, [65, 66, 70, 8]), (4, 2, 128, 24, 40, 5, [130, 67, 9]), (8, 1, 64, 8, 300, 0, [129, 90, 2]),
                                                                (16, 1, 128, 32, 64, 70, [200, 65, 16]), (32, 1, 64, 40, 33, 1, [67, 66, 3]),
                                                                (4, 1, 128, 16, 300, 0, [17, 31, 16, 1, 2]), (8, 2, 128, 24, 70, 5, [130, 3, 32]),
                                                                (8, 1, 128, 40, 64, 70, [140, 1, 5]), (4, 1, 128, 128, 5000, 0, [2080, 2080, 10])])
def test_window_attention(heads, kv, dim, page, window, keep, cuts):
    cfg = P.config([P.attention(heads=heads, kv_heads=kv, dim=dim, vdim=dim, size=window, keep=keep, mlp=P.dense(64))], width=64, vocab=50)
    check(cfg, P.random_checkpoint(cfg, seed=heads, gain=1.3), sum(cuts) + 2, cuts, page=page)


# ... and of several requests beside each other
@pytest.mark.parametrize("requests,cuts", [(2, [33, 4, 1]), (5, [70, 1, 2]), (8, [20, 1])])
def test_window_attention_of_requests(requests, cuts):
    cfg = P.config([P.attention(heads=8, kv_heads=2, dim=128, vdim=128, size=40, keep=3, mlp=P.moe(8, 2, 2048, 4, 2)),
                    P.attention(heads=8, kv_heads=2, dim=128, vdim=128, size=40, keep=3, mlp=P.dense(96), kv_from=0)], width=256, vocab=50)
    check(cfg, P.random_checkpoint(cfg, seed=requests), sum(cuts) + 2, cuts, requests=requests)


# Stacks of post-normed layers, more than 16 rows: the norm leaves the rows that a product reads as bf16 (rows of one, two and four pieces of 1024
# columns, and of a width that it takes element by element); entries of an expert listed in one round and in several
@pytest.mark.parametrize("rows,width", [(17, 64), (40, 1088), (33, 2112), (20, 4096), (20, 70), (700, 128)])
def test_stack_of_post_normed_layers(rows, width):
    cfg = P.config([P.attention(mlp=P.dense(128), **ATT), P.attention(mlp=P.moe(4, 2, 64, 0, 0), kv_from=0, **ATT), P.attention(mlp=P.moe(9, 3, 64, 3, 2), **ATT),
                    P.attention(mlp=None, **ATT), P.attention(mlp=P.dense(64), **ATT)], width=width, vocab=50)
    check(cfg, P.random_checkpoint(cfg, seed=width), rows + 10, [rows, 8])


# The other designs' epilogues (residual sums with and without a scale, tanh, gelu, squared relu, loops) in products of 300, 33 and few rows
@pytest.mark.parametrize("name", ["sirodra", "fusanex", "dipivik", "sizitar", "gaparax"])
def test_other_designs(name):
    if name == "sirodra":
        cfg = U.config([U.hgrn2(heads=4, dim=32, vdim=64, ff=1088), U.attention(heads=4, kv_heads=2, dim=64, vdim=64, window=50, pool=8, ff=512), U.mlstm(heads=4, dim=32, vdim=64)],
                       width=512, vocab=700, loop=(0, 2, 2))
        S = U.random_checkpoint(cfg, seed=1)
    elif name == "fusanex":
        m = FU.moe(experts=6, identity=1, top=2, ff=128, shared=(576, 0.8))
        cfg = FU.config([FU.parallel(heads=4, kv_heads=2, dim=64, vdim=64, rheads=4, rdim=64, mlp=m), FU.rglru(width=512, blocks=4, mlp=m)], width=512, vocab=700)
        S = FU.random_checkpoint(cfg, seed=2, lora=64)
    elif name == "dipivik":
        cfg = DU.config([DU.retention(heads=4, dim=64, vdim=64, rot=32, mlp=DU.dense(1088)), DU.latent(heads=4, dim=64, rot_dim=32, vdim=64, q_rank=128, kv_rank=128, window=60,
                                                                                                       mlp=DU.moe(experts=6, top=2, ff=128, shared=576))], width=512, vocab=700)
        S = DU.random_checkpoint(cfg, seed=3)
    elif name == "sizitar":
        cfg = ZU.config([ZU.channel_delta(heads=4, kv_heads=2, dim=64, vdim=64, decay_rank=64, gate_rank=64, mlp=ZU.dense(1088)),
                         ZU.attention(heads=4, kv_heads=2, dim=64, vdim=64, rot=32, mlp=ZU.moe(experts=6, top=2, ff=128, shared=576))], width=512, vocab=700, loop=(0, 2, 2))
        S = ZU.random_checkpoint(cfg, seed=4)
    else:
        cfg = GU.config([GU.latent(heads=4, dim=64, rot_dim=32, vdim=64, kv_rank=128, mlp=GU.dense(1088)), GU.attention(heads=4, kv_heads=2, dim=64, vdim=64, size=64, bias_max=40, rows=16,
                                                                                                                         mlp=GU.moe(experts=8, top=2, ff=128, count=4, keep=2))],
                        width=512, vocab=700)
        S = GU.random_checkpoint(cfg, seed=5)
    check(cfg, S, 350, [300, 33, 8, 2], page=64)
