"""Prompts: their linears (k_gemm_slabs, k_post_norm_rows) and attention (k_attn_prompt, k_attn_decode) against the launches that serve fewer rows, bit for bit."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import voxref as vr

from .test_gpu_ops import Bits, T, dev  # noqa: F401  (dev: fixture)

pytestmark = pytest.mark.gpu


def stack(dev, H, heads, kvh, D, F, rows, tokens, page, seed, bias, norm=False, skew=0):  # noqa: F811
    from vox_serve_amd import _native as N
    from vox_serve_amd.engine import StackCfg, _stack_config, rope_table
    rng = np.random.default_rng(seed)
    w = lambda *s: T(vr.f2bf(rng.standard_normal(s, dtype=np.float32) * np.float32(0.05)), dev)
    g = lambda n: T(vr.f2bf(1 + 0.1 * rng.standard_normal(n).astype(np.float32)), dev)
    c = StackCfg(H, 2, heads, kvh, D, F, 1e-6, 1e6, 1.0, None, norm, None, False, bias)
    arr, keep = (N.LayerWeights * 2)(), []
    for l in range(2):
        ts = dict(wqkv=w((heads + 2 * kvh) * D, H), wo=w(H, heads * D), wgate=w(F, H), wup=w(F, H), wdown=w(H, F), ln1=g(H), ln2=g(H))
        if bias:
            ts["bqkv"] = w((heads + 2 * kvh) * D)
        if norm:
            ts.update(qnorm=g(D), knorm=g(D))
        for k, v in ts.items():
            keep.append(v)
            setattr(arr[l], k, v.data_ptr())
    fn, rope = g(H), rope_table(tokens, c, dev)
    if skew:      # the table `skew` floats off a 16-byte boundary
        rope = torch.cat([rope.new_zeros(skew), rope.reshape(-1)])[skew:]
    sc, h = _stack_config(c, page, rows, tokens), ctypes.c_void_p()
    N.check(N.lib().vox_stack_create(N.ctx(), ctypes.byref(sc), arr, fn.data_ptr(), rope.data_ptr(), tokens, ctypes.byref(h)))
    return h, keep + [fn, rope]


def forward(dev, h, x, kv, page, kvh, D, parts, pages):  # noqa: F811
    """The prompt x in portions: their hidden rows, and what they leave in kv."""
    from vox_serve_amd import _native as N
    out, at = [], 0
    i32 = lambda v: torch.as_tensor(np.asarray(v), dtype=torch.int32).to(dev)
    for n in parts:
        pos = np.arange(at, at + n)
        tens = [i32(pos), i32(np.zeros(n)), i32(pos + 1), i32(np.asarray(pages)[pos // page]), i32(pos % page), i32([0, len(pages)]), i32(pages)]
        rows = N.Rows(*[t.data_ptr() for t in tens], n, at + n, None, 0, 0, -1, 0, 1)
        xi, y = x[at: at + n].clone(), torch.empty(n, x.shape[1], dtype=torch.bfloat16, device=dev)
        N.check(N.lib().vox_stack_forward(h, N.stream(), xi.data_ptr(), y.data_ptr(), kv.data_ptr(), kv[0].numel(), ctypes.byref(rows)))
        torch.cuda.synchronize()
        out.append(y)
        at += n
    return torch.cat(out)


# K = 320: one 256-column sum and a quarter; 1088: four and a quarter; 704: two and three quarters.  Rows behind a tile of 64, 128 and 256, one row in the last tile.  The
# tiles: those of q | k | v (a norm in front, bias), o (residual, the next norm behind), gate and up, down.
@pytest.mark.parametrize("rows,H,heads,kvh,D,F,bias,tiles", [(129, 320, 4, 2, 64, 704, True, (0, 0, 0, 0)), (193, 320, 4, 2, 64, 704, False, (0, 0, 0, 0)), (257, 1088, 4, 4, 128, 448, True, (0, 0, 0, 0)),
                                                             (300, 320, 2, 1, 64, 6208, False, (0, 0, 4, 0)), (520, 320, 3, 1, 128, 12352, False, (0, 0, 3, 0)),
                                                             (1000, 1088, 2, 2, 64, 2112, True, (0, 2, 4, 2)), (233, 320, 33, 11, 64, 1088, True, (1, 0, 1, 0)),
                                                             (233, 320, 33, 33, 64, 2112, True, (2, 0, 2, 0)), (233, 320, 33, 33, 128, 4160, True, (3, 0, 3, 0)),
                                                             (450, 320, 33, 33, 128, 6208, True, (4, 0, 4, 0)), (450, 1088, 4, 2, 64, 448, False, (0, 1, 0, 1)),
                                                             (1000, 2112, 4, 2, 64, 448, False, (0, 3, 1, 3))])
def test_prompt_in_one_portion_and_in_many(dev, rows, H, heads, kvh, D, F, bias, tiles):  # noqa: F811
    """Portions of at most 100 rows take k_gemm_splitk (no width here is one of k_gemm_fullk's)."""
    from vox_serve_amd import _native as N
    form = N.lib().vox_linear_form
    assert tuple(form(256, rows, n, k, norm, glu, 1) - 16 for n, k, norm, glu in (((heads + 2 * kvh) * D, H, 1, 0), (H, heads * D, 0, 0), (F, H, 1, 1), (H, F, 0, 0))) == tiles
    page, n = 32, -(-rows // 32)
    rng = np.random.default_rng(rows)
    h, keep = stack(dev, H, heads, kvh, D, F, rows, n * page, page, rows, bias)
    x = T(vr.f2bf(rng.standard_normal((rows, H), dtype=np.float32)), dev)
    pages = list(rng.permutation(n + 2)[:n])
    got = []
    for parts in ([rows], [100] * (rows // 100) + ([rows % 100] if rows % 100 else [])):
        kv = torch.zeros(2, n + 2, 2, page, kvh, D, dtype=torch.bfloat16, device=dev)
        got.append((forward(dev, h, x, kv, page, kvh, D, parts, pages), kv))
    N.lib().vox_stack_destroy(h)
    assert np.array_equal(Bits(got[0][0]), Bits(got[1][0])) and np.array_equal(Bits(got[0][1]), Bits(got[1][1]))
    assert torch.isfinite(got[0][0].float()).all()


def attend(dev, q, kv, q_req, kvlen, indptr, indices, Hkv, page, top, one_by_one, form):  # noqa: F811
    """vox_paged_attention_of on all rows at once, which the launch `form` serves, or on one row at a time (k_attn_partial and k_attn_merge: 300 tokens are more than any group's single
    row leaves to the others)."""
    from vox_serve_amd import _native as N
    i32 = lambda v: torch.as_tensor(np.asarray(v), dtype=torch.int32).to(dev)
    n, Hq, D = q.shape
    top, n_req = (max(top, 300), 1) if one_by_one else (top, len(indptr) - 1)
    assert N.lib().vox_attention_form(0, 1 if one_by_one else n, n_req, Hq, Hkv, D, page, top) == (0 if one_by_one else form)
    out = torch.full_like(q, 7.0)
    ip, ix = i32(indptr), i32(indices)
    ws = torch.empty(N.lib().vox_attn_workspace_bytes(n, Hq, D, top) // 4, dtype=torch.float32, device=dev)
    for i, j in ([(0, n)] if not one_by_one else [(i, i + 1) for i in range(n)]):
        qr, kl = i32(q_req[i:j]), i32(kvlen[i:j])
        N.check(N.lib().vox_paged_attention_of(N.ctx(), N.stream(), q[i:j].data_ptr(), N.ptr(kv), N.ptr(qr), N.ptr(kl), N.ptr(ip), N.ptr(ix), out[i:j].data_ptr(), N.ptr(ws), j - i, Hq, Hkv,
                                               D, page, top, float(D ** -0.5), n_req))
    torch.cuda.synchronize()
    return out


def prompt_case(seed, lens, ctx, page):
    """Rows of requests behind one another: (q_req, kvlen, indptr, indices)."""
    rng = np.random.default_rng(seed)
    q_req, kvlen, indptr, total = [], [], [0], 0
    for r, (n, c) in enumerate(zip(lens, ctx)):
        q_req += [r] * n
        kvlen += list(range(c + 1, c + n + 1))
        total += -(-(c + n) // page)
        indptr.append(total)
    return q_req, kvlen, indptr, list(rng.permutation(total + 3)[:total])


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("Hq,Hkv,D,page,lens,ctx", [(16, 8, 128, 128, [200], [0]), (16, 8, 128, 32, [1, 197, 3, 2, 260, 33], [0, 300, 31, 5, 7, 64]),
                                                    (32, 8, 64, 24, [330, 240, 5, 7], [11, 0, 90, 40]), (8, 8, 64, 24, [130, 5, 140], [11, 290, 0]), (18, 6, 128, 16, [170, 90], [100, 0]),
                                                    (15, 5, 64, 8, [257], [0]), (12, 12, 64, 8, [257], [0]), (56, 8, 64, 16, [121, 90], [0, 9]), (32, 2, 128, 128, [70], [200]),
                                                    (32, 8, 64, 128, [290], [0]), (8, 8, 128, 128, [1031], [0])])
def test_prompt_attention_against_single_rows(dev, Hq, Hkv, D, page, lens, ctx, special, form=2):  # noqa: F811
    """Several requests in a tile, tiles of 16, 8, 5 (a column of the 16 idle), 4, 2 (two idle) and 1 rows, ragged chunks, pages that no power of two divides, four and eight waves; with
    infinities and NaN among keys and values (single rows never read the tokens behind them), and a row without tokens in between."""
    g = torch.Generator(device=dev).manual_seed(sum(lens))
    q_req, kvlen, indptr, indices = prompt_case(sum(lens), lens, ctx, page)
    top = max(kvlen)
    q = torch.randn(len(q_req), Hq, D, generator=g, device=dev).bfloat16()
    kv = torch.randn(max(indices) + 1, 2, page, Hkv, D, generator=g, device=dev).bfloat16()
    if special:
        kvlen[len(kvlen) // 2] = 0
        for page_id in indices[:: max(1, len(indices) // 5)]:
            kv[page_id, 1, page // 3, 0, 1] = float("inf")
            kv[page_id, 1, page // 2, Hkv - 1, D - 2] = float("nan")
            kv[page_id, 0, page - 1, 0, 3] = float("-inf")
    a, b = (attend(dev, q, kv, q_req, kvlen, indptr, indices, Hkv, page, top, one, form) for one in (False, True))
    nan = torch.isnan(a.float()) & torch.isnan(b.float())
    same = (a.view(torch.int16) == b.view(torch.int16)) | nan
    assert same.all(), (~same).nonzero()[:4].tolist()
    assert special or not nan.any()


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("Hq,Hkv,D,page,lens,ctx", [(16, 8, 128, 128, [75], [0]), (4, 2, 128, 32, [5, 33, 1, 20], [0, 30, 95, 60]), (16, 8, 128, 96, [9, 16], [191, 240]),
                                                    (32, 8, 64, 64, [20, 2], [76, 31]), (32, 8, 64, 32, [2, 12], [254, 128]), (32, 2, 128, 128, [24], [190]),
                                                    (6, 1, 128, 32, [40], [0]), (2, 1, 64, 32, [2], [31])])
def test_short_prompt_attention_against_single_rows(dev, Hq, Hkv, D, page, lens, ctx, special):  # noqa: F811
    """A wave per chunk, four and eight waves: rows of one chunk to eight that end at and around a chunk's last token, several requests; with infinities and NaN, also behind
    the last token of a row, and a row without tokens."""
    test_prompt_attention_against_single_rows(dev, Hq, Hkv, D, page, lens, ctx, special, form=1)


@pytest.mark.parametrize("rows,N,K,tile", [(33, 151, 1152, 0), (65, 130, 640, 0), (129, 2048, 128, 0), (300, 2050, 1152, 1), (450, 2050, 1152, 2), (1000, 2048, 640, 2), (520, 4100, 640, 3),
                                           (257, 6000, 384, 3)])
def test_linears_of_many_rows_against_portions(dev, rows, N, K, tile):  # noqa: F811
    """vox_linear on all rows (k_gemm_slabs with four chains, every tile) and on portions of at most 24 (k_linear_mfma): ragged rows and columns, one k-tile pair to many, with and
    without SiLU, bias and residual."""
    from vox_serve_amd import _native as NV
    assert NV.lib().vox_linear_form(256, rows, N, K, 0, 0, 0) == 16 + tile
    g = torch.Generator(device=dev).manual_seed(rows + tile)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).bfloat16()
    W, b, x, res = rnd(N, K), rnd(N), rnd(rows, K), rnd(rows, N)
    cuts = np.cumsum([0] + [len(p) for p in np.array_split(np.arange(rows), -(-rows // 24))])
    for act, bias, residual in [(0, b, res), (1, b, None), (1, None, res), (0, None, None)]:
        ys = []
        for bounds in ([0, rows], list(cuts)):
            y = torch.full((rows, N), 7.0, dtype=torch.bfloat16, device=dev)
            for i, j in zip(bounds, bounds[1:]):
                NV.check(NV.lib().vox_linear(NV.ctx(), NV.stream(), NV.ptr(W), NV.ptr(bias) if bias is not None else None, x[i:j].data_ptr(),
                                             residual[i:j].data_ptr() if residual is not None else None, y[i:j].data_ptr(), j - i, N, K, act))
            torch.cuda.synchronize()
            ys.append(Bits(y))
        assert np.array_equal(*ys), (act, bias is not None, residual is not None)


@pytest.mark.parametrize("heads,kvh,D,norm,bias,rows", [(16, 8, 128, True, False, 40), (3, 1, 128, False, True, 361), (14, 2, 64, False, True, 101), (32, 8, 64, True, False, 40),
                                                        (32, 8, 64, False, False, 38)])
def test_heads_of_a_row_together(dev, heads, kvh, D, norm, bias, rows):  # noqa: F811
    """k_head_rows against k_head_prepare, which takes RoPE tables that lie on no 16 bytes: hidden rows and cache bit for bit; heads that fill a block and that do not."""
    from vox_serve_amd import _native as N
    H, page = 256, 32
    pages = list(np.random.default_rng(rows).permutation(-(-rows // page) + 1)[: -(-rows // page)])
    assert N.lib().vox_heads_form(rows, heads + 2 * kvh, D, norm) == 1 and (norm or N.lib().vox_heads_form(20, heads + 2 * kvh, D, 0) == 0)
    x = T(vr.f2bf(np.random.default_rng(3).standard_normal((rows, H), dtype=np.float32)), dev)
    got = []
    for skew in (0, 2):
        h, keep = stack(dev, H, heads, kvh, D, 512, rows, page * len(pages), page, 9, bias, norm, skew)
        kv = torch.zeros(2, len(pages) + 1, 2, page, kvh, D, dtype=torch.bfloat16, device=dev)
        got.append((Bits(forward(dev, h, x, kv, page, kvh, D, [rows], pages)), Bits(kv)))
        N.lib().vox_stack_destroy(h)
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
    assert np.abs(vr.bf2f(got[0][1])).max() > 0.01
