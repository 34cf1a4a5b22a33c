"""Decode attention over more than 256 tokens by a wave per chunk (k_attn_decode) against k_attn_partial and k_attn_merge, which take pages that are no multiple of 32 tokens: the
same tokens in pages of both kinds, bit for bit.  Rows of one chunk to many, chunks that end at every kind of place, one and two heads a block, NaN in every slot that holds no token."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import voxref as vr

from .test_gpu_ops import Bits, T, dev  # noqa: F401  (dev: fixture)
from .test_gpu_prompt_rows import stack

pytestmark = pytest.mark.gpu

LENS = [700, 1, 31, 32, 33, 257, 288, 289, 300, 511, 512, 513, 64, 95, 543, 544]


@pytest.mark.parametrize("heads,kvh,D,rows,top,page", [(16, 8, 128, 16, 700, 32), (16, 8, 128, 17, 700, 96), (4, 2, 128, 40, 513, 128), (32, 8, 64, 8, 700, 64), (32, 8, 64, 9, 513, 32),
                                                       (32, 2, 128, 3, 700, 128), (32, 2, 128, 9, 1000, 32),
                                                       (16, 8, 128, 12, 1900, 128), (16, 8, 128, 24, 1900, 128), (16, 8, 128, 14, 2304, 96), (16, 8, 128, 24, 2304, 32), (16, 8, 128, 24, 4096, 128),
                                                       (32, 8, 64, 8, 1300, 32), (32, 8, 64, 24, 4096, 128), (16, 8, 128, 17, 512, 32), (32, 8, 64, 16, 480, 96)])
def test_long_contexts_against_pages_of_sixteen(dev, heads, kvh, D, rows, top, page):  # noqa: F811
    """(16 rows and more of up to 512 tokens in pages of 16: k_attn_decode8 with two chunks a group.)"""
    from vox_serve_amd import _native as N
    assert [N.lib().vox_attention_form(1, rows, rows, heads, kvh, D, size, top) for size in (16, page)] == [3 if rows >= 16 and top <= 512 else 0, 1]
    H, F = 256, 512
    lens = [top] + [min(LENS[i % len(LENS)], top) for i in range(1, rows)]
    rng = np.random.default_rng(rows)
    g = torch.Generator(device=dev).manual_seed(rows)
    x0 = T(vr.f2bf(rng.standard_normal((rows, H), dtype=np.float32)), dev)
    past = [torch.randn(2, 2, n, kvh, D, generator=g, device=dev).bfloat16() for n in lens]      # [layer][K | V][token]
    i32 = lambda v: torch.as_tensor(np.asarray(v), dtype=torch.int32).to(dev)
    got = []
    for size in (16, page):
        per = -(-top // size)
        perm = rng.permutation(rows * per)
        table = perm.reshape(rows, per)
        h, keep = stack(dev, H, heads, kvh, D, F, rows, top + 8, size, 5, False)
        kv = torch.full((2, rows * per, 2, size, kvh, D), float("nan"), dtype=torch.bfloat16, device=dev)
        for r, n in enumerate(lens):
            tok = torch.arange(n - 1)
            kv[:, torch.as_tensor(table[r])[tok // size], :, tok % size] = past[r][:, :, : n - 1].permute(2, 0, 1, 3, 4)
        last = [n - 1 for n in lens]
        tens = [i32(last), i32(range(rows)), i32(lens), i32([table[r][n // size] for r, n in enumerate(last)]), i32([n % size for n in last]),
                i32(np.arange(rows + 1) * per), i32(table.reshape(-1))]
        ptab = i32(table)
        rs = N.Rows(*[t.data_ptr() for t in tens], rows, top, ptab.data_ptr(), per, 0, -1, 0)
        x, y = x0.clone(), torch.empty(rows, H, dtype=torch.bfloat16, device=dev)
        N.check(N.lib().vox_stack_forward(h, N.stream(), x.data_ptr(), y.data_ptr(), kv.data_ptr(), kv[0].numel(), ctypes.byref(rs)))
        torch.cuda.synchronize()
        N.lib().vox_stack_destroy(h)
        new = torch.stack([kv[:, int(table[r][n // size]), :, n % size] for r, n in enumerate(last)])
        assert torch.isfinite(y.float()).all() and torch.isfinite(new.float()).all()
        got.append((Bits(y), Bits(new), int(torch.isnan(kv.float()).sum()) + sum(lens) * 4 * kvh * D == kv.numel()))
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    assert got[0][2]


def decode(dev, h, x0, kv, lens, pos, page, slot, table, top):  # noqa: F811
    """Decode rows with a page table: their hidden rows; kv holds their new tokens."""
    from vox_serve_amd import _native as N
    rows, per = len(lens), len(table[0])
    i32 = lambda v: torch.as_tensor(np.asarray(v), dtype=torch.int32).to(dev)
    ptab = i32(table)
    tens = [i32(pos), i32(range(rows)), i32(lens), i32(page), i32(slot), i32(np.arange(rows + 1) * per), ptab.reshape(-1)]
    rs = N.Rows(*[t.data_ptr() for t in tens], rows, top, ptab.data_ptr(), per, 0, -1, 0)
    x, y = x0.clone(), torch.empty_like(x0)
    N.check(N.lib().vox_stack_forward(h, N.stream(), x.data_ptr(), y.data_ptr(), kv.data_ptr(), kv[0].numel(), ctypes.byref(rs)))
    torch.cuda.synchronize()
    return y


@pytest.mark.parametrize("heads,kvh,D,rows", [(16, 8, 128, 16), (16, 8, 128, 17), (32, 8, 64, 8), (32, 8, 64, 9)])
def test_rows_longer_than_their_call_says(dev, heads, kvh, D, rows):  # noqa: F811
    """Rows of 321 to 400 tokens in a call of up to 320: what the block keeps of a row ends with the call's ten chunks, so that such a row is one of 320 tokens (its newest is the last of
    them), and its neighbours are untouched by it."""
    from vox_serve_amd import _native as N
    H, page, per, top = 256, 32, 13, 320
    lens = [(400, 320, 321, 33, 352, 319, 385)[r % 7] for r in range(rows)]
    g = torch.Generator(device=dev).manual_seed(rows)
    x0 = torch.randn(rows, H, generator=g, device=dev).bfloat16()
    kv0 = torch.randn(2, rows * per, 2, page, kvh, D, generator=g, device=dev).bfloat16()
    table = np.random.default_rng(rows).permutation(rows * per).reshape(rows, per)
    last = [n - 1 for n in lens]
    at = dict(pos=last, page=[table[r][n // page] for r, n in enumerate(last)], slot=[n % page for n in last], table=table, top=top)
    h, keep = stack(dev, H, heads, kvh, D, 512, rows, per * page, page, 5, False)
    got = []
    for said in (lens, [min(n, top) for n in lens]):
        kv = kv0.clone()
        got.append((Bits(decode(dev, h, x0, kv, said, **at)), Bits(kv)))
    N.lib().vox_stack_destroy(h)
    assert np.isfinite(vr.bf2f(got[0][0])).all()
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])


@pytest.mark.parametrize("heads,kvh,D,rows", [(16, 8, 128, 16), (16, 8, 128, 17), (32, 8, 64, 9)])
def test_table_entries_without_cached_tokens_are_not_used(dev, heads, kvh, D, rows):  # noqa: F811
    """Padding rows (one token, page -1) and rows whose newest token opens a page that their table does not list yet: -1 in the table wherever a page holds no cached token, against
    pages of 16 tokens (k_attn_partial, which never asks for those).  The page in front of the cache belongs to the same allocation."""
    from vox_serve_amd import _native as N
    H, top = 256, 513
    lens = [(513, 1, 33, 129, 385, 1, 289, 130)[r % 8] for r in range(rows)]
    g = torch.Generator(device=dev).manual_seed(rows)
    x0 = torch.randn(rows, H, generator=g, device=dev).bfloat16()
    past = [torch.randn(2, 2, n, kvh, D, generator=g, device=dev).bfloat16() for n in lens]
    got = []
    for size in (16, 32):
        per = -(-top // size)
        table = np.random.default_rng(rows).permutation(rows * per).reshape(rows, per)
        h, keep = stack(dev, H, heads, kvh, D, 512, rows, per * size, size, 5, False)
        room = torch.zeros(1 + 2 * rows * per, 2, size, kvh, D, dtype=torch.bfloat16, device=dev)
        kv = room[1:].view(2, rows * per, 2, size, kvh, D)
        for r, n in enumerate(lens):
            tok = torch.arange(n - 1)
            kv[:, torch.as_tensor(table[r])[tok // size], :, tok % size] = past[r][:, :, : n - 1].permute(2, 0, 1, 3, 4)
        page = [-1 if n == 1 else int(table[r][(n - 1) // size]) for r, n in enumerate(lens)]
        bare = np.array([[table[r][j] if j * size < n - 1 else -1 for j in range(per)] for r, n in enumerate(lens)])
        y = decode(dev, h, x0, kv, lens, [n - 1 for n in lens], page, [(n - 1) % size for n in lens], bare, top)
        N.lib().vox_stack_destroy(h)
        got.append((Bits(y), Bits(torch.stack([kv[:, p, :, (n - 1) % size] for p, n in zip(page, lens) if n > 1])), float(room[0].abs().max())))
    assert np.isfinite(vr.bf2f(got[0][0])).all() and got[0][2] == got[1][2] == 0
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
