"""Prompts of more than 128 tokens: their linears (k_gemm_slabs, k_post_norm_rows) against the launches that serve fewer rows, bit for bit."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import voxref as vr

from .test_gpu_ops import Bits, T, dev  # noqa: F401  (dev: fixture)

pytestmark = pytest.mark.gpu


def stack(dev, H, heads, kvh, D, F, rows, tokens, page, seed, bias):  # noqa: F811
    from vox_serve_amd import _native as N
    from vox_serve_amd.engine import StackCfg, _stack_config, rope_table
    rng = np.random.default_rng(seed)
    w = lambda *s: T(vr.f2bf(rng.standard_normal(s, dtype=np.float32) * np.float32(0.05)), dev)
    g = lambda n: T(vr.f2bf(1 + 0.1 * rng.standard_normal(n).astype(np.float32)), dev)
    c = StackCfg(H, 2, heads, kvh, D, F, 1e-6, 1e6, 1.0, None, False, None, False, bias)
    arr, keep = (N.LayerWeights * 2)(), []
    for l in range(2):
        ts = dict(wqkv=w((heads + 2 * kvh) * D, H), wo=w(H, heads * D), wgate=w(F, H), wup=w(F, H), wdown=w(H, F), ln1=g(H), ln2=g(H))
        if bias:
            ts["bqkv"] = w((heads + 2 * kvh) * D)
        for k, v in ts.items():
            keep.append(v)
            setattr(arr[l], k, v.data_ptr())
    fn, rope = g(H), rope_table(tokens, c, dev)
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
        rows = N.Rows(*[t.data_ptr() for t in tens], n, at + n, None, 0, 0, -1, 0)
        xi, y = x[at: at + n].clone(), torch.empty(n, x.shape[1], dtype=torch.bfloat16, device=dev)
        N.check(N.lib().vox_stack_forward(h, N.stream(), xi.data_ptr(), y.data_ptr(), kv.data_ptr(), kv[0].numel(), ctypes.byref(rows)))
        torch.cuda.synchronize()
        out.append(y)
        at += n
    return torch.cat(out)


# K = 320: one 256-column sum and a quarter; 1088: four and a quarter; 704: two and three quarters.  Rows behind a tile of 64, 128 and 256, one row in the last tile.  The
# wide ones reach the tiles of 128 and 256 rows.
@pytest.mark.parametrize("rows,H,heads,kvh,D,F,bias", [(129, 320, 4, 2, 64, 704, True), (193, 320, 4, 2, 64, 704, False), (257, 1088, 4, 4, 128, 448, True), (300, 320, 2, 1, 64, 6208, False),
                                                       (520, 320, 3, 1, 128, 12352, False), (1000, 1088, 2, 2, 64, 2112, True)])
def test_prompt_in_one_portion_and_in_many(dev, rows, H, heads, kvh, D, F, bias):  # noqa: F811
    """Portions of at most 100 rows take k_gemm_splitk (no width here is one of k_gemm_fullk's)."""
    from vox_serve_amd import _native as N
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
