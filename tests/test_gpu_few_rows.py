"""Linears of one and two rows by a wave per column (k_gemv) and by waves that walk the columns (k_gemv_walk), bit-exact against the oracle: fewer columns than waves, one, two, three
and more steps, a last step that only some waves have, every depth, gate and up together (K up to 2048) and one after the other."""
import numpy as np
import pytest
import torch

from oracle import voxref as vr

from .test_gpu_ops import Bits, T, dev, rnd  # noqa: F401  (dev: fixture)
from .test_gpu_prompt_rows import forward, stack

pytestmark = pytest.mark.gpu


def walks(B, N_, K, norm, glu):
    from vox_serve_amd import _native as N
    return N.lib().vox_linear_form(torch.cuda.get_device_properties(0).multi_processor_count, B, N_, K, norm, glu, 0)


@pytest.mark.parametrize("B", [1, 2])
@pytest.mark.parametrize("N_,K,walk", [(3, 1024, ()), (2048, 1024, (1, 2)), (2049, 2048, (2,)), (4100, 3072, (2,)), (6145, 4096, ()), (8190, 4096, (2,)), (10247, 1024, ()), (4096, 2048, (1, 2)),
                                       (2048, 3072, (1, 2)), (4096, 4096, (1, 2)), (10247, 2048, (2,))])
def test_linear_of_one_and_two_rows(dev, B, N_, K, walk):  # noqa: F811
    from vox_serve_amd import _native as N
    assert walks(B, N_, K, 0, 0) == (B in walk)
    rng = np.random.default_rng(B + N_ + K)
    W, bias, x, res = rnd(rng, N_, K, s=0.05), rnd(rng, N_), rnd(rng, B, K), rnd(rng, B, N_)
    Wt, bt, xt, rt = T(W, dev), T(bias, dev), T(x, dev), T(res, dev)
    for use_bias, use_res, act in ((False, False, 0), (True, True, 0), (True, False, 1)):
        y = torch.empty(B, N_, dtype=torch.bfloat16, device=dev)
        N.check(N.lib().vox_linear(N.ctx(), N.stream(), N.ptr(Wt), N.ptr(bt) if use_bias else None, N.ptr(xt), N.ptr(rt) if use_res else None, N.ptr(y), B, N_, K, act))
        ref = vr.linear(W, x, bias if use_bias else None, None, act=act)
        assert np.array_equal(Bits(y), vr.add(res, ref) if use_res else ref), (use_bias, use_res, act)


@pytest.mark.parametrize("B", [1, 2])
@pytest.mark.parametrize("N_,K,walk", [(5, 1024, ()), (2056, 1024, (2,)), (6147, 2048, (2,)), (2049, 3072, (1, 2)), (2048, 4096, (2,)), (6149, 4096, (2,)), (6147, 3072, (1, 2))])
def test_silu_mul_of_one_and_two_rows(dev, B, N_, K, walk):  # noqa: F811
    from vox_serve_amd import _native as N
    assert walks(B, N_, K, 0, 1) == (B in walk)
    rng = np.random.default_rng(B + N_ + K)
    Wg, Wu, x = rnd(rng, N_, K, s=0.05), rnd(rng, N_, K, s=0.05), rnd(rng, B, K)
    g, u, xt, h = T(Wg, dev), T(Wu, dev), T(x, dev), torch.empty(B, N_, dtype=torch.bfloat16, device=dev)
    N.check(N.lib().vox_linear_silu_mul(N.ctx(), N.stream(), N.ptr(g), N.ptr(u), N.ptr(xt), N.ptr(h), B, N_, K))
    assert np.array_equal(Bits(h), vr.linear_silu_mul(Wg, Wu, x))


@pytest.mark.parametrize("H,F,bias,walk", [(1024, 2112, True, 1), (2048, 6208, False, 1), (3072, 2112, True, 1), (4096, 4160, False, 1), (1024, 9024, False, 2), (2048, 1984, True, 0)])
def test_normed_linears_of_one_and_two_rows(dev, H, F, bias, walk):  # noqa: F811
    """The norm in front: a stack's q | k | v and gate and up rows, one and two rows at a time, against all four together, which the same context gives to k_gemv in pairs.  Ragged last
    steps; walk 2: two rows walk gate and up, one row does not; 0: fewer columns than waves (gate and up)."""
    from vox_serve_amd import _native as N
    heads, kvh, D, rows = 16, 8, 128, 4
    g = torch.Generator(device=dev).manual_seed(H + F)
    x = torch.randn(rows, H, generator=g, device=dev).bfloat16()
    assert walks(1, 4096, H, 1, 0) == walks(2, 4096, H, 1, 0) == 1
    assert (walks(1, F, H, 1, 1), walks(2, F, H, 1, 1)) == {0: (0, 0), 1: (1, 1), 2: (0, 1)}[walk]
    N.set_exact_rows(8)
    try:
        h, keep = stack(dev, H, heads, kvh, D, F, rows, 32, 32, 9, bias)
        got = []
        for parts in ([4], [1, 2, 1], [2, 1, 1]):
            kv = torch.zeros(2, 1, 2, 32, kvh, D, dtype=torch.bfloat16, device=dev)
            got.append((Bits(forward(dev, h, x, kv, 32, kvh, D, parts, [0])), Bits(kv)))
        N.lib().vox_stack_destroy(h)
    finally:
        N.set_exact_rows(2)
    assert np.isfinite(vr.bf2f(got[0][0])).all()
    for other in got[1:]:
        assert np.array_equal(got[0][0], other[0]) and np.array_equal(got[0][1], other[1])
