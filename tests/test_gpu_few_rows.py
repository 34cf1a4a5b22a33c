"""Linears of one and two rows whose waves walk the columns (k_gemv_walk): bit-exact against the oracle at fewer columns than waves, one, two, three and more steps, a last step
that only some waves have, every depth, gate and up together (K up to 2048) and one after the other."""
import numpy as np
import pytest
import torch

from oracle import voxref as vr

from .test_gpu_ops import Bits, T, dev, rnd  # noqa: F401  (dev: fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 2])
@pytest.mark.parametrize("N_,K", [(3, 1024), (2048, 1024), (2049, 2048), (4100, 3072), (6145, 4096), (10247, 1024)])
def test_linear_of_one_and_two_rows(dev, B, N_, K):  # noqa: F811
    from vox_serve_amd import _native as N
    rng = np.random.default_rng(B + N_ + K)
    W, bias, x, res = rnd(rng, N_, K, s=0.05), rnd(rng, N_), rnd(rng, B, K), rnd(rng, B, N_)
    Wt, bt, xt, rt = T(W, dev), T(bias, dev), T(x, dev), T(res, dev)
    for use_bias, use_res, act in ((False, False, 0), (True, True, 0), (True, False, 1)):
        y = torch.empty(B, N_, dtype=torch.bfloat16, device=dev)
        N.check(N.lib().vox_linear(N.ctx(), N.stream(), N.ptr(Wt), N.ptr(bt) if use_bias else None, N.ptr(xt), N.ptr(rt) if use_res else None, N.ptr(y), B, N_, K, act))
        ref = vr.linear(W, x, bias if use_bias else None, None, act=act)
        assert np.array_equal(Bits(y), vr.add(res, ref) if use_res else ref), (use_bias, use_res, act)


@pytest.mark.parametrize("B", [1, 2])
@pytest.mark.parametrize("N_,K", [(5, 1024), (2056, 1024), (6147, 2048), (2049, 3072), (2048, 4096), (6149, 4096)])
def test_silu_mul_of_one_and_two_rows(dev, B, N_, K):  # noqa: F811
    from vox_serve_amd import _native as N
    rng = np.random.default_rng(B + N_ + K)
    Wg, Wu, x = rnd(rng, N_, K, s=0.05), rnd(rng, N_, K, s=0.05), rnd(rng, B, K)
    g, u, xt, h = T(Wg, dev), T(Wu, dev), T(x, dev), torch.empty(B, N_, dtype=torch.bfloat16, device=dev)
    N.check(N.lib().vox_linear_silu_mul(N.ctx(), N.stream(), N.ptr(g), N.ptr(u), N.ptr(xt), N.ptr(h), B, N_, K))
    assert np.array_equal(Bits(h), vr.linear_silu_mul(Wg, Wu, x))
