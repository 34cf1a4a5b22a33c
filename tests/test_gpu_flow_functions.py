"""GPU: the scalar functions inside the codecs' and flows' kernels, one value at a time, against 64-bit values and against the functions of the same name in
the math library (torch's element-wise ones)."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

GELU, MISH, EXP = 0, 1, 2


def call(which, x):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vox_serve_amd import _native as N
    L = N.lib()
    L.vox_flow_function.restype, L.vox_flow_function.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int]
    x = x.to("cuda:0")
    y = torch.empty_like(x)
    N.check(L.vox_flow_function(N.stream(), which, x.data_ptr(), y.data_ptr(), x.numel()))
    return x, y


def same_bits(a, b):
    return torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(a[~a.isnan()].view(torch.int32), b[~b.isnan()].view(torch.int32))


def ulps(got, want):
    """Difference in units of the last place of a float of the size of `want` (float64; normal range)."""
    w = want.abs()
    return (got.double() - want).abs() / torch.exp2(torch.floor(torch.log2(w)) - 23)


SPECIAL = [0.0, -0.0, 1e-40, -1e-40, 1e-30, -1e-30, 3e38, -3e38, 1e5, -1e5, float("inf"), float("-inf"), float("nan")]


def test_exponential_of_the_attention():
    """Scores less their largest: 0 down to -inf.  Rounding alone is 0.5 units at worst and 0.289 in the mean square."""
    x, y = call(EXP, torch.linspace(-10, 0, 1_000_003))
    u = ulps(y, torch.exp(x.double()))
    print("exp", u.max().item(), u.square().mean().sqrt().item())
    assert u.max() < 1.0 and u.square().mean().sqrt() < 0.32      # one of the two neighbours, and nearly rounding alone
    x, y = call(EXP, torch.cat([torch.linspace(-110, 0, 1_000_003), torch.tensor([v for v in SPECIAL if not v > 0])]))
    assert same_bits(y, torch.exp(x))
    assert (y[(x < -88) & (x > -103)] > 0).all() and y[x == float("-inf")].eq(0).all()


def test_mish():
    x, y = call(MISH, torch.cat([torch.randn(4_000_000, generator=torch.Generator().manual_seed(0)), torch.linspace(-120, 120, 100_001), torch.tensor(SPECIAL)]))
    assert same_bits(y, x * torch.tanh(torch.where(x > 20, x, torch.log1p(torch.exp(x)))))
    n = slice(0, 4_000_000)
    w = x[n].double() * torch.tanh(torch.log1p(torch.exp(x[n].double())))
    e = (y[n].double() - w).norm() / w.norm()
    print("mish", e.item())
    assert e < 3.5e-8


def test_gelu():
    x, y = call(GELU, torch.cat([torch.randn(4_000_000, generator=torch.Generator().manual_seed(0)), torch.linspace(-120, 120, 100_001), torch.tensor(SPECIAL)]))
    n = slice(0, 4_000_000)
    w = x[n].double() * 0.5 * (1 + torch.erf(x[n].double() * 0.5 ** 0.5))
    e = (y[n].double() - w).norm() / w.norm()
    print("gelu", e.item())
    assert same_bits(y, 0.5 * x * (1 + torch.erf(x * 0.70710678118654752440)))
    assert e < 4e-8
