"""Linears of 33..128 rows with K >= 2048 (k_gemm_rows, k_norm_rows): bit-exact against the oracle in the order it routes them to, at the
row counts where a tile, a row half or the last 16 rows end, with one and two column tiles per block, row-major and fragment-major
operands (the bare linears and the decoder stack's hand-offs)."""
import numpy as np
import pytest
import torch

from oracle import voxref as vr
from oracle.policy import EPI_STORE, Call, route

from .oracle_tape import Tape
from .test_gpu_ops import Bits, T, dev, rnd, stack_rows_case  # noqa: F401  (dev: fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,N_,K", [(33, 128, 2048), (48, 256, 2048), (49, 128, 3072), (64, 4096, 2048), (65, 128, 6144), (80, 128, 2048),
                                    (81, 4096, 2048), (97, 128, 4096), (128, 384, 2048), (35, 4224, 2048), (64, 6144, 2048), (79, 5120, 3072), (50, 8192, 2048)])
def test_linear_rows_bit_exact(dev, B, N_, K):  # noqa: F811
    from vox_serve_amd import _native as N
    rng = np.random.default_rng(B + N_ + K)
    W, bias, x, res = rnd(rng, N_, K, s=0.05), rnd(rng, N_), rnd(rng, B, K), rnd(rng, B, N_)
    Wt, bt, xt, rt = T(W, dev), T(bias, dev), T(x, dev), T(res, dev)
    order = route(Call(B=B, N=N_, K=K, epi=EPI_STORE))[0]
    for use_bias, use_res in ((False, False), (True, True)):
        y = torch.empty(B, N_, dtype=torch.bfloat16, device=dev)
        N.check(N.lib().vox_linear(N.ctx(), N.stream(), N.ptr(Wt), N.ptr(bt) if use_bias else None, N.ptr(xt), N.ptr(rt) if use_res else None,
                                   N.ptr(y), B, N_, K, 0))
        ref = vr.linear(W, x, bias if use_bias else None, None, order=order, act=0)
        assert np.array_equal(Bits(y), vr.add(res, ref) if use_res else ref), (use_bias, use_res)


@pytest.mark.parametrize("n_rows,dims", [(33, (2048, 16, 8, 512)), (81, (2048, 2, 1, 384)), (100, (2048, 2, 1, 256)), (40, (4096, 2, 1, 256)),
                                         (75, (4096, 2, 1, 384))])
def test_stack_rows_with_norms(dev, n_rows, dims):  # noqa: F811
    stack_rows_case(Tape(), dev, n_rows, dims=dims)


@pytest.mark.parametrize("n_rows,dims", [(3, (4096, 2, 1, 8224)), (8, (4096, 32, 2, 4128)), (9, (4096, 32, 2, 4128)), (16, (4096, 2, 1, 4160))])
def test_stack_few_rows_more_column_tiles_than_cus(dev, n_rows, dims):  # noqa: F811
    """Up to 16 rows of 4096 values whose norm runs inside k_gemm_tiles: one and two rows a wave, 257 .. 514 column tiles (the last round of blocks nearly
    empty), and the down projection behind them on k_linear_mfma_stream with its input fragment-major, waves with a k-step more than others among them."""
    stack_rows_case(Tape(), dev, n_rows, dims=dims)
