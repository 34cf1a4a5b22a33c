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


@pytest.mark.parametrize("B,V", [(8, 12305), (9, 8192), (9, 8197), (9, 12288), (16, 12305), (16, 16400), (3, 20487), (16, 20480)])
@pytest.mark.parametrize("bias", [False, True])
def test_head_of_few_rows_walks_column_tiles(dev, B, V, bias):  # noqa: F811
    """A 4096-wide model's head (k_gemm_tiles, plain outputs): two to five rounds of a block per CU and one tile more, a last tile of a few columns, one and two rows
    a wave.  The layer's outputs are zero, so the head reads the embeddings: rmsnorm and linear on them, in launches of their own, have the same bits."""
    from vox_serve_amd import _native as N
    from vox_serve_amd.engine import LMCfg, LMEngine, StackCfg
    H, D, F = 4096, 128, 64
    rng = np.random.default_rng(B + V)
    w = lambda *s, m=0.0, sd=0.05: T(vr.f2bf(m + rng.standard_normal(s, dtype=np.float32) * np.float32(sd)), dev)
    zero = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=dev)
    layer = dict(wqkv=w(4 * D, H), wo=zero(H, 2 * D), wgate=w(F, H), wup=w(F, H), wdown=zero(H, F), ln1=w(H, m=1.0), ln2=w(H, m=1.0))
    norm, emb, head, b = w(H, m=1.0), w(B, H, sd=1.0), w(V, H), w(V, sd=1.0) if bias else None
    eng = LMEngine(LMCfg(StackCfg(H, 1, 2, 1, D, F, qk_norm=False), B, V, max_pos=64), [layer], norm, emb, head, b, max_batch=B, page_size=16, max_pages=B, max_seq_len=16,
                   max_prefill_rows=16, device=dev)
    eng.input_ids[:, 0] = torch.arange(B, dtype=torch.int32, device=dev)
    eng.upload_plan(pos=[0] * B, kvlen=[1] * B, page=range(B), slot=[0] * B, indptr=range(B + 1), indices=range(B))
    eng.frame(B, 1, eng.sampling_cfg(greedy=True), feedback=False)
    xn, want = torch.empty_like(emb), torch.empty(B, V, dtype=torch.bfloat16, device=dev)
    N.check(N.lib().vox_rmsnorm(N.ctx(), N.stream(), N.ptr(emb), N.ptr(norm), N.ptr(xn), B, H, 1e-6))
    N.check(N.lib().vox_linear(N.ctx(), N.stream(), N.ptr(head), N.ptr(b) if bias else None, N.ptr(xn), None, N.ptr(want), B, V, H, 0))
    got = eng.out_logits[:B]
    assert want.float().std() > 0 and np.array_equal(Bits(got), Bits(want)), (got != want).nonzero()[:4].tolist()
