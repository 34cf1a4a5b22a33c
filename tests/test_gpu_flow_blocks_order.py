"""GPU: the flow estimator's fused transformer blocks against the launches that blocks of other sizes take, on the same weights: the same bits.

A zero bias on q | k | v, which the fused blocks do not take, sends a block to the general launches and changes no sum."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from oracle import flow_ref as FR
from tests.test_gpu_flow import flow_plugin_cfg, rms

pytestmark = pytest.mark.gpu


class _GeneralBlocks:
    """The native library with a create call that gives every transformer block's q | k | v a zero bias."""

    def __init__(self, lib, zeros, blocks):
        self._lib, self._zeros, self._blocks = lib, zeros, blocks

    def __getattr__(self, name):
        f = getattr(self._lib, name)
        if name not in ("vox_flow_create", "vox_glmflow_create"):
            return f

        def create(ctx, cfg, fw, *rest):
            for i in range(self._blocks):
                fw._obj.tblocks[i].qkv.bias = self._zeros.data_ptr()
            return f(ctx, cfg, fw, *rest)
        return create


# rows of the estimator (2 guidance halves x B x 2 T): below a tile, whole tiles, remainders, many tiles; 42, 41 and 20 tiles, of which the eight XCDs have
# unequal numbers of blocks; blocks that are first, between and last
@pytest.mark.parametrize("B,T,blocks", [(1, 1, 1), (1, 7, 2), (3, 9, 3), (2, 28, 2), (8, 28, 4), (6, 28, 2), (7, 23, 2), (5, 16, 1)])
def test_fused_blocks_add_as_the_general_launches(monkeypatch, B, T, blocks):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vox_serve_amd.tokenizer import cosyvoice_flow as CF
    fc = FR.FlowCfg(vocab=200, enc_layers=1, up_layers=1, est_mid=1, est_blocks=blocks)
    W, g = FR.random_flow_weights(fc, seed=T), torch.Generator().manual_seed(B)
    ptok, tok = torch.randint(0, 200, (1, 5), generator=g), torch.randint(0, 200, (B, T), generator=g)
    pfeat, spk = 0.7 * torch.randn(1, 10, fc.mel, generator=g), torch.randn(1, fc.spk_dim, generator=g)
    z0, z1 = FR.cfm_noise(1, 0, fc.mel, 16), FR.cfm_noise(1, 1, fc.mel, 2 * T)

    def mels():
        flow = CF.CosyVoice2Flow(W, flow_plugin_cfg(fc), device="cuda:0", max_batch=B, max_T=T, max_prompt_T=48, seed=1)
        try:
            return flow.set_prompt(ptok, pfeat, spk, noise=z0).cpu().numpy(), flow.forward_chunk(tok, noise=z1).cpu().numpy()
        finally:
            flow.close()

    prompt, got = mels()
    zeros = torch.zeros(3 * fc.est_heads * fc.est_head_dim, device="cuda:0")
    lib = CF.N.lib()
    with monkeypatch.context() as mp:
        mp.setattr(CF.N, "lib", lambda: _GeneralBlocks(lib, zeros, fc.n_att))
        prompt_general, general = mels()
    assert rms(got) > 0.5 and np.array_equal(prompt, prompt_general) and np.array_equal(got, general)


# GLM-4-Voice's flow: two row counts a step (all mel frames and every second), an odd number of frames among them;
# 1032 and 1376 rows: four and two column tiles a wave
@pytest.mark.parametrize("B,T,blocks", [(1, 3, 1), (3, 8, 2), (2, 25, 4), (6, 25, 2), (8, 25, 2), (8, 12, 2)])
def test_glm_blocks_add_as_the_general_launches(monkeypatch, B, T, blocks):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from oracle import glm_dec_ref as GR
    from tests.test_gpu_glm_decoder import glm_flow_plugin_cfg
    from vox_serve_amd.tokenizer import glm as GM
    fc = GR.GlmFlowCfg(vocab=113, enc_layers=1, est_mid=1, est_blocks=blocks)
    W = GR.random_glm_flow_weights(fc, seed=T)
    tok = torch.randint(0, 113, (B, T), generator=torch.Generator().manual_seed(B))
    z = GR.glm_cfm_noise(1, 0, B, fc.mel, fc.mel_len(T))

    def mels():
        flow = GM.GLMFlow(W, glm_flow_plugin_cfg(fc), device="cuda:0", max_batch=B, max_T=T, seed=1)
        try:
            return flow.inference(tok, noise=z).cpu().numpy()
        finally:
            flow.close()

    got = mels()
    zeros = torch.zeros(3 * fc.est_heads * fc.est_head_dim, device="cuda:0")
    lib = GM.N.lib()
    with monkeypatch.context() as mp:
        mp.setattr(GM.N, "lib", lambda: _GeneralBlocks(lib, zeros, (4 + fc.est_mid) * blocks))
        general = mels()
    assert rms(got) > 0.3 and np.array_equal(got, general)


def _mels(path):
    from vox_serve_amd.tokenizer import cosyvoice_flow as CF
    fc = FR.FlowCfg(vocab=200, enc_layers=1, up_layers=1, est_mid=1, est_blocks=2)
    g = torch.Generator().manual_seed(3)
    flow = CF.CosyVoice2Flow(FR.random_flow_weights(fc, seed=3), flow_plugin_cfg(fc), device="cuda:0", max_batch=2, max_T=40, max_prompt_T=48, seed=1)
    try:
        flow.set_prompt(torch.randint(0, 200, (1, 5), generator=g), 0.7 * torch.randn(1, 10, fc.mel, generator=g), torch.randn(1, fc.spk_dim, generator=g),
                        noise=FR.cfm_noise(1, 0, fc.mel, 16))
        np.save(path, flow.forward_chunk(torch.randint(0, 200, (2, 40), generator=g), noise=FR.cfm_noise(1, 1, fc.mel, 80)).cpu().numpy())
    finally:
        flow.close()


def test_attention_of_four_waves_reaches_the_fused_blocks(tmp_path):
    """VOX_FLOW_ATTN_WV=4 adds a query's keys in four parts instead of eight: other bits beyond 64 keys, the same mels.  (A process of its own: the switch is read once.)"""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    out = []
    for waves in ("8", "4"):
        path = tmp_path / f"{waves}.npy"
        subprocess.run([sys.executable, "-c", f"from tests.test_gpu_flow_blocks_order import _mels; _mels({str(path)!r})"], check=True, timeout=100,
                       cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))), env=dict(os.environ, VOX_FLOW_ATTN_WV=waves))
        out.append(np.load(path))
    assert rms(out[0]) > 0.5 and not np.array_equal(*out) and rms(out[0] - out[1]) < 1e-4
