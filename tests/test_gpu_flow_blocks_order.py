"""GPU: the flow estimator's fused transformer blocks against the launches that blocks of other sizes take, on the same weights: the same bits.

A zero bias on q | k | v, which the fused blocks do not take, sends a block to the general launches and changes no sum."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import flow_ref as FR
from tests.test_gpu_flow import flow_plugin_cfg, rms

pytestmark = pytest.mark.gpu


class _GeneralBlocks:
    """The native library with a create call that gives every transformer block's q | k | v a zero bias."""

    def __init__(self, lib, zeros):
        self._lib, self._zeros = lib, zeros

    def __getattr__(self, name):
        f = getattr(self._lib, name)
        if name != "vox_flow_create":
            return f

        def create(ctx, cfg, fw, *rest):
            c, w = cfg._obj, fw._obj
            for i in range((2 + c.est_mid) * c.est_blocks):
                w.tblocks[i].qkv.bias = self._zeros.data_ptr()
            return f(ctx, cfg, fw, *rest)
        return create


# rows of the estimator (2 guidance halves x B x 2 T): below a tile, whole tiles, remainders, many tiles; blocks that are first, between and last
@pytest.mark.parametrize("B,T,blocks", [(1, 1, 1), (1, 7, 2), (3, 9, 3), (2, 28, 2), (8, 28, 4)])
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
        mp.setattr(CF.N, "lib", lambda: _GeneralBlocks(lib, zeros))
        prompt_general, general = mels()
    assert rms(got) > 0.5 and np.array_equal(prompt, prompt_general) and np.array_equal(got, general)
