"""GPU: the flow estimator's fused transformer blocks (256 channels, 8 heads of 64) at row counts around their 16-row tiles, against the fp32
restatement (oracle/flow_ref.py).  Tolerance: mel RMS error 1e-4 at a mel RMS near 1, as for the full-size flow."""
import numpy as np
import pytest
import torch

from oracle import flow_ref as FR
from tests.test_gpu_flow import flow_plugin_cfg, rms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,blocks", [(1, 1, 1), (1, 7, 2), (3, 9, 3), (2, 28, 2)])
def test_rows_around_a_tile(B, T, blocks):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vox_serve_amd.tokenizer.cosyvoice_flow import CosyVoice2Flow
    fc = FR.FlowCfg(vocab=200, enc_layers=1, up_layers=1, est_mid=1, est_blocks=blocks)
    W, g = FR.random_flow_weights(fc, seed=T), torch.Generator().manual_seed(B)
    ptok, tok = torch.randint(0, 200, (1, 5), generator=g), torch.randint(0, 200, (B, T), generator=g)
    pfeat, spk = 0.7 * torch.randn(1, 10, fc.mel, generator=g), torch.randn(1, fc.spk_dim, generator=g)
    z0, z1 = FR.cfm_noise(1, 0, fc.mel, 16), FR.cfm_noise(1, 1, fc.mel, 2 * T)
    fr = FR.FlowRef(fc, W)
    with torch.no_grad():
        pm_o, cache = fr.init_cache(ptok, pfeat, spk, z0)
        want, _ = fr.flow_chunk(tok, torch.zeros(1, 0, fc.mel), spk, z1, cache)
    flow = CosyVoice2Flow(W, flow_plugin_cfg(fc), device="cuda:0", max_batch=B, max_T=28, max_prompt_T=48, seed=1)
    try:
        pm = flow.set_prompt(ptok, pfeat, spk, noise=z0).cpu().numpy()
        got = flow.forward_chunk(tok, noise=z1).cpu().numpy()
        alone = flow.forward_chunk(tok[-1:], noise=z1).cpu().numpy()
    finally:
        flow.close()
    assert rms(want) > 0.5 and rms(pm - pm_o.numpy()) < 1e-4 and rms(got - want.numpy()) < 1e-4
    assert np.array_equal(got[-1:], alone)          # a request's mels do not depend on its batch


# more row tiles than six blocks each fit the chip: three column tiles a wave, with a remainder of 12 rows and with none
@pytest.mark.parametrize("B,T,blocks", [(7, 25, 2), (8, 28, 1)])
def test_rows_of_many_tiles(B, T, blocks):
    test_rows_around_a_tile(B, T, blocks)
