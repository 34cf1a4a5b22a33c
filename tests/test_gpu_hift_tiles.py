"""HiFT's convolutions over three-term rows (k_conv_dma with two weight planes per tap) at row counts on both sides of every tile rule.

A request's samples must be the same bits in any batch: all tiles add in one order, so the equality is exact.  Against the oracle the
vocoder's own bar holds (waveform RMS <= 1e-4 in fp32)."""
import pytest
import torch

from .test_gpu_hift import dev, rms, to_plugin_cfg  # noqa: F401  (dev: fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,n", [(1, 2), (3, 5), (7, 8), (33, 3), (56, 8)])
def test_hift_rows_do_not_choose_the_order(dev, T, n):  # noqa: F811
    from oracle import hift_ref as HR
    from vox_serve_amd.tokenizer.hifigan import HiFTGenerator
    cfg = HR.HiftCfg()
    W = HR.random_hift_weights(cfg, seed=6)
    voc = HiFTGenerator(W, to_plugin_cfg(cfg), device=dev, max_batch=n, max_T=T, seed=3)
    mel = 0.8 * torch.randn(n, cfg.in_channels, T, generator=torch.Generator().manual_seed(T))
    sb = torch.arange(n, dtype=torch.int32) * 2
    both, _ = voc.forward_chunk(mel, stream_base=sb)
    for i in (0, n - 1):
        one, _ = voc.forward_chunk(mel[i:i + 1], stream_base=sb[i:i + 1])
        assert torch.equal(both[i], one[0])
    if T <= 7:
        ini, nz = HR.make_noise(cfg, n, T, seed=9)
        wav, src = voc.forward_chunk(mel, noise=nz)
        ref, _ = HR.HiftRef(cfg, W).forward_chunk(mel, ini, nz)
        assert rms(ref.numpy()) > 1e-3 and rms(wav.cpu().numpy() - ref.numpy()) < 1e-4
    voc.close()
