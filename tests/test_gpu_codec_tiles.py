"""The LDS-DMA convolutions of the Qwen3 codec and of Mimi (k_conv_dma, k_conv_unit) at the shapes where their tiles can go wrong, against the CPU oracle in fp32.

Channel counts that are multiples of 32, 64, 128 and 256 only (the k-steps of the tiles), fewer rows than one tile and rows that do not
fill the last one, intermediate sizes that end inside a gate / up pair, chunks shorter than a conv's look-back (the history shifts in
place) and a batch whose requests end inside a tile.

Tolerance: the waveform bar of the decoder, RMS <= 1e-4 against fp32 (two bf16 terms keep 16 significand bits of every operand: relative
2^-17 per product, and the sums are fp32).  In the bf16 operand mode one term keeps 8 bits, 2^-9 per operand, through some 30 convs in
sequence: sqrt(30) * 2^-9 of the signal, times four = 4.3e-2 (a waveform of the mode is off by 1.4e-2 to 2.3e-2; 32 channels of one tap lost
anywhere move it by 8e-2 to 1.8e-1 at the median of all weights)."""
import numpy as np
import pytest
import torch

from oracle import qwen3_codec_ref as CR
from .test_gpu_codec import dev, oracle_exact, rms  # noqa: F401  (dev: fixture)

pytestmark = pytest.mark.gpu


def cfg_of(codebook_dim, latent, hidden, inter, heads, head_dim, decoder, rates):
    return CR.CodecCfg(codebook_size=64, codebook_dim=codebook_dim, latent_dim=latent, decoder_dim=decoder, hidden_size=hidden,
                       intermediate_size=inter, head_dim=head_dim, num_heads=heads, num_layers=2, num_quantizers=3, sliding_window=12,
                       upsample_rates=rates, upsampling_ratios=[2, 2])


CASES = [
    # codebook, latent, hidden, intermediate, heads, head_dim, decoder, rates, requests, frames per chunk
    ((64, 96, 96, 96, 2, 16, 512, [2, 2, 2, 2]), 1, 1),        # 32-channel steps, one row, look-back longer than the chunk
    ((64, 96, 32, 160, 2, 16, 1536, [3, 2, 2, 2]), 3, 2),      # 1536 -> 768 ... 96 channels, gate / up pairs ending inside a column tile
    ((128, 64, 64, 96, 4, 16, 512, [4, 2, 2, 2]), 5, 3),       # 64-channel steps, 15 rows of a 16-row tile
    ((256, 128, 128, 128, 2, 64, 512, [2, 3, 2, 2]), 17, 1),   # 128-channel steps, 17 rows: one into a second tile; head dim 64
    ((512, 384, 384, 640, 6, 64, 1024, [2, 2, 2, 3]), 2, 4),   # 128-channel steps only
    ((64, 96, 96, 96, 2, 16, 1536, [2, 2, 2, 2]), 3, 1),       # whole residual units of 64 rows whose look-back (54) is nearly all history
    ((512, 256, 512, 768, 8, 64, 512, [8, 5, 4, 3]), 4, 2),    # 256-channel steps, the last block's 32 channels over many rows
    ((64, 96, 32, 160, 2, 16, 1536, [8, 5, 4, 3]), 18, 1),     # whole units of 192 channels (11 520 rows) and, in eight waves, of 96 (34 560)
]
BF16_BAR = 4 * 30 ** 0.5 * 2 ** -9      # of the signal


@pytest.mark.parametrize("shape,n,chunk", CASES)
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
def test_conv_tiles_against_fp32(dev, shape, n, chunk, precision):  # noqa: F811
    from vox_serve_amd.tokenizer.qwen3_codec import Qwen3CodecConfig, Qwen3TTSDecoder
    cfg = cfg_of(*shape)
    W = CR.random_codec_weights(cfg, seed=7)
    g = torch.Generator().manual_seed(5)
    codes = torch.randint(0, cfg.codebook_size, (n, cfg.num_quantizers, 3 * chunk), generator=g)
    ref = oracle_exact(cfg, W, codes, chunk)
    pc = Qwen3CodecConfig(**{k: getattr(cfg, k) for k in Qwen3CodecConfig.__dataclass_fields__})
    dec = Qwen3TTSDecoder(W, pc, device=dev, max_batch=n, max_slots=n, detokenize_interval=chunk, operand_precision=precision)
    cache = dec.init_cache(n)
    got = torch.cat([dec.decode_chunk(codes[:, :, t:t + chunk], cache)[0].cpu().clone() for t in range(0, 3 * chunk, chunk)], -1).numpy()
    assert got.shape == ref.shape and rms(ref) > 1e-3
    assert rms(got - ref) < (1e-4 if precision == "fp32" else BF16_BAR * rms(ref)), (rms(got - ref), rms(ref))
    dec.close()


@pytest.mark.parametrize("shape,n,chunk", [c for c in CASES if c[1] > 1])
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
def test_a_request_does_not_depend_on_its_batch(dev, shape, n, chunk, precision):  # noqa: F811
    """Rows choose tiles, tiles do not choose the order of an output's sum: the same bits alone and in a batch, as in the decoders' other modes."""
    from vox_serve_amd.tokenizer.qwen3_codec import Qwen3CodecConfig, Qwen3TTSDecoder
    cfg = cfg_of(*shape)
    pc = Qwen3CodecConfig(**{k: getattr(cfg, k) for k in Qwen3CodecConfig.__dataclass_fields__})
    dec = Qwen3TTSDecoder(CR.random_codec_weights(cfg, seed=7), pc, device=dev, max_batch=n, max_slots=2 * n, detokenize_interval=chunk, operand_precision=precision)
    codes = torch.randint(0, cfg.codebook_size, (n, cfg.num_quantizers, 2 * chunk), generator=torch.Generator().manual_seed(5))

    def run(rows):
        cache = dec.init_cache(len(rows))
        out = torch.cat([dec.decode_chunk(codes[rows][:, :, t:t + chunk], cache)[0].cpu().clone() for t in (0, chunk)], -1)
        dec.release_cache(cache)
        return out
    both = run(list(range(n)))
    for i in (0, n - 1):
        assert torch.equal(run([i])[0], both[i])
    dec.close()


@pytest.mark.parametrize("n,T", [(18, 2), (5, 3), (2, 1)])
def test_mimi_does_not_depend_on_its_batch(dev, n, T):  # noqa: F811
    """Mimi at its real widths: whole units of 128 and of 64 rows, and (odd frame counts) the two launches in their place; the same bits alone
    and in a batch."""
    from oracle import mimi_ref as MR
    from vox_serve_amd.tokenizer.mimi import MimiConfig, MimiDecoder
    cfg = MR.MimiCfg()
    W = MR.random_mimi_weights(cfg, seed=2)
    pc = MimiConfig(**{k: getattr(cfg, k) for k in MimiConfig.__dataclass_fields__ if hasattr(cfg, k)})
    dec = MimiDecoder(W, pc, device=dev, max_batch=n, max_frames=T)
    codes = torch.randint(0, cfg.bins, (n, cfg.n_q, T), generator=torch.Generator().manual_seed(n))
    both = dec.decode(codes).cpu().clone()
    assert rms(both.numpy()) > 1e-4
    for i in (0, n - 1):
        assert torch.equal(dec.decode(codes[i:i + 1]).cpu()[0], both[i])
    if n == 2:
        ref = MR.MimiRef(cfg, W).decode(codes).numpy()
        assert rms(both.numpy() - ref) < 1e-5 * max(1.0, rms(ref))
    dec.close()


@pytest.mark.parametrize("n", [1, 8, 9, 32, 33, 320, 321])
def test_mimi_norm_and_linear_in_one_launch(dev, n):  # noqa: F811
    """Two transformer rows a request and frame: two rows, a whole tile of 16, two into the next, 64 (the last of the two-wave form), 66 (the
    eight-wave form, two rows in its last tile), 640 (the last of it), 642 (two launches).  The last request alone takes the two-wave form, bit for bit the same; against the oracle in
    fp32 with the bar of the test above (relative 1e-5, fp32 rounding through eight layers: 2^-24 * sqrt(500 launches' roundings) = 1.3e-6)."""
    from oracle import mimi_ref as MR
    from vox_serve_amd.tokenizer.mimi import MimiConfig, MimiDecoder
    cfg = MR.MimiCfg()
    W = MR.random_mimi_weights(cfg, seed=3)
    pc = MimiConfig(**{k: getattr(cfg, k) for k in MimiConfig.__dataclass_fields__ if hasattr(cfg, k)})
    dec = MimiDecoder(W, pc, device=dev, max_batch=n, max_frames=1)
    codes = torch.randint(0, cfg.bins, (n, cfg.n_q, 1), generator=torch.Generator().manual_seed(n))
    got = dec.decode(codes).cpu().clone()
    assert torch.equal(dec.decode(codes[-1:]).cpu()[0], got[-1])
    ref = MR.MimiRef(cfg, W).decode(codes[-33:]).numpy()
    assert rms(ref) > 1e-4 and rms(got[-33:].numpy() - ref) < 1e-5 * max(1.0, rms(ref))
    dec.close()


def test_sine_behind_the_first_conv_is_exact_at_large_arguments(dev):  # noqa: F811
    """The SnakeBeta between the decoder's first conv and its first transposed conv takes libm's accuracy: with alpha = e^9 a sine that
    reduces its argument in fp32 is off by some 8000 * 2^-24 = 5e-4.  The conv's weights are zero, so what the sine reads is exact (its bias).
    Bar: two-term operands through some 30 convs in sequence, sqrt(30) * 2^-17 = 4e-5 of the signal, times four."""
    from vox_serve_amd.tokenizer.qwen3_codec import Qwen3CodecConfig, Qwen3TTSDecoder
    cfg = cfg_of(64, 96, 32, 160, 2, 16, 512, [3, 2, 2, 2])
    W = CR.random_codec_weights(cfg, seed=7)
    g = torch.Generator().manual_seed(3)
    W["decoder.0.conv.weight"].zero_()
    W["decoder.0.conv.bias"] = 2 * torch.rand(cfg.decoder_dim, generator=g) - 1
    W["decoder.1.block.0.alpha"].fill_(9.0)
    codes = torch.randint(0, cfg.codebook_size, (2, cfg.num_quantizers, 4), generator=g)
    ref = oracle_exact(cfg, W, codes, 2)
    pc = Qwen3CodecConfig(**{k: getattr(cfg, k) for k in Qwen3CodecConfig.__dataclass_fields__})
    dec = Qwen3TTSDecoder(W, pc, device=dev, max_batch=2, max_slots=2, detokenize_interval=2)
    cache = dec.init_cache(2)
    got = torch.cat([dec.decode_chunk(codes[:, :, t:t + 2], cache)[0].cpu().clone() for t in (0, 2)], -1).numpy()
    off, size = rms(got - ref), rms(ref)
    assert size > 1e-2 and off < 1.6e-4 * size
    dec.close()
