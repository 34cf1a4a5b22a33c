"""The work that a user of this framework has it do, as cases that can be timed and compared: speech-LM frames and prompts, token -> waveform
decoding, and the hybrid text LM, through the engines and decoders that the workers drive.

Weights are random-init tensors of the named architectures (`vox_serve_amd.synth`), made once per process like a checkpoint that is loaded
once; every state owns its engine or decoder, its caches and its inputs.  Language-model steps keep their plan (positions, pages) from pass to
pass and take the tokens that the pass before fed back; codec chunks continue their stream.

`exact` restates every path in 64-bit torch: no caches in 16 bits, no rounding between the operations.
"""
import functools
import math

import numpy as np
import torch
import torch.nn.functional as F

from vox_serve_amd import synth
from vox_serve_amd.engine import CSMCfg, CSMEngine, LMEngine, Qwen3Cfg, Qwen3Engine
from vox_serve_amd.engine_hybrid import HybridCfg, HybridEngine, MixerCfg, MoECfg
from vox_serve_amd.model import kazozen
from vox_serve_amd.model.glm_voice import GLMVoiceConfig, pack_glm_weights
from vox_serve_amd.tokenizer.cosyvoice2 import CosyVoice2Decoder
from vox_serve_amd.tokenizer.cosyvoice_flow import FlowConfig
from vox_serve_amd.tokenizer.hifigan import HiFTConfig
from vox_serve_amd.tokenizer.mimi import MimiConfig, MimiDecoder
from vox_serve_amd.tokenizer.mimi import param_shapes as mimi_shapes
from vox_serve_amd.tokenizer.qwen3_codec import Qwen3CodecConfig, Qwen3TTSDecoder
from vox_serve_amd.tokenizer.qwen3_codec import param_shapes as codec_shapes

DEV = "cuda"
PAGE = 128


def listed():
    return [
        # one stream being spoken: a frame of audio tokens in the middle of a sentence
        dict(name="qwen3_frame_b1", kind="qwen3_frame", batch=1, kv=200, top_k=0),
        # continuous batching at 32 requests with the sampling that the model ships with (top-k 50, temperature 0.9)
        dict(name="qwen3_frame_b32", kind="qwen3_frame", batch=32, kv=325, top_k=50),
        # a request arrives: 64 text tokens and the prompt template around them
        dict(name="qwen3_prefill_75", kind="qwen3_prefill", rows=75),
        # the first audio of a stream tuned for a fast start: two frames of one request
        dict(name="qwen3_codec_b1_t2", kind="qwen3_codec", batch=1, frames=2, precision="fp32"),
        # one stream's regular chunk of ten frames
        dict(name="qwen3_codec_b1_t10", kind="qwen3_codec", batch=1, frames=10, precision="fp32"),
        # 32 streams' chunks together
        dict(name="qwen3_codec_b32_t10", kind="qwen3_codec", batch=32, frames=10, precision="fp32"),
        # CSM-1B at 16 requests: backbone and 31 depth passes a frame
        dict(name="csm_frame_b16", kind="csm_frame", batch=16, kv=125),
        # its codec at the same load
        dict(name="mimi_b16_t10", kind="mimi", batch=16, frames=10),
        # CosyVoice2's detokenizer: a 28-token window of 8 requests through flow matching and vocoder
        dict(name="cosyvoice2_detok_b8", kind="cosyvoice2_detok", batch=8, tokens=28),
        # GLM-4-Voice-9B, one GPU's 8 requests, the model's own top-p sampling
        dict(name="glm_frame_b8", kind="glm_frame", batch=8, kv=128),
        # the hybrid engine: a long prompt of a text request
        dict(name="kazozen_prefill_2048", kind="kazozen_prefill", rows=2048),
        # and 8 requests generating text
        dict(name="kazozen_decode_b8", kind="kazozen_decode", batch=8, context=1024),
    ]


def draw(rng):
    def log(lo, hi):
        return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))
    kind = rng.choice(["qwen3_frame", "qwen3_prefill", "qwen3_codec", "qwen3_codec", "csm_frame", "mimi", "cosyvoice2_detok", "glm_frame",
                       "kazozen_prefill", "kazozen_decode"])
    if kind == "qwen3_frame":
        return dict(kind=kind, batch=log(1, 32), kv=log(64, 2000), top_k=rng.choice([0, 50]))
    if kind == "qwen3_prefill":
        return dict(kind=kind, rows=log(16, 1000))
    if kind == "qwen3_codec":
        return dict(kind=kind, batch=log(1, 32), frames=rng.randint(1, 10), precision=rng.choice(["fp32", "fp32", "bf16"]))
    if kind == "csm_frame":
        return dict(kind=kind, batch=log(1, 16), kv=log(64, 1000))
    if kind == "mimi":
        return dict(kind=kind, batch=log(1, 16), frames=rng.randint(1, 10))
    if kind == "cosyvoice2_detok":
        return dict(kind=kind, batch=rng.randint(1, 8), tokens=rng.randint(10, 28))
    if kind == "glm_frame":
        return dict(kind=kind, batch=log(1, 8), kv=log(64, 900))
    if kind == "kazozen_prefill":
        return dict(kind=kind, rows=log(64, 2048))
    return dict(kind=kind, batch=log(1, 8), context=log(64, 2000))


# ---- weights, made once per process ----------------------------------------------------------------------------------------------------

def _on_gpu(W):
    return {k: v.to(DEV) for k, v in W.items()}


def kazozen_cfg(width=2048, blocks=3, vocab=32000):
    """Window attention + dense unit | the same on shared keys and values + 8 routed experts, twice per block (the layer pattern that
    `bench.py --kazozen` drives)."""
    h = width // 128

    def attn(kv_from, **ff):
        return MixerCfg("window_attention", h, 128, 128, kv_heads=h // 4, window=1024, keep_first=4, scale=128 ** -0.5, rot_dims=128, rot_base=1e6,
                        rot_yarn=(4.0, 4096.0, 32.0, 1.0), kv_from=kv_from, out_gate=True, qk_norm_whole=True, block="post_norm", **ff)
    dense = dict(ff=(8 * width // 3 + 255) // 256 * 256, ff_kind="gated", ff_act="swish", ff_limit=7.0, ff_alpha=1.702, ff_up_offset=1.0)
    layers = []
    for _ in range(2 * blocks):
        moe = MoECfg(experts=8, identity=0, top=2, ff=width, limit=7.0, act_alpha=1.702, score="sigmoid", renorm=False, up_offset=1.0, groups=4,
                     keep=2, group_best_two=True)
        layers += [attn(None, **dense), attn(len(layers), moe=moe)]
    return HybridCfg(width, vocab, 1e-5, layers, None, norm_kind="layer", embed_scale=width ** 0.5, logit_softcap=30.0, bigram=(4096, 1009, 17))


def _kazozen_weights(cfg):
    """Random checkpoint tensors under the names that `kazozen.pack_weights` reads."""
    g, W = torch.Generator(device=DEV).manual_seed(0), cfg.width

    def lin(*shape):
        return (torch.randn(*shape, generator=g, device=DEV) / shape[-1] ** 0.5).to(torch.bfloat16)

    def vec(n, mean=0.0):
        return (mean + 0.1 * torch.randn(n, generator=g, device=DEV)).to(torch.bfloat16)
    S = {"embed": lin(cfg.vocab, W), "final.norm": vec(W, 1.0), "final.norm.b": vec(W), "bigram": 0.5 * lin(cfg.bigram[0] + 1, W) * W ** 0.5}
    for i, m in enumerate(cfg.layers):
        p, q, H, G, d, e = f"l{i}.mix.", f"l{i}.mlp.", m.heads, m.kv_heads, m.dim, m.vdim
        for n in ("norm1", "norm2"):
            S.update({f"l{i}.{n}": vec(W, 1.0), f"l{i}.{n}.b": vec(W)})
        S.update({p + "q": lin(H * d, W), p + "q.b": vec(H * d), p + "q.norm": vec(H * d, 1.0), p + "g": lin(H * e, W), p + "sink": vec(H), p + "o": lin(W, H * e)})
        if m.kv_from is None:
            S.update({p + "k": lin(G * d, W), p + "k.b": vec(G * d), p + "k.norm": vec(G * d, 1.0), p + "v": lin(G * e, W), p + "v.b": vec(G * e)})
        if m.moe is not None:
            for j in range(m.moe.experts):
                S.update({f"{q}e{j}.gate": lin(m.moe.ff, W), f"{q}e{j}.up": lin(m.moe.ff, W), f"{q}e{j}.down": lin(W, m.moe.ff)})
            S.update({q + "router": lin(m.moe.experts, W), q + "correction": vec(m.moe.experts)})
        else:
            S.update({q + "gate": lin(m.ff, W), q + "up": lin(m.ff, W), q + "down": lin(W, m.ff)})
    return S


@functools.lru_cache(maxsize=None)
def _weights(family):
    if family == "qwen3":
        return synth.synth_qwen3_weights(Qwen3Cfg(), DEV)
    if family == "qwen3_codec":
        return _on_gpu(synth.synth_qwen3_codec_weights())
    if family == "csm":
        return synth.synth_csm_weights(CSMCfg(), DEV)
    if family == "mimi":
        return _on_gpu(synth.synth_mimi_weights())
    if family == "cosyvoice2":
        W, prompt = synth.synth_cosyvoice2_codec_weights()
        return _on_gpu(W["flow"]), _on_gpu(W["hift"]), _on_gpu(prompt)
    if family == "glm":
        return synth.synth_glm_weights(GLMVoiceConfig(), DEV)
    return _kazozen_weights(kazozen_cfg())


# ---- states --------------------------------------------------------------------------------------------------------------------------

class Owner:
    """Gives the native handle back when the state goes."""

    def __init__(self, *handles):
        self.handles = handles

    def __del__(self):
        for h in self.handles:
            h.close()


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _ints(g, hi, *shape):
    return torch.randint(0, hi, shape, generator=g, device=DEV, dtype=torch.int32)


def _normal(g, std, *shape):
    return (std * torch.randn(*shape, generator=g, device=DEV)).to(torch.bfloat16)


def _pages(kv):
    return (kv + PAGE - 1) // PAGE


def _past(case, seed, heads, dim, layers):
    """What the pages hold before the pass: [layers, pages, 2, PAGE, heads, dim]."""
    return _normal(_gen(seed + 1), 0.5, layers, case["batch"] * _pages(case["kv"]), 2, PAGE, heads, dim)


def _decode_plan(B, kv, pos):
    n = _pages(kv)
    return dict(pos=[pos] * B, kvlen=[kv] * B, page=[b * n + n - 1 for b in range(B)], slot=[(kv - 1) % PAGE] * B, indptr=[b * n for b in range(B + 1)],
                indices=list(range(B * n)))


def _prompt_plan(n):
    return dict(pos=np.arange(n), kvlen=np.arange(1, n + 1), page=np.arange(n) // PAGE, slot=np.arange(n) % PAGE, q_req=np.zeros(n), last_rows=[n - 1],
                indptr=[0, _pages(n)], indices=np.arange(_pages(n)))


def _inputs(case, seed):
    """The pass's inputs: what `prepare` stages and `exact` reads."""
    g, kind = _gen(seed), case["kind"]
    if kind == "qwen3_frame":
        ids = torch.full((case["batch"], 17), Qwen3Cfg().tts_pad_id, dtype=torch.int32, device=DEV)
        ids[:, 0] = _ints(g, 2048, case["batch"])
        return dict(ids=ids, feats=_normal(g, 0.08, case["batch"], 2048))
    if kind == "qwen3_prefill":
        ids = torch.zeros(case["rows"], 17, dtype=torch.int32, device=DEV)
        ids[:, 16], ids[:, 0] = _ints(g, 151000, case["rows"]), _ints(g, 2048, case["rows"])
        masks = torch.zeros(case["rows"], dtype=torch.uint8, device=DEV)
        masks[-1] = 1
        return dict(ids=ids, masks=masks)
    if kind == "qwen3_codec":
        return dict(codes=_ints(g, 2048, case["batch"], case["frames"], 17))
    if kind == "csm_frame":
        masks = torch.ones(case["batch"], 33, dtype=torch.uint8, device=DEV)
        masks[:, 32] = 0
        return dict(ids=_ints(g, 2048, case["batch"], 33), masks=masks)
    if kind == "mimi":
        return dict(codes=_ints(g, 2048, case["batch"], case["frames"], 33))
    if kind == "cosyvoice2_detok":
        return dict(tokens=_ints(g, 6561, case["batch"], case["tokens"]))
    if kind == "glm_frame":
        c = GLMVoiceConfig()
        return dict(ids=c.audio_offset + _ints(g, c.padded_vocab_size - c.audio_offset, case["batch"]))
    n = case["rows"] if kind == "kazozen_prefill" else case["batch"] * (case["context"] + 1)
    return dict(ids=_ints(g, 32000, n))


def prepare(case, seed):
    kind, x = case["kind"], _inputs(case, seed)
    B = case.get("batch", 1)
    if kind in ("qwen3_frame", "qwen3_prefill"):
        cfg, n = Qwen3Cfg(), case.get("rows", 0)
        eng = Qwen3Engine(cfg, _weights("qwen3"), max_batch=B, page_size=PAGE, max_pages=B * _pages(case.get("kv", n)) + 1, max_seq_len=2304,
                          max_prefill_rows=max(n, 128))
        if n:
            eng.row_ids[:n], eng.row_masks[:n] = x["ids"], x["masks"]
            return dict(kind=kind, eng=eng, rows=n, plan=_prompt_plan(n), sampling=eng.sampling_cfg(greedy=True), owner=Owner(eng))
        eng.kv[:, : B * _pages(case["kv"])] = _past(case, seed, cfg.talker.kv_heads, cfg.talker.head_dim, cfg.talker.layers)
        eng.input_ids[:B], eng.input_features[:B] = x["ids"], x["feats"]
        eng.input_masks[:B] = 1
        sc = eng.sampling_cfg(greedy=False, top_k=50, temperature=0.9) if case["top_k"] else eng.sampling_cfg(greedy=True)
    elif kind == "csm_frame":
        cfg = CSMCfg()
        eng = CSMEngine(cfg, _weights("csm"), max_batch=B, page_size=PAGE, max_pages=B * _pages(case["kv"]) + 1, max_seq_len=1024, max_prefill_rows=64)
        eng.kv[:, : B * _pages(case["kv"])] = _past(case, seed, cfg.backbone.kv_heads, cfg.backbone.head_dim, cfg.backbone.layers)
        eng.input_ids[:B], eng.input_masks[:B] = x["ids"], x["masks"]
        sc = eng.sampling_cfg(greedy=True)
    elif kind == "glm_frame":
        gc = GLMVoiceConfig()
        lm = gc.lm_cfg(4096)
        layers, norm, emb, head = pack_glm_weights(_weights("glm"), gc)
        eng = LMEngine(lm, layers, norm, emb, head, None, max_batch=B, page_size=PAGE, max_pages=B * _pages(case["kv"]) + 1, max_seq_len=1024, max_prefill_rows=64)
        eng.kv[:, : B * _pages(case["kv"])] = _past(case, seed, lm.stack.kv_heads, lm.stack.head_dim, lm.stack.layers)
        eng.input_ids[:B, 0] = x["ids"]
        sc = eng.sampling_cfg(greedy=False, top_k=0, top_p=0.8, temperature=0.8)
    elif kind == "qwen3_codec":
        dec = Qwen3TTSDecoder(_weights("qwen3_codec"), device=DEV, max_batch=B, max_slots=B, detokenize_interval=10, operand_precision=case["precision"])
        return dict(kind=kind, dec=dec, cache=dec.init_cache(B), codes=x["codes"], owner=Owner(dec))
    elif kind == "mimi":
        dec = MimiDecoder(_weights("mimi"), num_codebooks=32, device=DEV, max_batch=B, max_frames=10)
        return dict(kind=kind, dec=dec, codes=x["codes"], owner=Owner(dec))
    elif kind == "cosyvoice2_detok":
        flow, hift, prompt = _weights("cosyvoice2")
        dec = CosyVoice2Decoder(flow, hift, device=DEV, max_batch=B, max_prompt_tokens=64)
        return dict(kind=kind, dec=dec, cache=dec.init_cache(prompt), tokens=x["tokens"], owner=Owner(dec))
    else:
        return _prepare_kazozen(case, x)
    return dict(kind=kind, eng=eng, batch=B, kv=case["kv"], plan=_decode_plan(B, case["kv"], case["kv"]), sampling=sc, owner=Owner(eng))


def _prepare_kazozen(case, x):
    cfg = kazozen_cfg()
    B, n = case.get("batch", 1), case.get("rows") or case["context"]
    per = _pages(n + 1)
    eng = HybridEngine(cfg, kazozen.pack_weights(_weights("kazozen"), cfg), dtype=torch.bfloat16, max_batch=B, page_size=PAGE, max_pages=B * per + 1,
                       max_seq_len=per * PAGE, max_prefill_rows=n, state_slots=B)
    sc = eng.sampling_cfg(greedy=True)
    if case["kind"] == "kazozen_prefill":
        eng.row_ids[:n, 0] = x["ids"]
        return dict(kind=case["kind"], eng=eng, rows=n, plan=dict(_prompt_plan(n), req_rows=[0, n], state=[0]), sampling=sc, owner=Owner(eng))
    tokens = x["ids"].view(B, n + 1)
    for b in range(B):
        eng.row_ids[:n, 0] = tokens[b, :n]
        eng.upload_plan(**dict(_prompt_plan(n), page=b * per + np.arange(n) // PAGE, indices=b * per + np.arange(_pages(n)), req_rows=[0, n], state=[b]))
        eng.prefill(n, 1, n, sc, feedback=False, use_graph=False)
    eng.input_ids[:B, 0] = tokens[:, n]
    plan = dict(pos=[n] * B, kvlen=[n + 1] * B, page=[b * per + n // PAGE for b in range(B)], slot=[n % PAGE] * B, q_req=np.arange(B), last_rows=np.arange(B),
                indptr=[b * per for b in range(B + 1)], indices=np.arange(B * per), req_rows=np.arange(B + 1), state=np.arange(B))
    return dict(kind=case["kind"], eng=eng, batch=B, kv=n + 1, plan=plan, sampling=sc, owner=Owner(eng))


def run(state):
    kind = state["kind"]
    if kind == "qwen3_codec":
        return dict(wav=state["dec"].decode_chunk(state["codes"], state["cache"], code_layout="BTQ")[0])
    if kind == "mimi":
        return dict(wav=state["dec"].decode(state["codes"], code_layout="BTQ"))
    if kind == "cosyvoice2_detok":
        return dict(wav=state["dec"].decode_chunk(state["tokens"], state["tokens"].shape[1], state["cache"])[0])
    eng, sc = state["eng"], state["sampling"]
    eng.upload_plan(**state["plan"])
    if kind == "kazozen_prefill":
        eng.prefill(state["rows"], 1, state["rows"], sc, feedback=False)
        return dict(logits=eng.out_logits[:1], caches=eng.caches)
    if kind == "kazozen_decode":
        eng.frame(state["batch"], state["kv"], sc, feedback=False)
        return dict(logits=eng.out_logits[: state["batch"]], caches=eng.caches)
    if kind == "qwen3_prefill":
        B = 1
        eng.prefill(state["rows"], 1, state["rows"], sc, feedback=True)
    else:
        B = state["batch"]
        eng.frame(B, state["kv"], sc, feedback=True)
    out = dict(ids=eng.out_ids[:B], logits=eng.out_logits[:B], kv=eng.kv)
    if kind in ("qwen3_frame", "qwen3_prefill"):
        # the 1024 control entries behind the codes are masked out before sampling, all but the end of the stream
        V = eng.cfg.vocab - 1024
        out.update(logits=eng.out_logits[:B, :V], end=eng.out_logits[:B, eng.cfg.eos_id], next_features=eng.input_features[:B])
    if kind != "glm_frame":
        out.update(hidden=eng.out_hidden[:B])
    return out


# ---- what a pass cannot do without --------------------------------------------------------------------------------------------------------

def _stack_params(c):
    return c.layers * (c.hidden * c.head_dim * (2 * c.heads + 2 * c.kv_heads) + 3 * c.hidden * c.ffn)


def _conv_work(shapes, steps):
    """(bf16 weight bytes, flops) of conv / linear tensors: steps(name) = how often a weight is used per request (0: a table)."""
    n = {k: math.prod(s) for k, s in shapes.items()}
    return sum(2 * v for k, v in n.items() if steps(k)), sum(2 * v * steps(k) for k, v in n.items() if len(shapes[k]) > 1)


def work(case):
    kind, B = case["kind"], case.get("batch", 1)
    if kind in ("qwen3_frame", "qwen3_prefill"):
        c = Qwen3Cfg()
        t, d, n = c.talker, c.depth, case.get("rows", B)
        pt, pd = _stack_params(t) + 2 * c.text_hidden * c.text_hidden, _stack_params(d) + t.hidden * d.hidden
        heads = (c.n_groups - 1) * c.depth_vocab * d.hidden
        kv_row = t.layers * 2 * t.kv_heads * t.head_dim * 2
        seen = B * case["kv"] if "kv" in case else n
        pairs = B * case["kv"] if "kv" in case else n * (n + 1) / 2
        return dict(bytes=2 * (pt + pd + heads + c.vocab * t.hidden) + seen * kv_row + n * (4 * t.hidden + 68),
                    flops=2 * n * pt + 2 * B * ((c.n_groups - 1) * pd + heads + c.vocab * t.hidden) + 4 * pairs * t.layers * t.heads * t.head_dim)
    if kind == "csm_frame":
        c = CSMCfg()
        b, d, G = c.backbone, c.depth, c.n_codebooks
        pb, pd, heads = _stack_params(b), _stack_params(d) + b.hidden * d.hidden, (G - 1) * c.vocab * d.hidden
        return dict(bytes=2 * (pb + pd + heads + c.vocab * b.hidden) + B * case["kv"] * b.layers * 4 * b.kv_heads * b.head_dim + B * 2 * (G + 1) * b.hidden,
                    flops=2 * B * (pb + (G - 1) * pd + heads + c.vocab * b.hidden) + 4 * B * case["kv"] * b.layers * b.heads * b.head_dim)
    if kind == "glm_frame":
        g = GLMVoiceConfig()
        c = g.lm_cfg().stack
        p = _stack_params(c) + g.padded_vocab_size * c.hidden
        return dict(bytes=2 * p + B * case["kv"] * c.layers * 4 * c.kv_heads * c.head_dim + 2 * B * g.padded_vocab_size,
                    flops=2 * B * p + 4 * B * case["kv"] * c.layers * c.heads * c.head_dim)
    if kind == "qwen3_codec":
        c, T = Qwen3CodecConfig(), case["frames"]

        def steps(k):
            if "_codebook" in k or "input_proj.weight" in k and k.startswith("quantizer"):
                return 0
            if k.startswith("upsample."):
                u = int(k.split(".")[1])
                return T * 2 ** u * (1 if ".0.conv" in k else 2)
            if k.startswith("decoder."):
                i = int(k.split(".")[1])
                r = T * 4 * math.prod(c.upsample_rates[: min(i, 4)])
                return r // c.upsample_rates[i - 1] if ".block.1.conv" in k else r
            return T
        w, f = _conv_work(codec_shapes(c), steps)
        return dict(bytes=w + B * T * (68 + 4 * 1920 + 16 * 1024), flops=B * f)
    if kind == "mimi":
        c, T = MimiConfig(), case["frames"]

        def steps(k):
            if "_codebook" in k:
                return 0
            if k.startswith("quantizer") or k.startswith("upsample"):
                return T
            if k.startswith("decoder.model."):
                i = int(k.split(".")[2])                  # 0 | 2, 3 | 5, 6 | 8, 9 | 11, 12 | 14
                r = 2 * T * math.prod(c.ratios[: min((i + 1) // 3, 4)])
                return r // c.ratios[(i + 1) // 3 - 1] if "convtr" in k else r
            return 2 * T
        w, f = _conv_work(mimi_shapes(c), steps)
        return dict(bytes=w + B * T * (132 + 4 * 1920 + 32 * 1024), flops=B * f)
    if kind == "cosyvoice2_detok":
        T, f = case["tokens"], FlowConfig()
        fw, hw, _ = _weights_shapes()

        def flow_steps(k):
            if k in ("input_embedding.weight", "spk_embed_affine_layer.weight") or "time_mlp" in k or ".mlp.1." in k:
                return 0
            if k.startswith("decoder."):
                return 2 * 2 * T * f.n_timesteps          # both guidance branches of every step
            return T if k.startswith("encoder.encoders") or "embed.out" in k and "up_" not in k or "pre_look" in k else 2 * T

        def hift_steps(k):
            up = HiFTConfig().upsample_rates
            if k.startswith("ups."):
                return 2 * T * math.prod(up[: int(k.split(".")[1])])
            if k.startswith("resblocks.") or k.startswith("source_resblocks.") or k.startswith("source_downs."):
                i = int(k.split(".")[1])
                return 2 * T * math.prod(up[: (i // 3 if k.startswith("resblocks.") else i) + 1])
            return 2 * T * math.prod(up) if k.startswith("conv_post") else 2 * T
        w1, f1 = _conv_work(fw, flow_steps)
        w2, f2 = _conv_work(hw, hift_steps)
        return dict(bytes=w1 + w2 + B * T * (4 + 4 * 960), flops=B * (f1 + f2))
    cfg = kazozen_cfg()
    W, n = cfg.width, case.get("rows", B)
    seen, m0 = case.get("context", 0) + 1, cfg.layers[0]
    read, per_row = W * cfg.vocab, 0
    for m in cfg.layers:
        mix, e = m.n_in * W + W * m.heads * m.vdim, m.moe
        used = min(e.experts, n * e.top) if e else 0
        read += mix + (3 * used * e.ff * W + 2 * e.experts * W if e else 3 * m.ff * W)
        per_row += mix + (3 * e.top * e.ff * W if e else 3 * m.ff * W)
    pairs = sum(min(i + 1, m0.window + m0.keep_first) for i in range(n)) if "rows" in case else B * min(seen, m0.window + m0.keep_first)
    rows_seen = n if "rows" in case else pairs
    return dict(bytes=2 * read + rows_seen * (len(cfg.layers) // 2) * 2 * m0.cache_values() + B * 4 * cfg.vocab + n * 4,
                flops=2 * (n * per_row + B * W * cfg.vocab) + 4 * pairs * len(cfg.layers) * m0.heads * m0.dim)


@functools.lru_cache(maxsize=None)
def _weights_shapes():
    flow, hift, prompt = _weights("cosyvoice2")
    return {k: tuple(v.shape) for k, v in flow.items()}, {k: tuple(v.shape) for k, v in hift.items() if v.dim() == 3 and v.shape[1:] != (1, 1)}, None


def tolerance(case):
    """The speech LMs promise their tokens and bits (a fixed order of every sum); elsewhere about four times the distance from `exact`."""
    if case["kind"] in ("qwen3_frame", "qwen3_prefill", "csm_frame", "glm_frame"):
        return "exact"
    return dict(rel=RELATIVE[case["kind"] + ("_bf16" if case.get("precision") == "bf16" else "")])


RELATIVE = {"qwen3_codec": 2.5e-4, "qwen3_codec_bf16": 0.03, "mimi": 1e-5, "cosyvoice2_detok": 3e-3, "kazozen_prefill": 0.03, "kazozen_decode": 0.03}


# ---- the same in 64 bits -----------------------------------------------------------------------------------------------------------------

def _d(t):
    return t.double()


def _rms(x, w, eps):
    return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + eps) * _d(w)


def _angles(pos, c):
    rot = c.rope_dim or c.head_dim
    f = c.rope_theta ** (-torch.arange(0, rot, 2, dtype=torch.float64, device=DEV) / rot)
    if c.rope_llama31:
        lo, hi, ctx = c.rope_llama31
        s = ((f * ctx / (2 * math.pi) - lo) / (hi - lo)).clamp(0, 1)
        f = (1 - s) * f / c.rope_scale + s * f
    else:
        f = f / c.rope_scale
    return pos.double()[:, None, None] * f


def _turn(x, ang, interleave):
    n = 2 * ang.shape[-1]
    r, rest = x[..., :n], x[..., n:]
    a, b = (r[..., 0::2], r[..., 1::2]) if interleave else (r[..., : n // 2], r[..., n // 2:])
    a, b = a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()
    return torch.cat([torch.stack([a, b], -1).flatten(-2) if interleave else torch.cat([a, b], -1), rest], -1)


def _stack(layer, c, x, pos, past):
    """Decoder layers.  layer(i): tensors by name.  past: None (the rows are one causal sequence) or (pages [layers, B * n, ...], visible tokens):
    one row per request behind its cached tokens."""
    R, ang = x.shape[0], _angles(pos, c)
    for i in range(c.layers):
        L = layer(i)
        h = _rms(x, L["ln1"], c.eps)
        qkv = h @ _d(L["wqkv"]).T + (_d(L["bqkv"]) if L.get("bqkv") is not None else 0)
        q, k, v = (t.view(R, -1, c.head_dim) for t in qkv.split([c.heads * c.head_dim, c.kv_heads * c.head_dim, c.kv_heads * c.head_dim], -1))
        if c.qk_norm:
            q, k = _rms(q, L["qnorm"], c.eps), _rms(k, L["knorm"], c.eps)
        q, k = _turn(q, ang, c.rope_interleave), _turn(k, ang, c.rope_interleave)
        g = c.heads // c.kv_heads
        if past is None:
            s = torch.einsum("rhd,jhd->hrj", q, k.repeat_interleave(g, 1)) / math.sqrt(c.head_dim)
            later = torch.ones(R, R, dtype=torch.bool, device=DEV).triu(1)
            a = torch.einsum("hrj,jhd->rhd", s.masked_fill(later, -math.inf).softmax(-1), v.repeat_interleave(g, 1))
        else:
            pages, n = past
            old = _d(pages[i]).view(R, -1, 2, PAGE, c.kv_heads, c.head_dim).transpose(1, 2).reshape(R, 2, -1, c.kv_heads, c.head_dim)[:, :, : n - 1]
            K, V = torch.cat([old[:, 0], k[:, None]], 1), torch.cat([old[:, 1], v[:, None]], 1)
            s = torch.einsum("rhd,rjhd->rhj", q, K.repeat_interleave(g, 2)) / math.sqrt(c.head_dim)
            a = torch.einsum("rhj,rjhd->rhd", s.softmax(-1), V.repeat_interleave(g, 2))
        x = x + a.reshape(R, -1) @ _d(L["wo"]).T
        h = _rms(x, L["ln2"], c.eps)
        x = x + (F.silu(h @ _d(L["wgate"]).T) * (h @ _d(L["wup"]).T)) @ _d(L["wdown"]).T
    return x


def _by_name(W, prefix):
    def layer(i):
        p = f"{prefix}.layers.{i}."
        a, m = p + "self_attn.", p + "mlp."
        return dict(ln1=W[p + "input_layernorm.weight"], ln2=W[p + "post_attention_layernorm.weight"], qnorm=W.get(a + "q_norm.weight"), knorm=W.get(a + "k_norm.weight"),
                    wqkv=torch.cat([W[a + n + "_proj.weight"] for n in "qkv"], 0), wo=W[a + "o_proj.weight"], wgate=W[m + "gate_proj.weight"],
                    wup=W[m + "up_proj.weight"], wdown=W[m + "down_proj.weight"])
    return layer


def _exact_qwen3(case, seed):
    c, W, x = Qwen3Cfg(), _weights("qwen3"), _inputs(case, seed)
    B, ids = case.get("batch", 1), x["ids"].long()
    lin = lambda n, t: t @ _d(W[n + ".weight"]).T + _d(W[n + ".bias"])
    e = lin("talker.text_projection.linear_fc2", F.silu(lin("talker.text_projection.linear_fc1", _d(W["talker.model.text_embedding.weight"][ids[:, 16]]))))
    codec = _d(W["talker.model.codec_embedding.weight"][ids[:, 0]])
    if "rows" in case:
        e = e + x["masks"].double()[:, None] * codec
        h = _stack(_by_name(W, "talker.model"), c.talker, e, torch.arange(case["rows"], device=DEV), None)[-1:]
    else:
        past = _past(case, seed, c.talker.kv_heads, c.talker.head_dim, c.talker.layers), case["kv"]
        h = _stack(_by_name(W, "talker.model"), c.talker, e + codec + _d(x["feats"]), torch.full((B,), case["kv"], device=DEV), past)
    h = _rms(h, W["talker.model.norm.weight"], c.talker.eps)
    logits = h @ _d(W["talker.codec_head.weight"]).T
    return dict(ids=None, logits=logits[:, : c.vocab - 1024], end=logits[:, c.eos_id], kv=None, next_features=None, hidden=h)


def _exact_csm(case, seed):
    c, W, x = CSMCfg(), _weights("csm"), _inputs(case, seed)
    ids = x["ids"].long()[:, :32] + torch.arange(32, device=DEV) * c.vocab
    e = _d(W["backbone_model.embed_tokens.embed_audio_tokens.weight"][ids]).sum(1)
    b = c.backbone
    h = _stack(_by_name(W, "backbone_model"), b, e, torch.full((case["batch"],), case["kv"], device=DEV), (_past(case, seed, b.kv_heads, b.head_dim, b.layers), case["kv"]))
    h = _rms(h, W["backbone_model.norm.weight"], b.eps)
    return dict(ids=None, logits=h @ _d(W["lm_head.weight"]).T, kv=None, hidden=h)


def _exact_glm(case, seed):
    g, x = GLMVoiceConfig(), _inputs(case, seed)
    c = g.lm_cfg().stack
    layers, norm, emb, head = pack_glm_weights(_weights("glm"), g)
    h = _stack(lambda i: layers[i], c, _d(emb[x["ids"].long()]), torch.full((case["batch"],), case["kv"], device=DEV),
               (_past(case, seed, c.kv_heads, c.head_dim, c.layers), case["kv"]))
    h = _rms(h, norm, c.eps)
    return dict(ids=None, logits=torch.cat([h @ _d(w).T for w in head.split(16384)], -1), kv=None)


def _conv(x, w, b=None, dilation=1, stride=1):
    """Conv1d without padding, one product per tap.  x [B, C, T], w [O, C, k]."""
    k, n = w.shape[2], (x.shape[2] - (w.shape[2] - 1) * dilation - 1) // stride + 1
    y = sum(_d(w[:, :, j]).contiguous() @ x[:, :, j * dilation: j * dilation + (n - 1) * stride + 1: stride].contiguous() for j in range(k))
    return y if b is None else y + _d(b)[None, :, None]


def _causal(x, w, b, dilation=1):
    return _conv(F.pad(x, ((w.shape[2] - 1) * dilation, 0)), w, b, dilation)


def _same(x, w, b, dilation=1):
    p = (w.shape[2] - 1) * dilation // 2
    return _conv(F.pad(x, (p, p)), w, b, dilation)


def _tconv(x, w, b, stride):
    """ConvTranspose1d, untrimmed.  w [C, O, k]."""
    B, _, T = x.shape
    k = w.shape[2]
    y = x.new_zeros(B, w.shape[1], (T - 1) * stride + k)
    for j in range(k):
        y[:, :, j: j + (T - 1) * stride + 1: stride] += _d(w[:, :, j]).T.contiguous() @ x
    return y if b is None else y + _d(b)[None, :, None]


def _exact_qwen3_codec(case, seed):
    c, W, B, T = Qwen3CodecConfig(), _weights("qwen3_codec"), case["batch"], case["frames"]
    codes = _inputs(case, seed)["codes"].long()
    book = lambda name, j: _d(W[f"quantizer.{name}.vq.layers.{j}._codebook.embedding_sum"]) / \
        _d(W[f"quantizer.{name}.vq.layers.{j}._codebook.cluster_usage"]).clamp(min=1e-5)[:, None]
    rest = sum(book("rvq_rest", j)[codes[:, :, j + 1]] for j in range(c.num_quantizers - 1))
    h = book("rvq_first", 0)[codes[:, :, 0]] @ _d(W["quantizer.rvq_first.output_proj.weight"][:, :, 0]).T + rest @ _d(W["quantizer.rvq_rest.output_proj.weight"][:, :, 0]).T
    h = _causal(h.transpose(1, 2), W["pre_conv.conv.weight"], W["pre_conv.conv.bias"]).transpose(1, 2)
    p = "pre_transformer."
    lin = lambda n, t: t @ _d(W[p + n + ".weight"]).T + (_d(W[p + n + ".bias"]) if p + n + ".bias" in W else 0)
    h = lin("input_proj", h)
    H, D, Wn = c.num_heads, c.head_dim, c.sliding_window
    inv = c.rope_theta ** (-torch.arange(0, D, 2, dtype=torch.float64, device=DEV) / D)
    ang = torch.arange(T, device=DEV).double()[:, None, None] * inv
    # the window's slots before the start of the stream hold zeros and are seen
    seen = torch.arange(Wn, device=DEV)[None] <= (Wn - T + torch.arange(T, device=DEV))[:, None]
    for i in range(c.num_layers):
        L = f"layers.{i}."
        n = _rms(h, W[p + L + "input_layernorm.weight"], c.rms_eps)
        q, k, v = (lin(L + f"self_attn.{s}_proj", n).view(B, T, H, D) for s in "qkv")
        q, k = _turn(q, ang, False), _turn(k, ang, False)
        K, V = (F.pad(t, (0, 0, 0, 0, Wn - T, 0)) for t in (k, v))
        s = torch.einsum("bthd,bjhd->bhtj", q, K) / math.sqrt(D)
        a = torch.einsum("bhtj,bjhd->bthd", s.masked_fill(~seen, -math.inf).softmax(-1), V).reshape(B, T, H * D)
        h = h + _d(W[p + L + "self_attn_layer_scale.scale"]) * lin(L + "self_attn.o_proj", a)
        n = _rms(h, W[p + L + "post_attention_layernorm.weight"], c.rms_eps)
        h = h + _d(W[p + L + "mlp_layer_scale.scale"]) * lin(L + "mlp.down_proj", F.silu(lin(L + "mlp.gate_proj", n)) * lin(L + "mlp.up_proj", n))
    h = lin("output_proj", _rms(h, W[p + "norm.weight"], c.rms_eps)).transpose(1, 2)
    for u, f_ in enumerate(c.upsampling_ratios):
        p = f"upsample.{u}."
        h = _tconv(h, W[p + "0.conv.weight"], W[p + "0.conv.bias"], f_)
        w = _d(W[p + "1.dwconv.conv.weight"])[:, 0]
        e = F.pad(h, (6, 0))
        y = sum(w[None, :, j, None] * e[:, :, j: j + h.shape[2]] for j in range(7)) + _d(W[p + "1.dwconv.conv.bias"])[None, :, None]
        y = F.layer_norm(y.transpose(1, 2), (h.shape[1],), _d(W[p + "1.norm.weight"]), _d(W[p + "1.norm.bias"]), 1e-6)
        y = F.gelu(y @ _d(W[p + "1.pwconv1.weight"]).T + _d(W[p + "1.pwconv1.bias"])) @ _d(W[p + "1.pwconv2.weight"]).T + _d(W[p + "1.pwconv2.bias"])
        h = h + (_d(W[p + "1.gamma"]) * y).transpose(1, 2)

    def snake(t, n):
        a, b = _d(W[n + ".alpha"]).exp()[None, :, None], _d(W[n + ".beta"]).exp()[None, :, None]
        return t + (t * a).sin().square() / (b + 1e-9)
    h = _causal(h, W["decoder.0.conv.weight"], W["decoder.0.conv.bias"])
    nb = len(c.upsample_rates)
    for b, r in enumerate(c.upsample_rates):
        p = f"decoder.{b + 1}.block."
        n = h.shape[2] * r
        h = _tconv(snake(h, p + "0"), W[p + "1.conv.weight"], W[p + "1.conv.bias"], r)[:, :, :n]
        for u, d in enumerate((1, 3, 9)):
            q = f"{p}{u + 2}."
            y = _causal(snake(h, q + "act1"), W[q + "conv1.conv.weight"], W[q + "conv1.conv.bias"], d)
            h = h + _conv(snake(y, q + "act2"), W[q + "conv2.conv.weight"], W[q + "conv2.conv.bias"])
    wav = _causal(snake(h, f"decoder.{nb + 1}"), W[f"decoder.{nb + 2}.conv.weight"], W[f"decoder.{nb + 2}.conv.bias"])
    return dict(wav=wav.clamp(-1, 1))


def _exact_mimi(case, seed):
    c, W, B = MimiConfig(), _weights("mimi"), case["batch"]
    codes = _inputs(case, seed)["codes"].long()
    book = lambda name, j: _d(W[f"quantizer.{name}.vq.layers.{j}._codebook.embedding_sum"]) / \
        _d(W[f"quantizer.{name}.vq.layers.{j}._codebook.cluster_usage"]).clamp(min=1e-5)[:, None]
    rest = sum(book("rvq_rest", j)[codes[:, :, j + 1]] for j in range(c.n_q - 1))
    x = book("rvq_first", 0)[codes[:, :, 0]] @ _d(W["quantizer.rvq_first.output_proj.weight"][:, :, 0]).T + rest @ _d(W["quantizer.rvq_rest.output_proj.weight"][:, :, 0]).T
    w, T = _d(W["upsample.convtr.convtr.convtr.weight"])[:, 0], 2 * x.shape[1]
    y = x.new_zeros(B, T + 2, c.dim)
    for j in range(4):
        y[:, j: j + T - 1: 2] += x * w[:, j]
    x, H, D = y[:, :T], c.num_heads, c.dim // c.num_heads
    ang = torch.arange(T, device=DEV).double()[:, None, None] * c.max_period ** (-torch.arange(0, D, 2, dtype=torch.float64, device=DEV) / D)
    gap = torch.arange(T, device=DEV)[:, None] - torch.arange(T, device=DEV)[None]
    for i in range(c.num_layers):
        p = f"decoder_transformer.transformer.layers.{i}."
        n = F.layer_norm(x, (c.dim,), _d(W[p + "norm1.weight"]), _d(W[p + "norm1.bias"]), 1e-5)
        q, k, v = (n @ _d(W[p + "self_attn.in_projs.0.weight"]).T).view(B, T, 3, H, D).unbind(2)
        q, k = _turn(q, ang, True), _turn(k, ang, True)
        s = torch.einsum("bthd,bjhd->bhtj", q, k) / math.sqrt(D)
        a = torch.einsum("bhtj,bjhd->bthd", s.masked_fill((gap < 0) | (gap >= c.context), -math.inf).softmax(-1), v).reshape(B, T, c.dim)
        x = x + _d(W[p + "layer_scale_1.scale"]) * (a @ _d(W[p + "self_attn.out_projs.0.weight"]).T)
        n = F.layer_norm(x, (c.dim,), _d(W[p + "norm2.weight"]), _d(W[p + "norm2.bias"]), 1e-5)
        x = x + _d(W[p + "layer_scale_2.scale"]) * (F.gelu(n @ _d(W[p + "linear1.weight"]).T) @ _d(W[p + "linear2.weight"]).T)
    wb = lambda n: (W[f"decoder.model.{n}.weight"], W[f"decoder.model.{n}.bias"])
    x, i = _causal(x.transpose(1, 2), *wb("0.conv.conv")), 1
    for r in c.ratios:
        n = x.shape[2] * r
        x = _tconv(F.elu(x), *wb(f"{i + 1}.convtr.convtr"), r)[:, :, :n]
        x = x + _causal(F.elu(_causal(F.elu(x), *wb(f"{i + 2}.block.1.conv.conv"))), *wb(f"{i + 2}.block.3.conv.conv"))
        i += 3
    return dict(wav=_causal(F.elu(x), *wb(f"{i + 1}.conv.conv")))


def _philox(seed, stream, n):
    """Two words of Philox4x32-10 per element: counter (element, stream, 0, 0), key = seed."""
    M = 0xFFFFFFFF
    c = [np.arange(n, dtype=np.uint64), np.full(n, stream & M, np.uint64), np.zeros(n, np.uint64), np.zeros(n, np.uint64)]
    k0, k1 = seed & M, seed >> 32 & M
    for _ in range(10):
        a, b = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
        c = [(b >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), b & np.uint64(M), (a >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), a & np.uint64(M)]
        k0, k1 = k0 + 0x9E3779B9 & M, k1 + 0xBB67AE85 & M
    return (c[0] >> np.uint64(8)).astype(np.float64) / 2 ** 24, (c[1] >> np.uint64(8)).astype(np.float64) / 2 ** 24


def _normals(seed, stream, *shape):
    u, v = _philox(seed, stream, math.prod(shape))
    return torch.from_numpy((np.sqrt(-2 * np.log(u + 2.0 ** -24)) * np.cos(2 * math.pi * v)).reshape(shape)).to(DEV)


class _Flow64:
    """CosyVoice2's token -> mel flow (conformer encoder, ten Euler steps of the guided estimator) against a prompt's caches."""

    def __init__(self, W):
        self.c, self.W, self.es = FlowConfig(), W, "decoder.estimator."

    def w(self, n):
        return _d(self.W[n])

    def lin(self, x, n):
        return x @ self.w(n + ".weight").T + (self.w(n + ".bias") if n + ".bias" in self.W else 0)

    def ln(self, x, n, eps):
        return F.layer_norm(x, x.shape[-1:], self.w(n + ".weight"), self.w(n + ".bias"), eps)

    def conv(self, x, n, left=0, right=0):
        return _conv(F.pad(x, (left, right)), self.W[n + ".weight"], self.W[n + ".bias"])

    def conformer(self, x, p, old):
        B, T, D = x.shape
        H = self.c.enc_heads
        d, s = D // H, p + "self_attn."
        n = self.ln(x, p + "norm_mha", 1e-12)
        q, k, v = (self.lin(n, s + "linear_" + t).view(B, T, H, d) for t in "qkv")
        if old is not None:
            k, v = torch.cat([old[0].expand(B, -1, -1, -1), k], 1), torch.cat([old[1].expand(B, -1, -1, -1), v], 1)
        n = k.shape[1]
        # row r of the table encodes position n - 1 - r; with n keys the entry of query i and key j is row T - 1 - i + j (the shifted product)
        at = torch.arange(n - 1, -n, -1, dtype=torch.float64, device=DEV)[:, None] * torch.exp(torch.arange(0, D, 2, dtype=torch.float64, device=DEV) * -(math.log(10000.0) / D))
        table = torch.stack([at.sin(), at.cos()], -1).flatten(1)
        pe = (table @ self.w(s + "linear_pos.weight").T).view(2 * n - 1, H, d)
        bd = torch.einsum("bthd,rhd->bhtr", q + self.w(s + "pos_bias_v"), pe)
        bd = self.shifted(bd)
        a = ((torch.einsum("bthd,bjhd->bhtj", q + self.w(s + "pos_bias_u"), k) + bd) / math.sqrt(d)).softmax(-1)
        x = x + self.lin(torch.einsum("bhtj,bjhd->bthd", a, v).reshape(B, T, D), s + "linear_out")
        h = self.ln(x, p + "norm_ff", 1e-12)
        return x + self.lin(F.silu(self.lin(h, p + "feed_forward.w_1")), p + "feed_forward.w_2"), (k, v)

    @staticmethod
    def shifted(x):
        B, H, T, R = x.shape
        return F.pad(x, (1, 0)).view(B, H, R + 1, T)[:, :, 1:].reshape(B, H, T, R)[..., : R // 2 + 1]

    def embed(self, x, n):
        return self.ln(self.lin(x, n + ".out.0"), n + ".out.1", 1e-5) * math.sqrt(self.c.dim)

    def encoder(self, tok, old):
        c, new = self.c, []
        x = self.embed(self.w("input_embedding.weight")[tok], "encoder.embed")
        y = F.leaky_relu(self.conv(x.transpose(1, 2), "encoder.pre_lookahead_layer.conv1", 0, c.pre_lookahead_len))
        x = x + self.conv(y, "encoder.pre_lookahead_layer.conv2", 2).transpose(1, 2)
        for i in range(c.enc_layers):
            x, kv = self.conformer(x, f"encoder.encoders.{i}.", old and old[i])
            new.append(kv)
        x = self.embed(self.conv(x.transpose(1, 2).repeat_interleave(2, 2), "encoder.up_layer.conv", 4).transpose(1, 2), "encoder.up_embed")
        for i in range(c.up_layers):
            x, kv = self.conformer(x, f"encoder.up_encoders.{i}.", old and old[c.enc_layers + i])
            new.append(kv)
        return self.lin(self.ln(x, "encoder.after_norm", 1e-5), "encoder_proj"), new

    def block(self, x, p, old, new):
        x = torch.cat([old.pop(0).expand(x.shape[0], -1, -1) if old else x.new_zeros(*x.shape[:2], 2), x], 2)
        new.append(x[..., -2:])
        return F.mish(self.ln(self.conv(x, p + "block.0").transpose(1, 2), p + "block.2", 1e-5).transpose(1, 2))

    def group(self, x, p, t, old, new):
        c, N, T = self.c, x.shape[0], x.shape[2]
        H, d = c.est_heads, c.est_head_dim
        h = self.block(x, p + "0.block1.", old, new) + self.lin(F.mish(t), p + "0.mlp.1")[None, :, None]
        x = (self.block(h, p + "0.block2.", old, new) + self.conv(x, p + "0.res_conv")).transpose(1, 2)
        for j in range(c.est_blocks):
            b = f"{p}1.{j}."
            n = self.ln(x, b + "norm1", 1e-5)
            q, k, v = (self.lin(n, b + "attn1.to_" + s).view(N, T, H, d) for s in "qkv")
            if old:
                ok, ov = old.pop(0)
                k, v = torch.cat([ok.expand(N, -1, -1, -1), k], 1), torch.cat([ov.expand(N, -1, -1, -1), v], 1)
            new.append((k, v))
            a = (torch.einsum("bthd,bjhd->bhtj", q, k) * d ** -0.5).softmax(-1)
            x = x + self.lin(torch.einsum("bhtj,bjhd->bthd", a, v).reshape(N, T, H * d), b + "attn1.to_out.0")
            x = x + self.lin(F.gelu(self.lin(self.ln(x, b + "norm3", 1e-5), b + "ff.net.0.proj")), b + "ff.net.2")
        return x.transpose(1, 2)

    def estimator(self, x, temb, old, new):
        es = self.es
        x = self.group(x, es + "down_blocks.0.", temb, old, new)
        skip = x
        x = self.conv(x, es + "down_blocks.0.2", 2)
        for i in range(self.c.est_mid_blocks):
            x = self.group(x, f"{es}mid_blocks.{i}.", temb, old, new)
        x = self.group(torch.cat([x, skip], 1), es + "up_blocks.0.", temb, old, new)
        y = self.conv(self.conv(x, es + "up_blocks.0.2", 2), es + "final_block.block.0", 2)
        return self.conv(F.mish(self.ln(y.transpose(1, 2), es + "final_block.block.2", 1e-5).transpose(1, 2)), es + "final_proj")

    def __call__(self, tok, feat, spk, z, caches):
        """-> (mel [B, 80, 2 T], [encoder caches, per step and branch estimator caches]); spk [1, 192], z [80, 2 T] shared by the batch."""
        c, B = self.c, tok.shape[0]
        spk = self.lin(F.normalize(_d(spk), dim=1), "spk_embed_affine_layer")
        mu, enc = self.encoder(tok.long(), caches and caches[0])
        cond = torch.zeros_like(mu)
        if feat is not None:
            cond[:, : feat.shape[1]] = _d(feat)
        ts = 1 - torch.cos(torch.linspace(0, 1, c.n_timesteps + 1, dtype=torch.float64) * 0.5 * math.pi)
        half = 2 * c.mel
        freqs = torch.exp(torch.arange(half, dtype=torch.float64, device=DEV) * -(math.log(10000) / (half - 1)))
        x, ests = z[None].expand(B, -1, -1), []
        both = torch.stack([mu.transpose(1, 2), spk[..., None].expand(B, -1, mu.shape[1]), cond.transpose(1, 2)])
        for i in range(c.n_timesteps):
            ang = 1000 * float(ts[i]) * freqs
            temb = self.lin(F.silu(self.lin(torch.cat([ang.sin(), ang.cos()]), self.es + "time_mlp.linear_1")), self.es + "time_mlp.linear_2")
            out = []
            for on in (1, 0):                             # with and without the conditions
                new = []
                out.append(self.estimator(torch.cat([x, *(both * on)], 1), temb, list(caches[1][2 * i + 1 - on]) if caches else [], new))
                ests.append(new)
            x = x + float(ts[i + 1] - ts[i]) * ((1 + c.inference_cfg_rate) * out[0] - c.inference_cfg_rate * out[1])
        return x, [enc, ests]

    def prompt(self, prompt, seed):
        """The caches that the speaker prompt leaves, cut to the window (its first and its last entries)."""
        c, tok = self.c, prompt["prompt_speech_token"].long()
        tok = torch.cat([tok, tok[:, :3]], 1)
        enc, ests = self(tok, prompt["prompt_feat"], prompt["embedding"], _normals(seed, 0, c.mel, 2 * tok.shape[1]), None)[1]

        def cut(t, most, first):
            return t if t.shape[1] <= most else torch.cat([t[:, :first], t[:, t.shape[1] - (most - first):]], 1)
        M, P, n = c.max_cache_len, c.prefix_len, c.enc_layers
        enc = [tuple(cut(t, M // 2, P // 2) if i < n else cut(t, M, P) for t in kv) for i, kv in enumerate(enc)]
        return [enc, [[tuple(cut(t, M, P) for t in e) if isinstance(e, tuple) else e for e in one] for one in ests]]


def _vocoder64(W, mel, seed, streams):
    """HiFT: f0 -> harmonic source -> upsampling stages with the source's spectrum -> inverse STFT."""
    c, B, T = HiFTConfig(), mel.shape[0], mel.shape[2]

    def w(n):
        g, v = W.get(n + ".parametrizations.weight.original0"), W.get(n + ".parametrizations.weight.original1")
        return W[n + ".weight"] if g is None else _d(g) * _d(v) / _d(v).flatten(1).norm(dim=1).view(-1, 1, 1)
    x = mel
    for i in range(5):
        x = F.elu(_same(x, w(f"f0_predictor.condnet.{2 * i}"), W[f"f0_predictor.condnet.{2 * i}.bias"]))
    f0 = (x.transpose(1, 2) @ _d(W["f0_predictor.classifier.weight"]).T + _d(W["f0_predictor.classifier.bias"])).squeeze(-1).abs()
    up, H = c.upsample_scale, c.nb_harmonics + 1
    L = T * up
    ini = torch.stack([torch.from_numpy(_philox(seed, s, H)[0]) for s in streams]).to(DEV)
    ini[:, 0] = 0
    noise = torch.stack([_normals(seed, s + 1, L, H) for s in streams])
    f = f0[:, :, None].repeat_interleave(up, 1)
    rad = f * torch.arange(1, H + 1, device=DEV, dtype=torch.float64) / c.sampling_rate % 1
    rad[:, 0] += ini
    rad = F.interpolate(rad.transpose(1, 2), scale_factor=1 / up, mode="linear")
    phase = F.interpolate(rad.cumsum(2) * 2 * math.pi * up, scale_factor=up, mode="linear").transpose(1, 2)
    uv = (f > c.nsf_voiced_threshold).double()
    s = phase.sin() * c.nsf_alpha * uv + (uv * c.nsf_sigma + (1 - uv) * c.nsf_alpha / 3) * noise
    s = torch.tanh(s @ _d(W["m_source.l_linear.weight"]).T + _d(W["m_source.l_linear.bias"])).squeeze(-1)
    n, hop = c.istft_n_fft, c.istft_hop_len
    win = 0.5 - 0.5 * torch.cos(2 * math.pi * torch.arange(n, dtype=torch.float64, device=DEV) / n)
    e = F.pad(s[:, None], (n // 2, n // 2), mode="reflect")[:, 0].unfold(1, n, hop) * win
    base = torch.arange(n // 2 + 1, dtype=torch.float64, device=DEV)[:, None] * torch.arange(n, device=DEV) * (2 * math.pi / n)
    spec = torch.cat([e @ base.cos().T, -(e @ base.sin().T)], 2).transpose(1, 2)

    def snake(t, n_):
        a = _d(W[n_])[None, :, None]
        return t + (t * a).sin().square() / (a + 1e-9)

    def res(t, p):
        for j, d in enumerate(c.resblock_dilation_sizes):
            y = _same(snake(t, f"{p}.activations1.{j}.alpha"), w(f"{p}.convs1.{j}"), W[f"{p}.convs1.{j}.bias"], d)
            t = t + _same(snake(y, f"{p}.activations2.{j}.alpha"), w(f"{p}.convs2.{j}"), W[f"{p}.convs2.{j}.bias"])
        return t
    x, stages = _same(mel, w("conv_pre"), W["conv_pre.bias"]), len(c.upsample_rates)
    for i, (u, k) in enumerate(zip(c.upsample_rates, c.upsample_kernel_sizes)):
        p = (k - u) // 2
        x = _tconv(F.leaky_relu(x, c.lrelu_slope), w(f"ups.{i}"), W[f"ups.{i}.bias"], u)
        x = x[:, :, p: x.shape[2] - p]
        x = F.pad(x, (1, 0), mode="reflect") if i == stages - 1 else x
        st = math.prod(c.upsample_rates[i + 1:])
        q = st // 2 if st > 1 else 0
        x = x + res(_conv(F.pad(spec, (q, q)), W[f"source_downs.{i}.weight"], W[f"source_downs.{i}.bias"], stride=st), f"source_resblocks.{i}")
        x = sum(res(x, f"resblocks.{3 * i + j}") for j in range(3)) / 3
    x = _same(F.leaky_relu(x), w("conv_post"), W["conv_post.bias"])
    nb = n // 2 + 1
    mag, ph = x[:, :nb].exp().clamp(max=1e2), x[:, nb:].sin()
    both = torch.ones(nb, device=DEV, dtype=torch.float64) * 2
    both[0] = both[-1] = 1
    frames = ((mag * ph.cos() * both[:, None]).transpose(1, 2) @ base.cos() - (mag * ph.sin() * both[:, None]).transpose(1, 2) @ base.sin()) / n * win
    out = frames.new_zeros(B, n + hop * (frames.shape[1] - 1))
    den = torch.zeros_like(out[0])
    for j in range(n // hop):
        span = hop * frames.shape[1]
        out[:, j * hop: j * hop + span] += frames[:, :, j * hop: (j + 1) * hop].reshape(B, span)
        den[j * hop: j * hop + span] += (win[j * hop: (j + 1) * hop] ** 2).repeat(frames.shape[1])
    out = out / torch.where(den > 1e-8, den, torch.ones_like(den))
    return out[:, n // 2: out.shape[1] - n // 2].clamp(-c.audio_limit, c.audio_limit)


def _exact_cosyvoice2(case, seed):
    """A decoder's first chunk: the start noise is stream 1, request b's vocoder streams begin at 2 (b + 65536)."""
    W, H, prompt = _weights("cosyvoice2")
    flow, tok = _Flow64(W), _inputs(case, seed)["tokens"]
    mel, _ = flow(tok, None, prompt["embedding"], _normals(0, 1, 80, 2 * tok.shape[1]), flow.prompt(prompt, 0))
    wav = _vocoder64(H, mel, 0, [2 * (b + 65536) for b in range(tok.shape[0])])
    n = 6 * 480
    wav[:, :n] *= torch.from_numpy(np.hamming(2 * n)[:n]).to(DEV)
    return dict(wav=wav[:, : wav.shape[1] - n])


def _kazozen64(tokens):
    """Logits of the last token of one sequence."""
    cfg = kazozen_cfg()
    S, eps, T = _weights("kazozen"), cfg.eps, tokens.shape[0]
    w = lambda n: _d(S[n])
    n, a, b = cfg.bigram
    prev = torch.cat([tokens.new_zeros(1), tokens[:-1]])
    pair = (prev * a + tokens * b) % n
    pair[0] = n
    x = w("embed")[tokens] * cfg.embed_scale + w("bigram")[pair]
    m = cfg.layers[0]
    factor, original, fast, slow = m.rot_yarn
    place = lambda t: m.rot_dims * math.log(original / (2 * math.pi * t)) / (2 * math.log(m.rot_base))
    lo, hi = max(math.floor(place(fast)), 0), min(math.ceil(place(slow)), m.rot_dims - 1)
    i = torch.arange(m.rot_dims // 2, dtype=torch.float64, device=DEV)
    f = m.rot_base ** (-2 * i / m.rot_dims)
    r = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    ang, mag = torch.arange(T, device=DEV).double()[:, None, None] * (f / factor * r + f * (1 - r)), 0.1 * math.log(factor) + 1
    gap = torch.arange(T, device=DEV)[:, None] - torch.arange(T, device=DEV)[None]
    seen = (gap >= 0) & ((gap < m.window) | (torch.arange(T, device=DEV)[None] < m.keep_first))

    def unit(h, p):
        g, u = (h @ w(p + "gate").T).clamp(max=7.0), (h @ w(p + "up").T).clamp(-7.0, 7.0)
        return (g * torch.sigmoid(1.702 * g) * (u + 1)) @ w(p + "down").T
    made = {}
    for li, m in enumerate(cfg.layers):
        p, H, G = f"l{li}.mix.", m.heads, m.kv_heads
        turned = lambda s, h: mag * _turn(_rms(x @ w(p + s).T + w(p + s + ".b"), S[p + s + ".norm"], eps).view(T, h, m.dim), ang, True)
        if m.kv_from is None:
            made[li] = turned("k", G), (x @ w(p + "v").T + w(p + "v.b")).view(T, G, m.vdim)
        q, (k, v) = turned("q", H), made[li if m.kv_from is None else m.kv_from]
        out = []
        for h in range(H):
            g = h * G // H
            s = torch.cat([(q[:, h] @ k[:, g].T * m.scale).masked_fill(~seen, -math.inf), w(p + "sink")[h].expand(T, 1)], 1)
            out.append(s.softmax(-1)[:, :-1] @ v[:, g])
        y = (torch.cat(out, 1) * torch.sigmoid(x @ w(p + "g").T)) @ w(p + "o").T
        x = x + F.layer_norm(y, y.shape[-1:], w(f"l{li}.norm1"), w(f"l{li}.norm1.b"), eps)
        p = f"l{li}.mlp."
        if m.moe is None:
            y = unit(x, p)
        else:
            e = m.moe
            s = torch.sigmoid(x @ w(p + "router").T)
            choice = s + w(p + "correction")
            rank = choice.view(T, e.groups, -1).topk(2, -1).values.sum(-1)
            kept = torch.zeros_like(rank).scatter_(1, rank.topk(e.keep, -1).indices, 1).bool().repeat_interleave(e.experts // e.groups, 1)
            pick = torch.zeros_like(s).scatter_(1, choice.masked_fill(~kept, -math.inf).topk(e.top, -1).indices, 1) * s
            y = sum(pick[:, j: j + 1] * unit(x, f"{p}e{j}.") for j in range(e.experts))
        x = x + F.layer_norm(y, y.shape[-1:], w(f"l{li}.norm2"), w(f"l{li}.norm2.b"), eps)
    z = F.layer_norm(x[-1:], x.shape[-1:], w("final.norm"), w("final.norm.b"), eps) @ w("embed").T
    return cfg.logit_softcap * torch.tanh(z / cfg.logit_softcap)


def _exact_kazozen(case, seed):
    ids = _inputs(case, seed)["ids"].long()
    logits = torch.cat([_kazozen64(t) for t in ids.view(case.get("batch", 1), -1)])
    return dict(logits=logits, caches=None)


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    return {"qwen3_frame": _exact_qwen3, "qwen3_prefill": _exact_qwen3, "csm_frame": _exact_csm, "glm_frame": _exact_glm, "qwen3_codec": _exact_qwen3_codec,
            "mimi": _exact_mimi, "cosyvoice2_detok": _exact_cosyvoice2, "kazozen_prefill": _exact_kazozen, "kazozen_decode": _exact_kazozen}[kind](case, seed)
