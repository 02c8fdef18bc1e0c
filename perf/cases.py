"""The work whose speed this repository watches: cases, inputs and limits.

``listed`` names the watched cases and ``draw`` makes others of the same
ranges; ``prepare`` builds what a program holds before a call, ``run`` is one
pass through the public entry points, ``work`` the bytes and operations that a
pass cannot do without, ``tolerance`` how far results may lie apart and
``exact`` the results restated in 64 bits with plain torch.

Kinds of cases:

* ``logmel``  log_mel_spectrogram of 16 kHz audio: the first call of a transcription
* ``encode``  EncoderRunner: mels to audio features, full encoder
* ``block``   one encoder ResidualAttentionBlock_int, called as a layer
* ``logits``  Whisper_int.logits of whole token sequences: scoring, and the pass that
              word timestamps are taken from
* ``hooks``   TextDecoder_int over the key/value hooks: a caller's own token loop
* ``decode``  greedy_decode over a DecoderRunner: the cross-attention keys and values,
              the prompt and the token steps, plain or with the decoding filters

Weights are random with parameters chosen so that activations spread over the
integer ranges as a calibrated model's do (int8 activations of deviation ~25,
a residual stream of ~3000, attention over hundreds of keys). Whisper's five
widths, head counts, depths, vocabulary and contexts come from ``SHAPES``.
"""
import math

import numpy as np
import torch

import __graft_entry__

iw = __graft_entry__.load_package()

DEVICE = "cuda"
EOT, NO_TIMESTAMPS, TIMESTAMP_BEGIN = 50257, 50363, 50364
ACT, RES = 25.0, 3000.0   # deviations of int8 activations and of the residual stream
W_STD = 32.0              # deviation of int8 weights
EXACT_FLOPS = 6e13        # up to here the 64-bit restatement takes a few seconds


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # one utterance's 30 s window of audio: the smallest call
        dict(name="logmel_b1", kind="logmel", batch=1, samples=480000, n_mels=80),
        # a single short request on the smallest model
        dict(name="encode_tiny_b1", kind="encode", shape="tiny", batch=1, ctx=1500),
        # the benchmark's encoder-only workload
        dict(name="encode_base_b16", kind="encode", shape="base", batch=16, ctx=1500),
        # a few requests that arrived together
        dict(name="encode_medium_b5", kind="encode", shape="medium", batch=5, ctx=1500),
        # transcribing one utterance after the other with the best model
        dict(name="encode_large_b1", kind="encode", shape="large", batch=1, ctx=1500),
        # the benchmark's throughput workload
        dict(name="encode_large_b128", kind="encode", shape="large", batch=128, ctx=1500),
        # a caller's own encoder loop over layers, on audio cut to its real length
        dict(name="block_small_b3_t677", kind="block", shape="small", batch=3, ctx=677),
        # scoring transcripts of one length
        dict(name="logits_small_b4_t117", kind="logits", shape="small", batch=4, tokens=117, ctx=1500),
        # the reference's decoding loop (five candidates) on the layer API
        dict(name="hooks_base_b5", kind="hooks", shape="base", batch=5, tokens=4, steps=12, ctx=1500),
        # the benchmark's single-request workload
        dict(name="decode_tiny_b1", kind="decode", shape="tiny", batch=1, tokens=3, steps=32, ctx=1500,
             filters=False),
        # a server's batch with the decoding task's own filters
        dict(name="decode_small_b27_filters", kind="decode", shape="small", batch=27, tokens=3, steps=128,
             ctx=1500, filters=True),
        # the benchmark's throughput workload, the first steps of a transcript
        dict(name="decode_large_b128", kind="decode", shape="large", batch=128, tokens=3, steps=96, ctx=1500,
             filters=False),
    ]


def draw(rng):
    def log_int(lo, hi):
        return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))

    kind = rng.choice(["logmel", "encode", "encode", "encode", "block", "block", "logits", "hooks", "decode",
                       "decode"])
    if kind == "logmel":
        return dict(kind=kind, batch=log_int(1, 32), samples=log_int(16000, 480000), n_mels=rng.choice([80, 128]))
    case = dict(kind=kind, shape=rng.choice(sorted(iw.SHAPES)))
    if kind in ("encode", "block"):
        case["batch"] = log_int(1, 128)
        case["ctx"] = rng.choice([1500, rng.randint(100, 1500)])
    elif kind == "logits":
        case.update(batch=log_int(1, 16), tokens=log_int(2, 224), ctx=1500)
    elif kind == "hooks":
        case.update(batch=log_int(1, 16), tokens=log_int(1, 32), steps=log_int(1, 16), ctx=1500)
    else:
        case.update(batch=log_int(1, 128), tokens=log_int(1, 96), steps=log_int(8, 96),
                    ctx=rng.choice([1500, rng.randint(100, 1500)]), filters=rng.choice([False, True]))
    return case


# ---------------------------------------------------------------------------
# parameters
# ---------------------------------------------------------------------------

class _Gen:
    """Seeded random tensors on the device."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEVICE)
        self.g.manual_seed(1000003 * seed + 17)

    def normal(self, shape, std, mean=0.0):
        return torch.randn(shape, generator=self.g, device=DEVICE).mul_(std).add_(mean)

    def i8(self, shape, std, mean=0.0):
        return self.normal(shape, std, mean).round_().clamp_(-127, 127).to(torch.int8)

    def i32(self, shape, std):
        return self.normal(shape, std).round_().to(torch.int32)

    def ints(self, lo, hi, shape):
        return torch.randint(lo, hi, shape, generator=self.g, device=DEVICE)


def _set(t, value):
    value = torch.as_tensor(value)
    with torch.no_grad():
        if t.dtype in (torch.uint16, torch.uint32):
            value = value.cpu().to(torch.int64).expand(t.shape).contiguous().numpy()
            t.copy_(torch.from_numpy(value.astype(np.uint16 if t.dtype == torch.uint16 else np.uint32)))
        else:
            t.copy_(value.to(t.device, t.dtype).expand(t.shape))


def _mant(r, bits, extra=0):
    """r as an integer multiplier of ``bits`` bits and a right shift."""
    f, e = math.frexp(r)
    return int(f * 2 ** bits), -e + bits + extra


def _fill_linear(layer, g, act_std, out_std, wide):
    """``wide``: an int32 branch for the residual merge, else int8 outputs."""
    n, k = layer.weight.shape
    _set(layer.weight, g.i8((n, k), W_STD))
    _set(layer.wgt_zeros, g.i8((n,), 3.0))
    acc = math.sqrt(k) * act_std * W_STD
    if layer.bias is not None:
        _set(layer.bias, g.i32((n,), 0.2 * acc))
    r = out_std / acc
    if wide:  # mulh(acc, m) << s
        f, e = math.frexp(2.0 * r)
        m, s = int(f * 2 ** 31), e
    else:  # mulh(acc, m) >> s
        f, e = math.frexp(r)
        m, s = int(f * 2 ** 31), -e - 1
    # scales of channels differ by up to a third
    spread = 1.0 - g.normal((n,), 0.15).abs_().clamp_(max=0.33)
    _set(layer.req_multiplier, torch.clamp(m * spread.double().cpu(), 2 ** 29, 2 ** 31 - 1).long())
    _set(layer.req_shiftmount, torch.full((n,), s))


def _fill_ln(ln, g, signed=False):
    n = ln.weight.shape[0]
    gamma = g.normal((n,), 9.0, 90.0).round_().clamp_(1, 127)
    if signed:
        gamma = gamma * (2 * g.ints(0, 2, (n,)) - 1)
    _set(ln.weight, gamma)
    _set(ln.bias, g.i32((n,), 6000.0))
    alpha = 16383.0 / 5.0
    m, s = _mant(alpha, 7, extra=13)
    _set(ln.ln_req_multiplier, m)
    _set(ln.ln_req_shiftmount, s)
    f, e = math.frexp(ACT / (alpha * 90.0))
    _set(ln.out_req_multiplier, int(f * 2 ** 31))
    _set(ln.out_req_shiftmount, -e - 1)


def _fill_gelu(gelu):
    lut = np.round(255.0 / (1.0 + np.exp(-np.arange(-6.0, 6.0, 0.75))))
    lut[0], lut[-1] = 0, 255
    _set(gelu.lut, torch.from_numpy(lut))
    for name, r in (("luti", 1.702 / (ACT * 0.75)), ("luto", 1.0 / 255.0)):
        m, s = _mant(r, 7)
        _set(getattr(gelu, name + "_req_multiplier"), m)
        _set(getattr(gelu, name + "_req_shiftmount"), s)


def _fill_attention(att, g, keys, score):
    """``score``: deviation of the real scores; ``keys``: how many are averaged."""
    for lin in (att.query, att.key, att.value):
        _fill_linear(lin, g, ACT, ACT, False)
    frac = 15 - (math.floor(math.log2(5.0 * score)) + 1)
    head = att.n_state // att.n_head
    m, s = _mant(score * 2 ** frac / (math.sqrt(head) * ACT * ACT), 7)
    _set(att.qk_req_multiplier, m)
    _set(att.qk_req_shiftmount, s)
    _set(att.qk_frac_bits, frac)
    m, s = _mant(math.sqrt(max(1.0, keys / math.exp(score * score))), 7)
    _set(att.av_req_multiplier, m)
    _set(att.av_req_shiftmount, s)
    _fill_linear(att.out, g, ACT, 0.25 * RES * 32768, True)


def _fill_block(block, g, keys, cross_keys):
    _fill_attention(block.attn, g, keys, 1.0)
    _fill_ln(block.attn_ln, g)
    if block.cross_attn is not None:
        _fill_attention(block.cross_attn, g, cross_keys, 1.2)
        _fill_ln(block.cross_attn_ln, g)
    _fill_linear(block.mlp[0], g, ACT, ACT, False)
    _fill_gelu(block.mlp[1])
    _fill_linear(block.mlp[2], g, 17.0, 0.25 * RES * 32768, True)
    _fill_ln(block.mlp_ln, g)
    for p in (block.attn_res_req_multiplier, block.cross_attn_res_req_multiplier, block.mlp_res_req_multiplier):
        _set(p, int(32768 * math.sqrt(1 - 0.0625)))


def _positions(ctx, d):
    inc = math.log(10000.0) / (d // 2 - 1)
    t = torch.arange(ctx)[:, None] * torch.exp(-inc * torch.arange(d // 2))[None, :]
    return torch.cat([torch.sin(t), torch.cos(t)], 1)


def _encoder(case, g):
    d = iw.SHAPES[case["shape"]]
    with torch.device(DEVICE):
        enc = iw.AudioEncoder_int(d.n_mels, case["ctx"], d.n_audio_state, d.n_audio_head, d.n_audio_layer)
    enc = enc.to(DEVICE).eval()
    _set(enc.input_alpha, 127.0 / 1.5)
    for conv, std in ((enc.conv1, 45.0), (enc.conv2, 17.0)):
        n, k = conv.weight.shape
        _set(conv.weight, g.i8((n, k), W_STD))
        acc = math.sqrt(k) * std * W_STD
        _set(conv.bias, g.i32((n,), 0.2 * acc))
        f, e = math.frexp(ACT / acc)
        _set(conv.req_multiplier, int(f * 2 ** 31))
        _set(conv.req_shiftmount, -e - 1)
    _fill_gelu(enc.gelu1)
    _fill_gelu(enc.gelu2)
    _set(enc.positional_embedding, (_positions(case["ctx"], d.n_audio_state) * ACT).round())
    m, s = _mant(RES / ACT, 15)
    _set(enc.req_multiplier, m)
    _set(enc.req_shiftmount, s)
    for b in enc.blocks:
        _fill_block(b, g, case["ctx"], 0)
    _fill_ln(enc.ln_post, g)
    return enc


def _whisper(case, g):
    """A model with its whole decoder (audio features are the decode cases' input)."""
    d = iw.SHAPES[case["shape"]]
    dims = iw.ModelDimensions(d.n_mels, case["ctx"], d.n_audio_state, d.n_audio_head, 0, d.n_vocab, d.n_text_ctx,
                              d.n_text_state, d.n_text_head, d.n_text_layer)
    with torch.device(DEVICE):
        model = iw.Whisper_int(dims)
    model = model.to(DEVICE).eval()
    dec = model.decoder
    _set(dec.token_embedding.weight, g.i8(dec.token_embedding.weight.shape, 30.0))
    _set(dec.positional_embedding, g.i8(dec.positional_embedding.shape, 12.0))
    _set(dec.req_multiplier, 100)
    _set(dec.req_shiftmount, 0)
    f, e = math.frexp(22.0 / (math.sqrt(d.n_text_state) * ACT * 30.0))
    _set(dec.clf_req_multiplier, int(f * 2 ** 31))
    _set(dec.clf_req_shiftmount, -e - 1)
    _set(dec.act_logits_alpha, 6.0)
    for b in dec.blocks:
        _fill_block(b, g, 16, case["ctx"])
    # signs of both kinds, so that the tied classifier does not repeat the input token
    _fill_ln(dec.ln, g, signed=True)
    return model


def _filters(case):
    if not case["filters"]:
        return None
    # symbols and special tokens, the blank rule and the timestamp rules, as a
    # transcription with timestamps has them
    suppress = list(range(1, 50257, 600)) + list(range(50258, 50363))
    return iw.LogitFilters(eot=EOT, suppress_tokens=suppress, suppress_blank=[220, EOT],
                           timestamp_begin=TIMESTAMP_BEGIN, no_timestamps=NO_TIMESTAMPS,
                           max_initial_timestamp_index=50)


def prepare(case, seed):
    g = _Gen(seed)
    kind, B = case["kind"], case["batch"]
    if kind == "logmel":
        n = case["samples"]
        t = torch.arange(n, device=DEVICE) / 16000.0
        f = 80.0 + 400.0 * torch.rand((B, 1), generator=g.g, device=DEVICE)
        voice = 0.2 * torch.sin(6.2831853 * f * t) * torch.sin(3.0 * t + f).clamp_min(0)
        return dict(case=case, audio=voice + g.normal((B, n), 0.01))
    if kind == "encode":
        enc = _encoder(case, g)
        mel = g.normal((B, enc.n_mels, 2 * case["ctx"]), 0.4, -0.5).clamp_(-1.5, 1.5)
        return dict(case=case, enc=enc, runner=iw.EncoderRunner(enc, B), mel=mel)
    d = iw.SHAPES[case["shape"]]
    if kind == "block":
        with torch.device(DEVICE):
            block = iw.ResidualAttentionBlock_int(d.n_audio_state, d.n_audio_head)
        block = block.to(DEVICE).eval()
        _fill_block(block, g, case["ctx"], 0)
        x = g.normal((B, case["ctx"], d.n_audio_state), RES).round_().clamp_(-16383, 16383).to(torch.int16)
        return dict(case=case, block=block, x=x)
    model = _whisper(case, g)
    state = dict(case=case, model=model, feats=g.i8((B, case["ctx"], d.n_audio_state), ACT),
                 prompt=g.ints(0, EOT, (B, case["tokens"])))
    if kind == "decode":
        state["filters"] = _filters(case)
        state["runner"] = iw.DecoderRunner(model.decoder, B, case["ctx"], filters=state["filters"])
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(state):
    case = state["case"]
    with torch.no_grad():
        return _RUN[case["kind"]](case, state)


def _run_logmel(case, s):
    return iw.audio.log_mel_spectrogram(s["audio"], case["n_mels"])


def _run_encode(case, s):
    return s["runner"](s["mel"])


def _run_block(case, s):
    return s["block"](s["x"])


def _run_logits(case, s):
    return s["model"].logits(s["prompt"], s["feats"])


def _run_hooks(case, s):
    model, tokens, picked = s["model"], s["prompt"], []
    cache, hooks = model.install_kv_cache_hooks()
    logits = model.decoder(tokens, s["feats"], kv_cache=cache)
    for _ in range(case["steps"]):
        tokens = logits[:, -1].argmax(-1, keepdim=True)
        picked.append(tokens)
        logits = model.decoder(tokens, s["feats"], kv_cache=cache)
    for h in hooks:
        h.remove()
    return dict(tokens=torch.cat(picked, 1), logits=logits)


def _run_decode(case, s):
    r = s["runner"]
    got = iw.greedy_decode(s["model"], s["feats"], s["prompt"], case["steps"], runner=r, filters=s["filters"],
                           return_result=True)
    return dict(tokens=got.tokens, sum_logprobs=got.sum_logprobs, logits=r.logits)


_RUN = dict(logmel=_run_logmel, encode=_run_encode, block=_run_block, logits=_run_logits, hooks=_run_hooks,
            decode=_run_decode)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _layer_work(rows, q, k, C, cross, B, audio_rows):
    """(operations, weight bytes) of one block over ``rows`` rows, q query and k key
    positions in each of B sequences; ``audio_rows``: rows whose cross keys and
    values are projected."""
    flops = 2.0 * rows * 12 * C * C + 4.0 * B * q * k * C
    weights = 12.0 * C * C
    if cross:
        flops += 2.0 * rows * 2 * C * C + 2.0 * audio_rows * 2 * C * C
        weights += 4.0 * C * C
    return flops, weights


def work(case):
    kind, B = case["kind"], case["batch"]
    if kind == "logmel":
        frames = B * (case["samples"] // 160)
        return dict(bytes=4.0 * B * case["samples"] + 4.0 * frames * case["n_mels"],
                    flops=frames * (5.0 * 512 * 9 + 4 * 257))
    d = iw.SHAPES[case["shape"]]
    C, V, ctx = d.n_audio_state, d.n_vocab, case["ctx"]
    if kind in ("encode", "block"):
        n = d.n_audio_layer if kind == "encode" else 1
        f, w = _layer_work(B * ctx, ctx, ctx, C, False, B, 0)
        flops, by = n * f, n * w
        if kind == "encode":
            flops += 2.0 * B * ctx * 3 * C * (2 * d.n_mels + C)
            by += 3.0 * C * (d.n_mels + C) + B * ctx * (8.0 * d.n_mels + C)
        else:
            by += 4.0 * B * ctx * C
        return dict(bytes=by, flops=flops)
    n, T = d.n_text_layer, case["tokens"]
    if kind == "logits":
        f, w = _layer_work(B * T, T, T + ctx, C, True, B, B * ctx)
        return dict(bytes=n * w + V * C + B * ctx * C + 4.0 * B * T * V,
                    flops=n * f + 2.0 * B * T * V * C)
    # The prompt, then token steps one after another: each needs the tokens of
    # the one before, so each reads the weights and the cached keys and values
    # (at large sizes far more than the caches hold).
    f, w = _layer_work(B * T, T, T + ctx, C, True, B, B * ctx)
    flops, by = n * f + 2.0 * B * (T if kind == "hooks" else 1) * V * C, n * w + V * C + B * ctx * C
    steps = case["steps"] if kind == "hooks" else case["steps"] - 1
    for i in range(steps):
        f, w = _layer_work(B, 1, T + i + 1 + ctx, C, True, B, 0)
        flops += n * f + 2.0 * B * V * C
        by += n * (w - 2.0 * C * C) + V * C + 2.0 * B * n * (T + i + 1 + ctx) * C
    return dict(bytes=by, flops=flops)


def tolerance(case):
    kind = case["kind"]
    if kind == "logmel":
        # 32-bit FFT and mel sums under a log10: 5e-7 to 9e-7 from 64 bits in norm, 1e-5 at most
        return dict(rel=4e-6, max=1e-4)
    if kind == "decode":
        # integers are exact; the sums of log-probabilities add 32-bit logarithms: 1e-7 to
        # 2e-7 from 64 bits
        return dict(rel=1e-6, max=4e-6, differ=0.0)
    return "exact"  # integers, and integers over one scale


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------

def exact(case, seed):
    if case["kind"] != "logmel" and work(case)["flops"] > EXACT_FLOPS:
        return None
    s = prepare(case, seed)
    with torch.no_grad():
        return _EXACT[case["kind"]](case, s)


def _long(t):
    if t.dtype in (torch.uint16, torch.uint32):
        return torch.from_numpy(t.detach().cpu().numpy().astype(np.int64)).to(t.device)
    return t.detach().to(torch.int64)


def _wrap(x, bits=32):
    h = 1 << (bits - 1)
    return ((x + h) & ((1 << bits) - 1)) - h


def _shr(x, s):
    """Right shift rounding half away from zero (32-bit add); s a number or a tensor, in [0, 31]."""
    s = torch.as_tensor(s, device=x.device)
    half = torch.where(s > 0, (1 << (s - 1).clamp(min=0)) - (x < 0).long(), torch.zeros_like(x))
    return _wrap(x + half) >> s


def _matmul(a, b):
    return (a.double() @ b.double()).long()


def _mulh(acc, m):
    return (_wrap(acc) * m) >> 32


def _linear(layer, x, wide=False):
    acc = _matmul(x, layer.weight.t().contiguous())
    acc -= x.long().sum(-1, keepdim=True) * _long(layer.wgt_zeros)
    if layer.bias is not None:
        acc += layer.bias
    y, s = _mulh(acc, _long(layer.req_multiplier)), _long(layer.req_shiftmount)
    return _wrap(y << s) if wide else _shr(y, s).clamp(-127, 127)


def _bits(x):
    return torch.where(x > 0, torch.frexp(x.double()).exponent.long(), torch.zeros_like(x))


def _rsqrt(x, off):
    """Integer inverse square root: the bit-level estimate and two Newton steps."""
    e = (_bits(x) - 1).clamp(min=0)
    sig = torch.where(e <= 23, x << (23 - e).clamp(min=0), x >> (e - 23).clamp(min=0)) & 0x7FFFFF
    i = torch.where(x == 0, torch.zeros_like(x), ((e + 127) << 23) | sig)
    raw = (0x5F3759DF - (i >> 1) + (off << 23)) & 0xFFFFFFFF
    e, sig = ((raw >> 23) & 255) - 127, (1 << 23) | (raw & 0x7FFFFF)
    y = torch.where(e >= 23, sig << (e - 23).clamp(0, 30), sig >> (23 - e).clamp(min=0, max=62))
    y = torch.where(e < 0, torch.zeros_like(y), _wrap(y))
    for _ in range(2):
        t = _wrap(_shr(_wrap(x * y), off) * y)
        y = _shr(_wrap(y * _wrap((3 << off) - t)), off + 1)
    return y


def _mean(v, n):
    if n in (384, 768):
        return _wrap(v + (v >> 2) + (v >> 3)) >> (9 if n == 384 else 10)
    return v >> (9 if n == 512 else 10) if n in (512, 1024) else _wrap(v + (v >> 1)) >> 11


def _ln(ln, x):
    x, n = x.long(), x.shape[-1]
    d = x - _mean(x.sum(-1, keepdim=True), n)
    sq = d * d
    rs = (_bits(sq.amax(-1, keepdim=True)) - 16).clamp(min=0)
    rs = (rs + 1) & ~1
    inv = _rsqrt(_mean(_shr(sq, rs).sum(-1, keepdim=True), n), 13)
    v = _wrap(_wrap(d * inv) * _long(ln.ln_req_multiplier))
    t = _shr(v, _long(ln.ln_req_shiftmount) + (rs >> 1)).clamp(-16383, 16383)
    y = _mulh(t * _long(ln.weight) + _long(ln.bias), _long(ln.out_req_multiplier))
    return _shr(y, _long(ln.out_req_shiftmount)).clamp(-127, 127)


def _gelu(gelu, x):
    idx = _shr(x * _long(gelu.luti_req_multiplier), _long(gelu.luti_req_shiftmount)).clamp(-8, 7) + 8
    v = x * _long(gelu.lut)[idx] * _long(gelu.luto_req_multiplier)
    return _shr(v, _long(gelu.luto_req_shiftmount)).clamp(-127, 127)


def _residual(branch, x, mult):
    return _shr(_wrap(branch + x.long() * _long(mult)), 15).clamp(-16383, 16383)


def _attend(att, q, k, v, causal):
    """Attention of q [B, Tq, C] over k and v [B, Tk, C], some sequences at a time."""
    (B, Tq, C), Tk, H = q.shape, k.shape[1], att.n_head
    n = max(1, 50_000_000 // (H * Tq * Tk))
    if n < B:
        return torch.cat([_attend(att, q[i:i + n], k[i:i + n], v[i:i + n], causal) for i in range(0, B, n)])

    def heads(t):
        return t.view(B, t.shape[1], H, C // H).transpose(1, 2).contiguous()

    score = _matmul(heads(q), heads(k).transpose(2, 3).contiguous())
    h = _shr(_wrap(score * _long(att.qk_req_multiplier)), _long(att.qk_req_shiftmount)).clamp(-32768, 32767)
    hide = None
    if causal:
        hide = torch.ones((Tq, Tk), dtype=torch.bool, device=q.device).triu_(1 + Tk - Tq)
        h = h.masked_fill(hide, -32768)
    f = int(att.qk_frac_bits)
    x = _wrap(h - (h.amax(-1, keepdim=True) + 1), 16)
    fix = _wrap(x + (x >> 1) - (x >> 4), 16)
    whole = fix >> f
    e = ((1 << f) + ((fix - (whole << f)) >> 1)) >> (-whole).clamp(0, 62)
    p = torch.where((x > 0) | (whole > 0) | (whole <= -16), torch.zeros_like(e), e)
    p = (p >> (f - 7) if f > 7 else p) & 255
    if hide is not None:
        p = p.masked_fill(hide, 0)
    inv, off = _rsqrt(p.sum(-1, keepdim=True), att.rsqrt_offset), att.rsqrt_offset
    y = _matmul(p, heads(v))
    for _ in range(2):
        y = _shr(_wrap(y * inv), off)
    y = _shr(_wrap(y * _long(att.av_req_multiplier)), _long(att.av_req_shiftmount)).clamp(-127, 127)
    return y.transpose(1, 2).reshape(B, Tq, C)


def _block(b, x, self_kv=None, cross_kv=None):
    """One block on x [B, T, C]; ``self_kv`` (a decoder): the keys and values so far,
    to which these are appended; ``cross_kv``: the audio's."""
    h = _ln(b.attn_ln, x)
    k, v = _linear(b.attn.key, h), _linear(b.attn.value, h)
    if self_kv is not None:
        k, v = (torch.cat([old, new], 1) for old, new in zip(self_kv, (k, v))) if self_kv else (k, v)
        self_kv[:] = [k, v]
    q = _linear(b.attn.query, h)
    wv = _attend(b.attn, q, k, v, self_kv is not None)
    x = _residual(_linear(b.attn.out, wv, True), x, b.attn_res_req_multiplier)
    if cross_kv is not None:
        q = _linear(b.cross_attn.query, _ln(b.cross_attn_ln, x))
        wv = _attend(b.cross_attn, q, *cross_kv, False)
        x = _residual(_linear(b.cross_attn.out, wv, True), x, b.cross_attn_res_req_multiplier)
    h = _gelu(b.mlp[1], _linear(b.mlp[0], _ln(b.mlp_ln, x)))
    return _residual(_linear(b.mlp[2], h, True), x, b.mlp_res_req_multiplier)


def _conv(conv, x, stride):
    """[B, Cin, T] -> [B, T', Cout]."""
    x = torch.nn.functional.pad(x, (1, 1)).unfold(2, 3, stride)  # B, Cin, T', 3
    x = x.permute(0, 2, 1, 3).reshape(x.shape[0], x.shape[2], -1)
    y = _mulh(_matmul(x, conv.weight.t().contiguous()) + conv.bias, _long(conv.req_multiplier))
    return _shr(y, _long(conv.req_shiftmount)).clamp(-127, 127)


def _exact_encode(case, s):
    enc = s["enc"]
    x = torch.round(s["mel"] * enc.input_alpha).clamp(-127, 127).long()
    x = _gelu(enc.gelu1, _conv(enc.conv1, x, 1)).transpose(1, 2)
    x = _gelu(enc.gelu2, _conv(enc.conv2, x, 2)) + _long(enc.positional_embedding)
    x = _shr(_wrap(x * _long(enc.req_multiplier)), _long(enc.req_shiftmount)).clamp(-16383, 16383)
    for b in enc.blocks:
        x = _block(b, x)
    return _ln(enc.ln_post, x)


class _Decoder:
    """The decoder over growing sequences of tokens, in 64 bits."""

    def __init__(self, dec, feats):
        self.dec, self.at, x = dec, 0, feats.long()
        self.own = [[] for _ in dec.blocks]
        self.cross = [(_linear(b.cross_attn.key, x), _linear(b.cross_attn.value, x)) for b in dec.blocks]

    def __call__(self, tokens):
        dec, T = self.dec, tokens.shape[1]
        x = dec.token_embedding.weight[tokens].long() + dec.positional_embedding[self.at:self.at + T]
        x = _shr(x * _long(dec.req_multiplier), _long(dec.req_shiftmount)).clamp(-16383, 16383)
        self.at += T
        for b, own, cross in zip(dec.blocks, self.own, self.cross):
            x = _block(b, x, own, cross)
        y = _mulh(_matmul(_ln(dec.ln, x), dec.token_embedding.weight.t().contiguous()), _long(dec.clf_req_multiplier))
        return _shr(y, _long(dec.clf_req_shiftmount)).clamp(-127, 127)


def _exact_hooks(case, s):
    dec = s["model"].decoder
    step, alpha = _Decoder(dec, s["feats"]), dec.act_logits_alpha.double()
    y, picked = step(s["prompt"]), []
    for _ in range(case["steps"]):
        picked.append(torch.argmax(y[:, -1], -1, keepdim=True))
        y = step(picked[-1])
    return dict(tokens=torch.cat(picked, 1), logits=y / alpha)


def _masked(logits, tokens, begin, f):
    """The decoding filters on float64 logits [B, V], -inf where a token may not come."""
    ninf, tb = -math.inf, f.timestamp_begin
    first = tokens.shape[1] == begin
    x = logits.clone()
    x[:, list(f.suppress_tokens) + [f.no_timestamps] + (list(f.suppress_blank) if first else [])] = ninf
    for i in range(len(x)):
        seq = tokens[i, begin:].tolist()
        last = bool(seq) and seq[-1] >= tb
        before = len(seq) < 2 or seq[-2] >= tb
        if last:
            if before:
                x[i, tb:] = ninf
            else:
                x[i, :f.eot] = ninf
        stamps = [t for t in seq if t >= tb]
        if stamps:
            x[i, tb:stamps[-1] + (0 if last and not before else 1)] = ninf
    if first:
        x[:, :tb] = ninf
        x[:, tb + f.max_initial_timestamp_index + 1:] = ninf
    stamp = torch.logsumexp(x[:, tb:], 1) > x[:, :tb].amax(1)
    x[:, :tb] = x[:, :tb].masked_fill(stamp[:, None], ninf)
    return x


def _exact_decode(case, s):
    dec, tokens, f = s["model"].decoder, s["prompt"], s["filters"]
    step, alpha = _Decoder(dec, s["feats"]), dec.act_logits_alpha.double()
    total = torch.zeros(case["batch"], dtype=torch.float64, device=tokens.device)
    y = step(tokens)[:, -1]
    for i in range(case["steps"]):
        x = y / alpha
        if f is not None:
            x = _masked(x, tokens, case["tokens"], f)
        nxt = torch.argmax(x, -1)
        ended = (tokens[:, -1] == EOT) & torch.tensor(f is not None, device=tokens.device)
        total += torch.where(ended, torch.zeros_like(total), torch.log_softmax(x, -1).gather(1, nxt[:, None])[:, 0])
        nxt = torch.where(ended, torch.full_like(nxt, EOT), nxt)
        tokens = torch.cat([tokens, nxt[:, None]], 1)
        if i + 1 < case["steps"]:
            y = step(nxt[:, None])[:, -1]
    return dict(tokens=tokens, sum_logprobs=total, logits=y)


def _exact_logmel(case, s):
    n, mels = 512, case["n_mels"]
    a = s["audio"].double()
    window = torch.hann_window(n, dtype=torch.float64, device=a.device)
    frames = torch.nn.functional.pad(a[:, None], (n // 2, n // 2), mode="reflect")[:, 0].unfold(1, n, 160)[:, :-1]
    power = torch.fft.rfft(frames * window).abs().square()

    def mel_to_hz(m):  # Slaney's scale: linear below 1 kHz, logarithmic above
        return np.where(m >= 15.0, 1000.0 * np.exp(np.log(6.4) / 27.0 * (m - 15.0)), 200.0 / 3 * m)

    top = 15.0 + np.log(8.0) / (np.log(6.4) / 27.0)
    edge = mel_to_hz(np.linspace(0.0, top, mels + 2))
    f = np.linspace(0.0, 8000.0, 1 + n // 2)
    up = (f - edge[:-2, None]) / (edge[1:-1] - edge[:-2])[:, None]
    down = (edge[2:, None] - f) / (edge[2:] - edge[1:-1])[:, None]
    bank = np.maximum(0.0, np.minimum(up, down)) * (2.0 / (edge[2:] - edge[:-2]))[:, None]
    y = torch.log10((power @ torch.from_numpy(bank.T.copy()).to(a.device)).clamp_min(1e-10)).transpose(1, 2)
    y = torch.maximum(y, y.amax((1, 2), keepdim=True) - 8.0) / 4.0 + 1.0
    return y


_EXACT = dict(logmel=_exact_logmel, encode=_exact_encode, block=lambda case, s: _block(s["block"], s["x"]),
              logits=lambda case, s: _Decoder(s["model"].decoder, s["feats"])(s["prompt"]) /
              s["model"].decoder.act_logits_alpha.double(),
              hooks=_exact_hooks, decode=_exact_decode)
