"""Shape and dtype checks of the batched runners, before any device work: a
mel batch, audio features or a prompt that do not match the runner's batch
and sizes raise ValueError instead of reading or writing past the runner's
buffers."""
from types import SimpleNamespace

import pytest
import torch


def enc_stub():
    return SimpleNamespace(B=4, T=1500, enc=SimpleNamespace(n_mels=80))


def dec_stub(filters=None):
    return SimpleNamespace(B=4, Ta=1500, C=384, Tcap=448, hist_cols=448, filters=filters,
                           dec=SimpleNamespace(n_ctx=448, n_vocab=51865))


@pytest.mark.parametrize("shape,dtype", [((3, 80, 3000), torch.float32), ((5, 80, 3000), torch.float32),
                                         ((4, 128, 3000), torch.float32), ((4, 80, 2000), torch.float32),
                                         ((4, 80, 3000), torch.float16)])
def test_encoder_runner_rejects_mismatched_mel(iw, shape, dtype):
    with pytest.raises(ValueError):
        iw.EncoderRunner.__call__(enc_stub(), torch.zeros(shape, dtype=dtype))


@pytest.mark.parametrize("shape,dtype", [((3, 1500, 384), torch.int8), ((8, 1500, 384), torch.int8),
                                         ((4, 1000, 384), torch.int8), ((4, 1500, 512), torch.int8),
                                         ((4, 1500, 384), torch.int16)])
def test_decoder_runner_rejects_mismatched_audio(iw, shape, dtype):
    with pytest.raises(ValueError):
        iw.DecoderRunner.set_audio(dec_stub(), torch.zeros(shape, dtype=dtype))


def test_decoder_runner_rejects_cpu_audio(iw):
    with pytest.raises(ValueError, match="GPU"):
        iw.DecoderRunner.set_audio(dec_stub(), torch.zeros((4, 1500, 384), dtype=torch.int8))


@pytest.mark.parametrize("shape,steps", [((3, 3), 5), ((4,), 5), ((4, 0), 5), ((4, 3), 0), ((4, 3), 446)])
def test_decoder_runner_rejects_bad_prompt(iw, shape, steps):
    with pytest.raises(ValueError):
        iw.DecoderRunner.run(dec_stub(), torch.zeros(shape, dtype=torch.int64), steps)


def test_greedy_decode_rejects_runner_with_other_filters(iw):
    runner = dec_stub(filters=iw.LogitFilters(eot=50257))
    model = SimpleNamespace(decoder=SimpleNamespace(n_ctx=448, n_vocab=51865))
    prompt = torch.zeros((4, 3), dtype=torch.int64)
    with pytest.raises(ValueError, match="filters"):
        iw.greedy_decode(model, torch.zeros((4, 1500, 384), dtype=torch.int8), prompt, 5, runner=runner)


@pytest.mark.parametrize("tokens,error", [([1.0, float("nan")], ValueError), ([float("inf"), 1.0], OverflowError),
                                          ([float("-inf"), 1.0], OverflowError), ([1, 100], RuntimeError),
                                          ([-1, 5], RuntimeError), ([0.5, -1.0], RuntimeError),
                                          ([0, 99], None), ([True, False], None), ([-0.5, 99.5], None)])
def test_decoder_forward_checks_tokens(iw, tokens, error):
    """Values that are no token of the vocabulary are refused before the embedding gather reads a
    row of the table for them; those that convert to one are passed on."""
    class Reached(Exception):
        pass

    def embed(*args):
        raise Reached

    dec = SimpleNamespace(backend="hip", n_vocab=100, embed=embed)
    with pytest.raises(error or Reached):
        iw.TextDecoder_int.forward(dec, torch.tensor([tokens]), None)


@pytest.mark.parametrize("how", ["subclass", "instance", "class"])
def test_decoder_forward_calls_an_overridden_classify(iw, monkeypatch, how):
    """forward divides what classify returns, also where a program has put its own in its place."""
    def classify(self, h):
        return torch.full((*h.shape[:2], self.n_vocab), 7, dtype=torch.int8)

    cls = iw.TextDecoder_int
    if how == "subclass":
        cls = type("Decoder", (cls,), {"classify": classify})
    elif how == "class":
        monkeypatch.setattr(cls, "classify", classify)
    dec = cls(n_vocab=20, n_ctx=8, n_state=384, n_head=6, n_layer=0)
    if how == "instance":
        dec.classify = lambda h: classify(dec, h)
    dec.embed = lambda x, offset: torch.zeros((*x.shape, 384), dtype=torch.int16)
    dec.ln.normalize = lambda x: x.to(torch.int8)
    dec.act_logits_alpha.data.fill_(2.0)
    assert torch.equal(dec(torch.tensor([[1, 2, 3]]), None), torch.full((1, 3, 20), 3.5))
