"""Token ids passed by value (at most 8) and copied (more), and the final
layernorm's rows in registers (at most 2048 values) and beyond: the decoder's
4e-3 bar against the oracle (test_gpu_decoder.py)."""
import numpy as np
import pytest

from oracle.decoder import Decoder as OD
from _decoder_params import decoder_params
from test_gpu_decoder import device_decoder, rel, step, torch  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [64, 2048, 2112])
@pytest.mark.parametrize("tokens", [1, 8, 9])
def test_prompt_lengths(torch, n, tokens):  # noqa: F811
    p = decoder_params(n=n, f=256, n_layer=1, n_vocab=90, n_ctx=24, dtype=3, seed=n + tokens)
    enc = np.random.default_rng(n).standard_normal((20, n)).astype(np.float32)
    d = device_decoder(torch, p, n // 64, 20)
    d.set_audio(torch.from_numpy(enc).to("cuda:0"))
    o = OD(p, n // 64, enc)
    for toks in (list(range(80, 80 - tokens, -1)), [89], list(range(tokens))):
        assert rel(step(torch, d, toks, n), o.forward_hidden(toks)) <= 4e-3
