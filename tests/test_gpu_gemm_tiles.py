"""Edges of the GEMM's tile choice and of the epilogues that write attention
operands (run_gemm's rules in rw_rocm.hip, GEMM_KOP / GEMM_VOP in
rw_kernels.hpp)."""
import numpy as np
import pytest

import oracle as O
from oracle.decoder import Decoder as OD
from oracle.encoder import encoder_layer
from rusty_whisper_amd import _abi as A
from _decoder_params import decoder_params
from test_gpu_decoder import device_decoder, rel, step, torch  # noqa: F401
from test_gpu_encoder_layer import build, rel_row

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [2, 7, 8])
@pytest.mark.parametrize("m", [3833, 3904, 2900, 1900])
def test_tile_choice_keeps_rows(torch, dtype, m):  # noqa: F811
    """3150 columns at k = 64 run 96 x 128 tiles at 3833 and 2900 rows (one round),
    128 x 64 at 3904, 96 x 64 at 1900, and 64-row tiles at 60; the same rows are
    the same bits in each, and within the matmul's 1e-3 of the oracle."""
    n, k = 3150, 64
    rng = np.random.default_rng(m + dtype)
    raw = O.quantize(dtype, (rng.standard_normal((n, k)) * 0.05).astype(np.float32))
    a, bias = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal(n).astype(np.float32)
    w = A.DeviceWeight(dtype, n, k, raw)
    full = w.matmul(a, bias)
    rows = np.r_[0:30, m - 30:m]
    assert np.array_equal(w.matmul(a[rows], bias).view(np.uint32), full[rows].view(np.uint32))
    ref = O.matmul_emul(a[rows], dtype, raw, n, bias=bias).astype(np.float64)
    assert np.max(np.abs(full[rows] - ref) / np.linalg.norm(ref, axis=1, keepdims=True)) <= 1e-3


@pytest.mark.parametrize("m", [3833, 1900])
def test_offset_rows_keep_64_column_tiles(torch, m):  # noqa: F811
    """Rows with a dominating minimum (an offset in the epilogue) at sizes where the
    rule would take 96 x 128 and 96 x 64 tiles without them."""
    n, k = 3150, 64
    rng = np.random.default_rng(m)
    x = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    x[::3] = 60000.0 + 6000.0 * rng.random((len(x[::3]), k))
    raw = O.quantize(7, x)
    a, bias = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal(n).astype(np.float32)
    w = A.DeviceWeight(7, n, k, raw)
    full = w.matmul(a, bias)
    rows = np.r_[0:30, m - 30:m]
    assert np.array_equal(w.matmul(a[rows], bias).view(np.uint32), full[rows].view(np.uint32))
    ref = O.matmul_emul(a[rows], 7, raw, n, bias=bias).astype(np.float64)
    assert np.max(np.abs(full[rows] - ref) / np.linalg.norm(ref, axis=1, keepdims=True)) <= 1e-3


def test_wide_tiles_with_gelu(torch, monkeypatch):  # noqa: F811
    """fc1 [5120, 64] over 2000 rows takes 96 x 128 tiles.  GELU and quantization in
    their epilogue: the operand's rows are those of a 60-row call (64-row tiles),
    bit for bit after fc2.  GELU alone, as the encoder layer runs it: the layer
    gives the same bits with fc1's epilogue quantizing and without."""
    t, n, f = 2000, 64, 5120
    p, dev = build(torch, n, f, 7, seed=3)
    x = np.random.default_rng(t).standard_normal((t, n)).astype(np.float32)

    def mlp(rows):
        m = len(rows)
        xd = torch.from_numpy(np.ascontiguousarray(rows)).to("cuda:0")
        ws = torch.empty(A.workspace_size(m, n), dtype=torch.uint8, device="cuda:0")
        A.quantize_dev(xd, m, n, ws, ws.numel())
        nxt = torch.empty(A.gelu_quantize_workspace_size(m, f), dtype=torch.uint8, device="cuda:0")
        A.matmul_prequant_gelu_quantize_dev(dev["fc1"], ws, m, dev["fc1_b"], nxt, nxt.numel())
        out = torch.empty(m, n, device="cuda:0")
        dev["fc2"].matmul_prequant_dev(nxt, m, out, dev["fc2_b"])
        torch.cuda.synchronize()
        return out.cpu().numpy()

    at = np.r_[0:30, t - 30:t]
    full = mlp(x)
    assert np.isfinite(full).all()
    assert np.array_equal(mlp(x[at]).view(np.uint32), full[at].view(np.uint32))
    outs = []
    for fused in (False, True):
        if fused:
            monkeypatch.setenv("RW_ENCODER_MLP", "fused")
        xd = torch.from_numpy(x).to("cuda:0")
        A.EncoderLayer(1, **dev).run(xd, t)
        torch.cuda.synchronize()
        outs.append(xd.cpu().numpy())
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))


def test_wide_tiles_with_residual(torch):  # noqa: F811
    """2816 tokens of a 3072-wide decoder: out and cross-out add to the residual
    stream from 96 x 128 tiles, where two halves of 1408 run 96 x 64; rows do not
    depend on the tile, so the hidden states are the same bits."""
    n, t = 3072, 2816
    p = decoder_params(n=n, f=64, n_layer=1, n_vocab=64, n_ctx=t, dtype=8, seed=5)
    enc = torch.from_numpy(np.random.default_rng(1).standard_normal((16, n)).astype(np.float32)).to("cuda:0")
    toks = np.arange(t) * 13 % 64
    d = device_decoder(torch, p, n // 64, 16)
    d.set_audio(enc)
    full = step(torch, d, toks, n)
    d.reset()
    halves = [step(torch, d, toks[:t // 2], n), step(torch, d, toks[t // 2:], n)]
    assert np.isfinite(full).all()
    assert np.array_equal(full.view(np.uint32), np.concatenate(halves).view(np.uint32))


@pytest.mark.parametrize("t,n", [(9, 64), (31, 128), (32, 128), (33, 192), (97, 1024), (640, 1024)], ids=str)
def test_encoder_layer_attention_operands(torch, t, n):  # noqa: F811
    """Rows around the 32-row blocks, one head up, k-split and single-wavefront
    launches: the encoder layer's bars (test_gpu_encoder_layer.py)."""
    p, dev = build(torch, n, 2 * n, 6, seed=t + n)
    x = np.random.default_rng(t).standard_normal((t, n)).astype(np.float32)
    xd = torch.from_numpy(x).to("cuda:0")
    A.EncoderLayer(n // 64, **dev).run(xd, t)
    torch.cuda.synchronize()
    got, ref = xd.cpu().numpy(), encoder_layer(x, p, n // 64)
    assert rel_row(got, ref) <= 2e-3
    assert rel_row(got - x, ref - x) <= 3e-3


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n_audio", [8, 9, 33, 64])
def test_cross_attention_operands(torch, n_audio, mixed):  # noqa: F811
    """The window's K and V from 8 rows (f32 rows, then split) and more (written
    by the products, one launch or one each), against the decoder's 4e-3 bar."""
    n, heads = 192, 3
    p = decoder_params(n=n, f=2 * n, n_layer=1, n_vocab=100, n_ctx=16, dtype=8, seed=n_audio,
                       dtypes={"cv": 7} if mixed else None)
    enc = np.random.default_rng(n_audio).standard_normal((n_audio, n)).astype(np.float32)
    d = device_decoder(torch, p, heads, n_audio)
    d.set_audio(torch.from_numpy(enc).to("cuda:0"))
    o = OD(p, heads, enc)
    for toks in ([1, 2, 3], [4], list(range(9))):
        assert rel(step(torch, d, toks, n), o.forward_hidden(toks)) <= 4e-3


@pytest.mark.parametrize("tokens", [9, 33, 64])
@pytest.mark.parametrize("n_audio", [1024, 1025, 1500])
def test_cross_attention_of_short_prompts(torch, n_audio, tokens):  # noqa: F811
    """Prompts of 9 to 64 tokens against a window whose kept blocks they read in one
    chain per wavefront (up to 1024 rows) or in runs, against the decoder's bar."""
    n, heads = 128, 2
    p = decoder_params(n=n, f=2 * n, n_layer=1, n_vocab=100, n_ctx=80, dtype=8, seed=n_audio + tokens)
    enc = np.random.default_rng(n_audio).standard_normal((n_audio, n)).astype(np.float32)
    d = device_decoder(torch, p, heads, n_audio)
    d.set_audio(torch.from_numpy(enc).to("cuda:0"))
    o = OD(p, heads, enc)
    for toks in ([t % 100 for t in range(tokens)], [4]):
        assert rel(step(torch, d, toks, n), o.forward_hidden(toks)) <= 4e-3
