"""Edges of the attention kernels' dispatch (rw_attn.hpp, run_attention): at
most 8 query rows, or 64 against over 384 keys of their own (k_attn), 9 to 64
rows (k_attn_tile splitting K and V itself), more (from split blocks), 32 or 64
query rows per workgroup; and scores that move the softmax's reference.

Bar: 1e-5 of the row's L2 norm against the float64 oracle (operands keep 22
bits, sums are f32: a few 2^-22 over scores of magnitude s, times s)."""
import numpy as np
import pytest

from oracle.attention import mha
from rusty_whisper_amd import _abi as A

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    A.init(0)


def err(got, q, k, v, heads, causal):
    ref = mha(q, k, v, heads, causal, dtype=np.float64)
    den = np.maximum(np.linalg.norm(ref, axis=1), 1e-30)
    return float(np.max(np.max(np.abs(got.astype(np.float64) - ref), axis=1) / den))


@pytest.mark.parametrize("t_q,t_kv,heads,causal", [
    (8, 33, 2, True), (9, 9, 2, True), (9, 31, 2, False), (32, 129, 1, True), (33, 33, 2, True), (64, 97, 2, True),
    (65, 65, 2, True), (65, 160, 3, False), (1030, 70, 24, False), (1030, 1030, 24, True), (9, 640, 2, True),
    (9, 641, 2, True), (33, 641, 3, False), (64, 1500, 2, True), (65, 1500, 2, False), (9, 384, 2, True),
    (9, 385, 2, True), (32, 385, 3, False), (33, 385, 3, False), (64, 1500, 20, False)], ids=str)
def test_dispatch_edges(t_q, t_kv, heads, causal):
    rng = np.random.default_rng(t_q + t_kv)
    q, k, v = (rng.standard_normal((t, 64 * heads)).astype(np.float32) for t in (t_q, t_kv, t_kv))
    assert err(A.attention(q, k, v, heads, causal), q, k, v, heads, causal) <= 1e-5


def test_rows_do_not_depend_on_the_tile():
    """One query row's result is the same bits from 64-row tiles, 32-row tiles
    and tiles that split K and V themselves."""
    rng = np.random.default_rng(3)
    q, k, v = (rng.standard_normal((t, 64 * 24)).astype(np.float32) for t in (1030, 300, 300))
    full = A.attention(q, k, v, 24, False)
    for t in (100, 64, 9):
        assert np.array_equal(A.attention(q[:t], k, v, 24, False).view(np.uint32), full[:t].view(np.uint32)), t


@pytest.mark.parametrize("t_q", [8, 40, 1030])
@pytest.mark.parametrize("step", [6.0, -6.0, 40.0])
def test_moving_maxima(t_q, step):
    """Scores that rise (or fall) so steeply that whatever came before a block (or
    comes after it) weighs nothing: rescale factors and weights of exactly 0."""
    heads, t_kv = 24, 140
    rng = np.random.default_rng(int(step) + t_q)
    q = np.zeros((t_q, 64 * heads), np.float32)
    k = (rng.standard_normal((t_kv, 64 * heads)) * 0.1).astype(np.float32)
    v = rng.standard_normal((t_kv, 64 * heads)).astype(np.float32)
    q[:, ::64] = 8.0  # score = the key's first value
    k[:, ::64] = (step * np.arange(t_kv, dtype=np.float32))[:, None]
    assert err(A.attention(q, k, v, heads, False), q, k, v, heads, False) <= 1e-5


@pytest.mark.parametrize("t_q", [8, 40, 100, 1030])
@pytest.mark.parametrize("step", [0.03, 0.06])
def test_rescales_that_matter(t_q, step):
    """Scores that rise by 4 or 8 nats over the 128 keys between a wavefront's
    blocks, in some query rows and not in others (12 blocks: two rescales each):
    what came before keeps a weight of 2^-6 or 2^-11, far above the bar."""
    heads, t_kv = 24, 384
    rng = np.random.default_rng(int(100 * step) + t_q)
    q = np.zeros((t_q, 64 * heads), np.float32)
    k = (rng.standard_normal((t_kv, 64 * heads)) * 0.1).astype(np.float32)
    v = rng.standard_normal((t_kv, 64 * heads)).astype(np.float32)
    slope = rng.choice(np.array([1.0, 0.9, 0.0, -1.0], np.float32), (t_q, heads))
    q[:, ::64] = 8.0 * slope  # score = slope x the key's first value
    k[:, ::64] = (step * np.arange(t_kv, dtype=np.float32))[:, None]
    assert err(A.attention(q, k, v, heads, False), q, k, v, heads, False) <= 1e-5


@pytest.mark.parametrize("t_q", [8, 40, 100, 1030])
@pytest.mark.parametrize("gap", [12, 16, 18, 20])
def test_mass_on_a_key_without_value(t_q, gap):
    """Rows whose probability sits on keys of value 0 (an attention sink), so
    that the output is made of the other keys' probabilities, 2^-gap of the
    row's largest.  P enters the products as f16 pairs of 2^12 or more at the
    maximum, in steps of 2^-24: an error of 2^-37 of the maximum per key,
    2^(gap - 37) of the others, and half of that over a row's norm leaves room
    for the sums (beside the 1e-6 of any row)."""
    heads, t_kv = 24, 320
    rng = np.random.default_rng(gap)
    q = np.zeros((t_q, 64 * heads), np.float32)
    k = np.zeros((t_kv, 64 * heads), np.float32)
    v = rng.standard_normal((t_kv, 64 * heads)).astype(np.float32)
    q[:, ::64] = 8.0  # score = the key's first value, exact in the f16 pairs
    k[:, ::64] = np.round(rng.uniform(-0.5, 0.5, (t_kv, heads)) * 1024) / 1024
    sinks = np.arange(0, 128, 32)  # one in each wavefront's first block
    k[sinks, ::64] = np.round(gap * np.log(2) * 256) / 256
    v[sinks] = 0.0
    got = A.attention(q, k, v, heads, False).astype(np.float64)
    ref = mha(q, k, v, heads, False, dtype=np.float64)
    rows = lambda x: x.reshape(t_q * heads, 64)  # noqa: E731  a head's row
    e = np.max(np.abs(rows(got - ref)), axis=1) / np.linalg.norm(rows(ref), axis=1)
    assert e.max() <= 1e-6 + 0.5 * 2.0 ** (gap - 37), e.max()


@pytest.mark.parametrize("t_q", [8, 40, 100, 1030])
@pytest.mark.parametrize("scale", [2048.0, 16384.0, 32768.0])
def test_scores_of_large_operands(t_q, scale):
    """q and k of +-scale (below the stated 65504): scores of up to 64 scale^2 / 8
    (8.6e9 at 32768), far beyond where log2(e) times one is known to a bit.  Every
    product and sum is exact, and a key that does not share the row's largest
    score is at least scale^2 / 4 below it, so each row is the mean of its best
    keys' values."""
    heads, t_kv = 24, 320
    rng = np.random.default_rng(int(scale))
    sign = lambda t: (rng.integers(0, 2, (t, 64 * heads)) * 2 - 1).astype(np.float32)  # noqa: E731
    q, k = sign(t_q) * np.float32(scale), sign(t_kv) * np.float32(scale)
    k[5::7] = k[:1]  # ties over blocks of every wavefront
    k[40:44, :] = q[:4]
    v = rng.standard_normal((t_kv, 64 * heads)).astype(np.float32)
    got = A.attention(q, k, v, heads, False)
    for hd in range(heads):
        c = slice(64 * hd, 64 * hd + 64)
        s = q[:, c].astype(np.float64) @ k[:, c].astype(np.float64).T
        best = s == s.max(axis=1, keepdims=True)
        ref = best @ v[:, c].astype(np.float64) / best.sum(axis=1, keepdims=True)
        assert np.max(np.max(np.abs(got[:, c] - ref), axis=1) / np.linalg.norm(ref, axis=1)) <= 1e-6, hd


@pytest.mark.parametrize("t_q", [40, 100, 1030])
def test_rows_of_little_spread(t_q):
    """Near-equal scores, whose row is a mean that cancels: what is random in each
    probability stays in it undivided.  The operands' 22 bits (2^-23 at most, 7e-8
    rms), the output's rounding (4e-8) and a few sums of that size leave 1.2e-7 of
    the rows' norm; an exponent rounded near 12 instead of near 0 added 1.9e-7
    (2^-21 / sqrt(3) times ln 2)."""
    heads, t_kv = 24, 100
    rng = np.random.default_rng(t_q)
    q, k, v = (rng.standard_normal((t, 64 * heads)).astype(np.float32) for t in (t_q, t_kv, t_kv))
    q *= np.float32(0.1)
    k *= np.float32(0.1)
    ref = mha(q, k, v, heads, False, dtype=np.float64)
    got = A.attention(q, k, v, heads, False).astype(np.float64)
    assert np.linalg.norm(got - ref) <= 1.7e-7 * np.linalg.norm(ref)
