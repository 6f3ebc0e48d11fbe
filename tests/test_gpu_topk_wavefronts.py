"""log_softmax + top-k where the candidates fall unevenly over the wavefronts
that pick them: all in one wavefront's ids, one per thread column, rows of one
value to 64 chunks.  Bar: the reference scan's ids (oracle/decoder.py) on
logits whose log-probs keep their order; log-probs as test_gpu_beams.py."""
import numpy as np
import pytest

from test_gpu_beams import check_rows, device_topk, torch  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 256, 2047, 2048, 2049, 131072])
@pytest.mark.parametrize("k", [1, 7, 16])
def test_sizes(torch, n, k):  # noqa: F811
    rng = np.random.default_rng(n + k)
    logits = np.stack([rng.permutation(n) for _ in range(3)]).astype(np.float32) * np.float32(2.0 ** -10)
    ids, lps = device_topk(torch, logits, k)
    check_rows(logits, k, ids, lps)


@pytest.mark.parametrize("k", [5, 16])
def test_one_wavefront_holds_every_candidate(torch, k):  # noqa: F811
    n = 6000
    logits = np.full((3, n), -30.0, np.float32)
    logits[0, 64:128] = np.arange(64) * 0.25       # consecutive ids
    logits[1, 5::256] = np.arange(24)[:len(logits[1, 5::256])] * 0.5  # one thread of each chunk
    logits[2, 4096:4160] = 3.0                     # ties, beyond the first chunk
    ids, lps = device_topk(torch, logits, k)
    check_rows(logits, k, ids, lps)
