"""Edges of the dense tier's dispatch: 1 to 8 rows (one kernel per row count),
16 x 16 and 32 x 32 tiles, k around the pieces (32), rounds (128) and chunks
(512) of the few-row kernel, k without a main part, rows off 16 bytes, and
values past the end of a row that must not reach it.  Bar: bit for bit against
the oracle's restatement of tensor::matmul_t (src/tensor.rs:104-238)."""
import numpy as np
import pytest

import oracle as O
from rusty_whisper_amd import _abi as A

pytestmark = pytest.mark.gpu


def check(m, n, k, infinities=False):
    rng = np.random.default_rng(m * 7919 + n * 31 + k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((n, k)).astype(np.float32)
    if infinities:  # a row's own ends; the next row's start follows in memory
        b[::2, 0] = np.inf
        b[::2, -1] = -np.inf
        a[:, -1] = 0.0
        a[:, 0] = 1.0
    with np.errstate(invalid="ignore"):
        want = O.matmul_t_dense(a, b)
    got = A.matmul_t_f32(a, b)
    same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
    assert same.all(), (m, n, k, int((~same).sum()))


@pytest.mark.parametrize("m", range(1, 10))
def test_row_counts(m):
    check(m, 43, 328)


@pytest.mark.parametrize("k", [1, 4, 8, 12, 31, 32, 40, 127, 128, 132, 512, 516, 520, 1032])
@pytest.mark.parametrize("m", [1, 8, 17])
def test_k_edges(m, k):
    check(m, 21, k)
    check(m, 10, k, infinities=True)


@pytest.mark.parametrize("m,n,k", [(16, 16, 64), (33, 17, 36), (513, 1025, 44), (512, 1024, 7), (515, 1030, 33)], ids=str)
def test_tiles(m, n, k):
    check(m, n, k)
