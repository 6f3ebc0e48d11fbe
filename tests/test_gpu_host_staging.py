"""Host-pointer results around the pinned staging's sizes (2 MB threshold, 1 MB
chunks, 4 slots): the bits of the device entry, on first and repeated calls and
from several threads."""
import threading

import numpy as np
import pytest

import oracle as O
from rusty_whisper_amd import _abi as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1023, 1024, 1025, 2048, 2561, 3000])
def test_sizes_match_the_device_entry(m):
    import torch

    A.init(0)
    n, k = 512, 32  # 2 KB per row: 2 MB at 1024 rows, 5 MB + 2 KB at 2561
    rng = np.random.default_rng(m)
    w = A.DeviceWeight(8, n, k, O.quantize(8, rng.standard_normal((n, k)).astype(np.float32)))
    a = rng.standard_normal((m, k)).astype(np.float32)
    da, out = torch.from_numpy(a).to("cuda:0"), torch.empty(m, n, device="cuda:0")
    w.matmul_dev(da, m, out)
    torch.cuda.synchronize()
    want = out.cpu().numpy()
    assert np.array_equal(w.matmul(a).view(np.uint32), want.view(np.uint32))
    got = [None] * 4

    def call(i):
        got[i] = w.matmul(a[::-1] if i % 2 else a)

    threads = [threading.Thread(target=call, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i, g in enumerate(got):
        assert np.array_equal(g.view(np.uint32), (want[::-1] if i % 2 else want).view(np.uint32)), i
