"""Which attention kernel a call takes (attn_route, rusty_whisper_amd/csrc/
rw_attn.hpp), on the CPU: k_attn_tile, whose wavefronts each run a chain of a
quarter of the kv blocks, or k_attn, whose kv runs go to workgroups of their own
and are merged by a second launch.  Built with g++ (tests/native/attn_route.cpp)."""
import os
import shutil
import subprocess

import pytest

from rusty_whisper_amd import _abi as A

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "rusty_whisper_amd", "csrc")

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("route") / "attn_route")
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{CSRC}", os.path.join(HERE, "native", "attn_route.cpp"), "-o", exe],
                   check=True)

    def call(t_q, t_kv, n_head, presplit):
        r = subprocess.run([exe], input=f"{t_q} {t_kv} {n_head} {int(presplit)}\n", capture_output=True, text=True,
                           check=True, timeout=20)
        return tuple(int(x) for x in r.stdout.split())

    return call


# Microseconds, both kernels on one MI355X: (query rows, kv rows, heads, K and V
# split beforehand): k_attn_tile, k_attn with the runs it would take + merge
MEASURED = [
    (9, 256, 6, False, 7.2, 7.9), (32, 256, 20, False, 7.9, 9.0), (64, 256, 12, False, 7.8, 8.4),
    (9, 448, 6, False, 9.8, 8.1), (9, 448, 20, False, 10.1, 8.2), (16, 640, 12, False, 11.9, 8.6),
    (32, 640, 20, False, 12.4, 10.8), (32, 1500, 6, False, 21.7, 9.8), (33, 768, 12, False, 13.7, 9.5),
    (48, 768, 16, False, 13.4, 10.4), (64, 768, 20, False, 14.0, 11.5), (64, 1500, 12, False, 22.1, 12.2),
    (64, 1500, 20, False, 22.3, 13.9),
    (9, 320, 6, True, 5.4, 7.2), (32, 640, 12, True, 7.2, 8.6), (64, 768, 20, True, 8.0, 11.2),
    (9, 1500, 6, True, 11.3, 8.3), (16, 1500, 12, True, 11.6, 10.4), (32, 1500, 6, True, 12.2, 9.2),
    (9, 1500, 20, True, 11.6, 9.6), (64, 1500, 6, True, 12.2, 9.4), (64, 1500, 12, True, 12.3, 11.5),
    (64, 1500, 20, True, 12.4, 12.9),
]


@pytest.mark.parametrize("t_q,t_kv,heads,presplit,tile,split", MEASURED, ids=str)
def test_takes_the_faster_kernel(route, t_q, t_kv, heads, presplit, tile, split):
    qt, rows, nsplit = route(t_q, t_kv, heads, presplit)
    assert rows == (not presplit)
    assert (qt == 1 and nsplit == 1) if tile < split else (qt == 0 and nsplit > 1)


@pytest.mark.parametrize("t_q,t_kv,heads,presplit,want", [
    # a decoding step's rows keep k_attn and its runs
    (1, 1, 6, False, (0, 1, 1)), (8, 224, 6, False, (0, 1, 1)), (8, 256, 6, False, (0, 1, 8)),
    (8, 1500, 20, True, (0, 0, 26)), (1, 1500, 6, True, (0, 0, 32)), (8, 1500, 256, True, (0, 0, 1)),
    # 9 to 64 rows, either side of each line
    (9, 384, 6, False, (1, 1, 1)), (9, 385, 6, False, (0, 1, 13)), (64, 384, 20, False, (1, 1, 1)),
    (64, 385, 20, False, (0, 1, 12)), (9, 1024, 20, True, (1, 0, 1)), (9, 1025, 20, True, (0, 0, 26)),
    (33, 1500, 12, True, (0, 0, 12)), (33, 1500, 13, True, (1, 0, 1)), (32, 1500, 24, True, (0, 0, 22)),
    # no runs to split into: too many heads
    (33, 1500, 256, False, (1, 1, 1)),
    # more rows: blocks, 64 rows per workgroup once those fill the chip
    (65, 1500, 6, False, (1, 0, 1)), (1500, 1500, 16, True, (2, 0, 1)), (1500, 1500, 15, True, (1, 0, 1)),
    (1024, 64, 24, False, (2, 0, 1)), (64, 64, 384, True, (2, 0, 1)), (64, 64, 384, False, (1, 1, 1)),
])
def test_lines(route, t_q, t_kv, heads, presplit, want):
    assert route(t_q, t_kv, heads, presplit) == want


@pytest.mark.parametrize("heads", [1, 6, 20, 300])
def test_workspace_holds_what_the_route_uses(route, heads):
    """K and v^T as operand blocks (16 KB per head and 32 keys), or the runs' partial
    results (64 rows of 64 values, a maximum and a sum per run and head)."""
    for t_q in (1, 8, 9, 32, 33, 64, 65, 1500):
        for t_kv in (1, 255, 256, 384, 385, 1500):
            qt, rows, nsplit = route(t_q, t_kv, heads, False)
            blocks = heads * ((t_kv + 31) // 32) * 16384 if qt and not rows else 0
            parts = nsplit * heads * 64 * 66 * 4 if nsplit > 1 else 0
            assert A.attention_workspace_size(t_q, t_kv, 64 * heads) >= blocks + parts, (t_q, t_kv)
