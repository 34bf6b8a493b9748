"""CPU address check of flash_duo_kernel (tests/duo_check.hip) over the shapes of
test_geometry.py and the edges of duo_plan's rules."""

import os
import shutil
import subprocess

import pytest
from test_geometry import line, run, shapes

HERE = os.path.dirname(os.path.abspath(__file__))

pytestmark = pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc is not on PATH")

# (batch, seq_q, seq_k, heads): each branch of duo_plan and both sides of its lines
EDGES = [(1, 300, 512, 3), (1, 300, 513, 3), (1, 130, 577, 3), (1, 384, 640, 85), (1, 384, 640, 86),  # 255, 258 items
         (1, 700, 700, 60), (1, 767, 767, 45), (1, 2112, 2112, 17), (3, 300, 300, 60), (1, 2050, 2050, 31),
         (1, 70, 4100, 3), (2, 500, 3000, 8), (1, 512, 2560, 21), (1, 512, 4096, 42), (1, 512, 6144, 17),
         (1, 700, 300, 50), (1, 1000, 2000, 40), (1, 1000, 1999, 40), (9, 50, 50, 130)]
# E = 128 calls on the 64-row kernel: (shape, causal, splits, pairs)
P64 = [((1, 6144, 6144, 11), True, 1, 1), ((1, 6150, 6200, 11), True, 1, 1), ((1, 250, 2570, 240), False, 1, 0),
       ((1, 250, 2570, 240), True, 1, 0), ((1, 500, 6150, 17), False, 7, 0), ((1, 500, 6150, 17), True, 7, 0)]


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("duo") / "duo_check")
    r = subprocess.run(["hipcc", "-x", "hip", "--offload-arch=gfx950", "-O1", "-std=c++17", "-w",
                        os.path.join(HERE, "duo_check.hip"), "-o", exe], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-3000:]
    return exe


def edges():
    return [line(e, True, causal, *s, lay) for e in (32, 64, 128) for causal in (False, True) for s in EDGES
            for lay in ("bshe", "bhse")]


def test_every_access_inside_its_tensor(checker):
    r = run(checker, shapes() + edges())
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout[-2000:] + r.stderr[-2000:]
    taken, accesses = map(int, r.stdout.split()[1:3])
    assert taken > 300 and accesses > 10 ** 7


def test_a_planted_window_mistake_is_caught(checker):
    r = run(checker, [line(64, True, True, 1, 257, 513, 8)], "--plant")
    assert r.returncode == 1 and "FAIL" in r.stdout, r.stdout


def test_calls_on_the_64_row_kernel(checker):
    """The shapes of test_flash_p64_gpu.py run what that test is about."""
    r = run(checker, [line(128, True, causal, *shape) for shape, causal, _, _ in P64], "--plans")
    assert r.stdout.splitlines() == [f"0 {splits} {pairs}" for _, _, splits, pairs in P64], r.stdout
    r = run(checker, [line(e, True, c, *s) for e in (32, 64) for s, c, _, _ in P64], "--plans")
    assert not any(x.startswith("0") for x in r.stdout.splitlines()), r.stdout
