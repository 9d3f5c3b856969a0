"""Which kernel variants the shapes of the GPU tests reach, worked out on the CPU
from the cost rules with the constants that stand in the sources, so that a
rule fitted anew cannot leave a variant without a test."""
import os
import re

import test_gpu_dense_tiles

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pyflamert_amd", "csrc", "rocm")
CUS = 256  # compute units of an MI355X


def up(a, b):
    return -(-a // b)


def test_dense_tiles():
    """Each tile: a K below its chunk, K of one chunk or a tail of several (three
    at least, so that both LDS buffers come round again), and whole chunks;
    rows of op(A) in 16-byte loads and in single ones."""
    text = open(os.path.join(SRC, "dense.hip")).read()
    costs = re.findall(r"cost\((\d+), (\d+), (\d+), \{(\d+), (\d+), (\d+), (\d+)\}\)", text)
    assert len(costs) == 4
    tiles = [tuple(map(int, c)) for c in costs]

    def tile(M, K, N):
        def cost(t):
            n = up(up(M, t[0]) * up(N, t[1]), CUS)
            return n * t[2] + K * (n // 4 * t[6] + (t[3 + n % 4 - 1] if n % 4 else 0))
        return min(reversed(tiles), key=cost)  # the larger tile where two are equal

    reached = set()
    for M, K, N in test_gpu_dense_tiles.SHAPES:
        t = tile(M, K, N)
        chunk = 64 if t[0] == 32 else 32
        form = "short" if K < chunk else ("tail" if K % chunk else "whole") if K > 2 * chunk else "two"
        reached |= {(t[:2], form), (t[:2], "vector" if K % 4 == 0 and K > chunk else "single")}
    for t in tiles:
        for form in ("tail", "whole", "vector", "single"):
            assert (t[:2], form) in reached, (t[:2], form)
        # (a K below 32 never pays on 128 x 64 outputs)
        assert t[0] == 128 or (t[:2], "short") in reached, t[:2]
