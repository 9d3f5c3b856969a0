"""Which kernel variants the shapes of the GPU tests reach, worked out on the CPU
from the cost rules with the constants that stand in the sources, so that a
rule fitted anew cannot leave a variant without a test."""
import os
import re

import test_gpu_dense_tiles
import test_gpu_sp24_small

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


def small_tile_rule():
    """plan_small of sp24.hip (activation rows N elements apart, output rows too),
    with its table from the source; the lines restated here must stand there."""
    text = open(os.path.join(SRC, "sp24.hip")).read()
    table = re.search(r"kSmallTiles\[\] = \{(.*?)\};", text, re.S).group(1)
    tiles = [tuple(map(int, t.split(","))) for t in re.findall(r"\{([\d, ]+)\}", table)]
    assert len(tiles) == 5
    for line in ("const double slow = 1 + (bf ? 0.1 : 0.25) * std::max(0.0, spill);",
                 "const double step = in_place && t.nb == 4 ? (bf && per_cu == 2 ? 140 : 170) : t.step;",
                 "const double rounds = full > 1 ? 0.75 * (double)full + 0.25 * (double)tiles / ctx->num_cu : 1;",
                 "std::min<int64_t>(380 + 9 * busy / 2, 600)", "(xrow ? 430 + 7 * busy / 10 : 500 + 14 * busy / 10)",
                 "const double scale = W->dtype == PFR_I8 && !xrow && whole ? 0.85 : 1;",
                 "const int64_t start = W->dtype == PFR_BF16 ? 6000 : 5000;",
                 "return start + (u8 ? 3000 : 0) + (int64_t)(rounds * (double)(steps * step) * scale);",
                 "return 4000 + bytes / 5000;"):
        assert line in text, line

    def small(M, K, N, size, in_place):
        slow = 1 + (0.1 if size == 2 else 0.25) * max(0.0, K * N * size / (4 << 20) - 1)
        steps, best = up(K, 128 // size), None
        for i, (rb, nb, _, start, each, step) in enumerate(tiles):
            if in_place and nb < 4 and 16 * nb < N:
                continue
            n = up(up(M, 16 * rb) * up(N, 16 * nb), CUS)
            if in_place and nb == 4:
                step = 140 if size == 2 and n == 2 else 170
            t = start + n * (each + int(steps * step * slow))
            if best is None or t < best[0]:
                best = (t, i)
        return best

    def large(M, K, N, size, xrow, u8, whole):
        tile_rows = up(M, 256) * up(N, 128)
        full, busy = up(tile_rows, CUS), min(tile_rows, CUS)
        rounds = 0.75 * full + 0.25 * tile_rows / CUS if full > 1 else 1
        step = min(380 + 9 * busy // 2, 600) if size == 2 else 430 + 7 * busy // 10 if xrow else 500 + 14 * busy // 10
        scale = 0.85 if size == 1 and not xrow and whole else 1
        pad = 512 if size == 1 else 256
        steps = up(K, pad) * pad // (128 // size)
        return (6000 if size == 2 else 5000) + (3000 if u8 else 0) + int(rounds * (steps * step) * scale)

    def plan(M, K, N, size, u8, pieces):
        """(tile or None, read in place); pieces: rows of whole, aligned 16-byte pieces."""
        pad = 512 if size == 1 else 256
        xrow = K % pad == 0 and N % 128 == 0 and (u8 or pieces)
        transpose = 4000 + K * N * size // 5000
        best, p = large(M, K, N, size, xrow, u8, pieces) + (0 if xrow else transpose), (None, False)
        if not xrow and small(M, K, N, size, False)[0] + transpose < best:
            t, i = small(M, K, N, size, False)
            best, p = t + transpose, (i, False)
        if pieces and small(M, K, N, size, True)[0] < best:
            p = (small(M, K, N, size, True)[1], True)
        return p

    def plan_qt(M, K, T):
        t, i = small(M, K, T, 1, False)
        return i if t < large(M, K, T, 1, False, False, False) + 8000 + T * K // 5000 + 4 * M * T // 5000 else None

    return plan, plan_qt


def test_small_tile_24():
    """Each tile of the small-tile 2:4 kernel with the activation transposed and read
    in place, for int8, uint8 and bf16, and in the x.W form with the rows of X
    themselves and padded; in place also with k rows that are no whole step."""
    plan, plan_qt = small_tile_rule()
    reached = set()
    for M, K, N in test_gpu_sp24_small.SHAPES:
        reached.add(("i8", *plan(M, K, N, 1, False, N % 16 == 0)))
        reached.add(("u8", *plan(M, K, N, 1, True, N % 16 == 0)))
        reached.add(("u8", *plan(M, K, N, 1, True, False)))  # inside wider rows
        reached.add(("bf16", *plan(M, K, N, 2, False, N % 8 == 0)))
        for kind, size, p in (("i8", 1, N % 16 == 0), ("bf16", 2, N % 8 == 0)):
            if plan(M, K, N, size, False, p)[1] and K % (128 // size):
                reached.add((kind, "ragged k in place"))
        reached.add(("x.W", plan_qt(M, K, N), K >= 16 and K % 16 == 0))  # ldx = K
    for tile in range(5):
        for kind in ("i8", "u8", "bf16", "x.W"):
            for in_place in (False, True):
                assert (kind, tile, in_place) in reached, (kind, tile, in_place)
    assert {("i8", "ragged k in place"), ("bf16", "ragged k in place")} <= reached
