"""The tiles that gemm.hip and fmodel.hip pick for a shape, for tests that claim
to run each of them: the tables are read from the sources, the rules around
them are repeated here."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nutllm_amd",
                    "csrc")


def table(name, start):
    """[(rows / 16, columns / 16, factor)] of the GemmTile table after `start`."""
    text = open(os.path.join(CSRC, name)).read()
    text = text[text.index(start):]
    body = text[:text.index("};")]
    body = body[body.index("GemmTile tiles[]"):]
    return [(int(i), int(j), float(f))
            for i, j, f in re.findall(r"\{(\d), (\d), ([\d.]+), 0\}", body)]


def pick(tiles, m, k, n):
    """gemm_f32_pick: (ti, tj, tiles of the grid)."""
    best = None
    for ti, tj, factor in tiles:
        if n < tj:
            continue
        rows, cols = 16 * ti, 16 * tj
        count = -(-m // rows) * -(-n // cols)
        cycles = -(-count // 256) * (rows * cols * k / 128.0 * factor + 2000.0)
        if best is None or cycles < best[0]:
            best = cycles, ti, tj, count
    return best[1:]


def matmul_form(m, k, n):
    """(ti, tj, waves, accumulators) of matmul_f32's launch."""
    wide = 4 if n > 32 else 2 if n > 16 else 1
    if k < 64 and -(-m // 64) * -(-n // (16 * wide)) >= 128:
        return 1, wide, 1, 2
    ti, tj, count = pick(table("gemm_f32.hpp", "gemm_f32_choose(int m"), m, k, n)
    deep = k >= 256
    if (ti, tj) == (4, 4):
        if (m // 64) * (n // 64) >= 256:
            return 4, 4, 4, 1
        return (4, 4, 8, 1) if deep else (4, 4, 4, 2)
    if (ti, tj) == (2, 2):
        return 2, 2, 8 if deep and count <= 256 else 4, 2
    return ti, tj, 8 if (ti, tj) == (1, 1) else 4, 2


MATMUL_FORMS = {(4, 4, 4, 1), (4, 4, 8, 1), (4, 4, 4, 2), (3, 4, 4, 2), (3, 3, 4, 2), (2, 4, 4, 2),
                (2, 2, 8, 2), (2, 2, 4, 2), (1, 2, 4, 2), (1, 1, 8, 2), (1, 4, 1, 2), (1, 2, 1, 2),
                (1, 1, 1, 2)}


def fgemm_form(epilogue, m, k, n):
    """(ti, tj, waves, runs of k) of an fp32 model's projection; epilogue "qkv",
    "add" or "swiglu", n all columns of the launch (gate and up both)."""
    if m <= 16:
        if epilogue == "add":
            runs = min(4, 256 // -(-n // 32))
            if runs > 1 and k >= 4096:
                return 1, 2, 8, runs
            return (1, 2, 16, 1) if n >= 4096 else (1, 1, 16, 1)
        return (1, 4, 8, 1) if n >= 8192 else (1, 2, 16, 1)
    ti, tj, _ = pick(table("fmodel.hip", "template <int EPI> void launch_fgemm"), m, k, n)
    return ti, tj, 8 if (ti, tj) == (1, 2) else 4, 1
