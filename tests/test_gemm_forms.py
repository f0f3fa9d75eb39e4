"""The tile forms that the GPU tests' shapes reach, by the dispatch's own rules.

The forms and their costs are read from the sources (k_gemm.hip, k_gemm_ks.hip)
and the rules restated here, so a change of a cost that leaves a form untested
fails on the CPU.
"""
import os
import re

from conftest import ROOT

CSRC = os.path.join(ROOT, "qwenasr_amd", "csrc")


def up(a, b):
    return -(-a // b)


def source(name):
    with open(os.path.join(CSRC, name)) as f:
        return f.read()


def rows_of(text, width):
    return [tuple(int(v) for v in r) for r in re.findall(r"\{" + ", ".join([r"(\d+)"] * width) + r"\}", text)]


def w8_form(M, N, K):
    """go_gemm_lds' choice: (rows, columns) of the tile, or "K groups"."""
    if up(N, 64) * up(M, 64) < 2048 and K // 64 >= 16 and up(N, 64) <= 32:
        return "K groups"
    src = source("k_gemm.hip")
    name = "shortk" if K < 512 else "longk"
    forms = rows_of(re.search(r"W8Form " + name + r"\[\] = \{(.*?)\};", src, re.S).group(1), 4)
    assert len(forms) == 6

    def cost(f):
        tiles = up(M, f[0]) * up(N, f[1])
        rounds = up(tiles, 256)
        return 512 * f[2] + (f[3] * (tiles + 256 * rounds - 512) if rounds > 1 else 0)
    return min(forms, key=cost)[:2]


def test_w8_shapes_reach_every_form():
    from test_gpu_w8_forms import EDGES
    seen = {}
    for M, N, K in EDGES:
        f = w8_form(M, N, K)
        vec = K >= 512 and N % 4 == 0
        bm, bn = (64, 64) if f == "K groups" else f
        assert M % bm and N % bn, (M, N, f)          # partial rows and columns
        seen.setdefault((f, K < 512), set()).add(vec)
    tiles = [(32, 64), (64, 64), (64, 128), (96, 128), (128, 128), (160, 128)]
    assert seen == {**{(t, False): {False, True} for t in tiles + ["K groups"]}, **{(t, True): {False} for t in tiles}}
