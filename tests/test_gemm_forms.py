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
    """go_gemm_lds' choice: (rows, columns) of the tile, or "K groups"; 16-byte stores."""
    if up(N, 64) * up(M, 64) < 2048 and K // 64 >= 16 and up(N, 64) <= 32:
        return "K groups", N % 4 == 0
    src = source("k_gemm.hip")
    name = "shortk" if K < 512 else "longk"
    forms = rows_of(re.search(r"W8Form " + name + r"\[\] = \{(.*?)\};", src, re.S).group(1), 4)
    assert len(forms) == 6

    def cost(f):
        tiles = up(M, f[0]) * up(N, f[1])
        rounds = up(tiles, 256)
        return 512 * f[2] + (f[3] * (tiles + 256 * rounds - 512) if rounds > 1 else 0)
    f = min(forms, key=cost)[:2]
    one_round = up(M, f[0]) * up(N, f[1]) <= 256
    return f, N % 4 == 0 and (f == (64, 64) or one_round == (f[1] == 128))


def test_w8_shapes_reach_every_form():
    from test_gpu_w8_forms import EDGES
    seen = {}
    for M, N, K in EDGES:
        f, vec = w8_form(M, N, K)
        bm, bn = (64, 64) if f == "K groups" else f
        assert M % bm and N % bn, (M, N, f)          # partial rows and columns
        seen.setdefault(f, set()).add((K < 512, vec))
    tiles = [(32, 64), (64, 64), (64, 128), (96, 128), (128, 128), (160, 128)]
    for f in tiles + ["K groups"]:
        assert {v for _, v in seen[f]} == {False, True}, f
        assert {k for k, _ in seen[f]} == ({False} if f == "K groups" else {False, True}), f


def ks_tables():
    src = source("k_gemm_ks.hip")
    t = [rows_of(x, 3) for x in re.findall(r"static const KsForm f\[\] = \{(.*?)\};", src, re.S)]
    assert [len(x) for x in t] == [6, 7, 3, 6]       # rows: 8 slices; 4 slices fragment-major, plain; convolutions
    two, one = (int(v) for v in re.search(r"return rounds / 2 \* (\d+) \+ rounds % 2 \* (\d+);", src).groups())
    return t, two, one


def ks_form(M, N, K, frag, alike):
    """go_ks_rows' choice: (slices, rows, columns) or "ring"."""
    t, two, one = ks_tables()
    eight = N < 2048 and K >= 512
    forms = t[0] if eight else t[1] if frag else t[2]

    def cost(f):
        return up(up(M, f[0]) * up(N, f[1]), 256) * f[2]
    best = min(forms, key=cost)
    rounds = up(up(M, 128) * up(N, 128), 256)
    if not frag and not alike and rounds // 2 * two + rounds % 2 * one <= cost(best):
        return "ring"
    return (8 if eight else 4,) + best[:2]


def test_linear_shapes_reach_every_plain_form():
    from test_gpu_gemm_slices import EPILOGUE, RING
    t, _, _ = ks_tables()
    seen = set()
    for M, N, K in EPILOGUE:
        f = ks_form(M, N, K, False, False)
        assert M % f[1] and N % f[2], (M, N, K, f)   # partial rows and columns
        seen.add(f)
    assert seen == {(8,) + f[:2] for f in t[0]} | {(4,) + f[:2] for f in t[2]}
    assert all(ks_form(M, N, K, False, False) == "ring" and M % 128 and N % 128 for M, N, K in RING)


def test_prefill_shapes_reach_every_fragment_major_form():
    from test_gpu_gemm_slices import ALIKE
    t, _, _ = ks_tables()
    want = {1024: {(8,) + f[:2] for f in t[0]}, 2048: {(4,) + f[:2] for f in t[1]}}
    for hidden, inter, rows in ALIKE:
        # o_proj and down (+=) each reach every form of their width
        for K in (2048, inter):
            assert {ks_form(M, hidden, K, True, True) for M in rows} == want[hidden], (hidden, K)


def test_encoder_shapes_reach_every_convolution_form():
    from test_gpu_gemm_slices import CONV
    t, _, _ = ks_tables()
    forms = t[3]
    seen = {min(forms, key=lambda f: up(up(800 * k, f[0]) * up(C, f[1]), 256) * f[2]) for C, k in CONV}
    assert seen == set(forms)
