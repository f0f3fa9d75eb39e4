"""The int8-weight GEMM at the edges of every tile form of its dispatch
(32 x 64 ... 160 x 128), rows and columns that are no multiple of a tile, and
K below and above a ring's stages."""
import numpy as np
import pytest

from conftest import bf16, bf16f, rng

pytestmark = pytest.mark.gpu

# by the dispatch's estimate: 32 x 64, 64 x 64, 64 x 128, 96 x 128, 128 x 128, 160 x 128
SHAPES = [(1, 3001, 64), (40, 4100, 192), (50, 20002, 64), (375, 4097, 320), (64, 151936, 64), (61, 60001, 128),
          (90, 60001, 64), (190, 30004, 128), (375, 20001, 64), (128, 40000, 192), (140, 60002, 64), (404, 10001, 128)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_w8_forms(dev, M, N, K):
    from qwenasr_amd import kernels as Kr
    print(f"w8 forms M={M} N={N} K={K}", flush=True)
    r = rng(M * 7 + N * 3 + K)
    a = bf16(r.normal(0, 1, (M, K)))
    w = r.integers(-127, 128, (N, K), dtype=np.int8)
    s = (r.uniform(0.05, 0.07, N) / 127).astype(np.float32)
    da, dw, ds = dev.upload(a), dev.upload(w), dev.upload(s)
    y = dev.zeros((M + 1, N), np.float32)
    Kr.gemm_w8_bf16(y, da, dw, ds, M, N, K)
    got = y.numpy()
    af, wf = bf16f(a).astype(np.float32), w.astype(np.float32)
    # both f32 sums: K roundings of partial sums no larger than sum |a w| each, and the scale's
    bound = (2 * K + 2) * 2.0 ** -24 * (np.abs(af) @ np.abs(wf).T) * s
    assert (np.abs(got[:M] - (af @ wf.T) * s) <= bound).all()
    assert (got[M] == 0).all()                       # nothing past the last row
    # the last row alone (another form, the same K-steps in the same order): the same bits
    y1 = dev.empty((1, N), np.float32)
    Kr.gemm_w8_bf16(y1, dev.upload(a[M - 1:]), dw, ds, 1, N, K)
    assert (y1.numpy()[0] == got[M - 1]).all()


# Every form with rows and columns that are no multiple of its tile, with vector and
# scalar stores, at short and long K: 32 x 64, 64 x 64, 64 x 128, 96 x 128, 128 x 128,
# 160 x 128, and the K groups (test_gemm_forms.py holds the list to the dispatch's
# rule)
EDGES = [(45, 3001, 576), (45, 4100, 576), (45, 10004, 576), (75, 8001, 512), (75, 8004, 512), (33, 151937, 512), (33, 151932, 512),
         (75, 20001, 576), (90, 20004, 576), (404, 8001, 512), (404, 8004, 512), (130, 20001, 576), (130, 20004, 576),
         (75, 2003, 1024), (75, 2004, 1088), (45, 3001, 64), (33, 20001, 192), (250, 8004, 64), (75, 30001, 128),
         (404, 8001, 64), (130, 20004, 64)]


@pytest.mark.parametrize("M,N,K", EDGES)
def test_w8_edges(dev, M, N, K):
    test_w8_forms(dev, M, N, K)
