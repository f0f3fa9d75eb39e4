"""The K-sliced f32-class GEMM at the edges of its tile forms.

Plain-row weights through the `linear` operator and fragment-major weights
through `prefill_logits` with a separate head; the two layouts run the same
sums, so their results are compared bit for bit.
"""
import numpy as np
import pytest

from conftest import bf16, bf16f, rng

pytestmark = pytest.mark.gpu

# 8 K slices below 2048 columns from K = 512 on, else 4; fewer K-steps than slices;
# partial row and column tiles (every form: EPILOGUE and ALIKE below)
SHAPES = [(1, 64, 32), (16, 1023, 512), (33, 2047, 96), (129, 1000, 2048), (600, 96, 1024), (2100, 1030, 64),
          (15, 2048, 32), (40, 2050, 160), (300, 2303, 1024), (1500, 2049, 64), (700, 6150, 96), (404, 6144, 64), (390, 2690, 96),
          (1300, 1030, 96), (790, 900, 160), (200, 2700, 64), (1300, 4100, 32)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_linear_slices(dev, M, N, K):
    from qwenasr_amd import kernels as Kr
    print(f"linear slices M={M} N={N} K={K}", flush=True)
    r = rng(M * 7 + N * 3 + K)
    x = r.normal(0, 1, (M, K)).astype(np.float32)
    w = bf16(r.normal(0, 0.02, (N, K)))
    dx, dw = dev.upload(x), dev.upload(w)
    y = dev.zeros((M + 1, N), np.float32)
    Kr.linear(y, dx, dw, None, M, K, N)
    got = y.numpy()
    xd, wd = x.astype(np.float64), bf16f(w).astype(np.float64)
    exact = xd @ wd.T
    # K roundings of partial sums no larger than sum |x w|, each at most 2^-24
    bound = K * 2.0 ** -24 * (np.abs(xd) @ np.abs(wd).T) + 1e-30
    assert (np.abs(got[:M] - exact) <= bound).all()
    assert (got[M] == 0).all()                       # nothing past the last row
    # a row's bits do not depend on how many rows share the call
    y1 = dev.empty((1, N), np.float32)
    Kr.linear(y1, dev.upload(x[M - 1:]), dw, None, 1, K, N)
    assert (y1.numpy()[0] == got[M - 1]).all()


@pytest.mark.parametrize("hidden,inter,vocab,rows", [(64, 64, 33, 1), (192, 320, 1003, 17), (1024, 448, 2050, 70),
                                                     (256, 192, 2047, 300), (64, 128, 6144, 404), (64, 64, 2690, 390),
                                                     (64, 64, 2700, 200), (64, 64, 4100, 500)])
def test_fragment_major_head(dev, hidden, inter, vocab, rows):
    """A separate head equal to the tied embedding (plain rows) gives its bits."""
    from qwenasr_amd.model import Decoder
    from qwenasr_amd.synth import SynthDecoder
    print(f"head layouts hidden={hidden} vocab={vocab} rows={rows}", flush=True)
    cfg = dict(n_layers=1, hidden=hidden, n_heads=16, n_kv_heads=8, head_dim=128, intermediate=inter, vocab=vocab,
               eps=1e-6, theta=1e6)
    w = SynthDecoder(cfg, seed=77)
    d = Decoder(dev, w, max_seq=512)
    emb = rng(rows).normal(0, 0.05, (rows, hidden)).astype(np.float32)
    tied = d.prefill_logits(emb)
    d.kv_len = 0
    d.set_lm_head(w.embed)
    own = d.prefill_logits(emb)
    d.close()
    assert np.isfinite(tied).all() and (tied == own).all()


# the ring of 128 x 128 tiles that plain rows take with many tiles: partial row and
# column tiles, vector (N % 4 == 0) and scalar stores, one to 32 K-steps
RING = [(4000, 2003, 32), (4000, 2004, 96), (1600, 4100, 1024), (8190, 1022, 512)]


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("M,N,K", RING)
def test_linear_ring(dev, M, N, K, accumulate):
    from qwenasr_amd import kernels as Kr
    print(f"linear ring M={M} N={N} K={K} accumulate={accumulate}", flush=True)
    r = rng(M * 7 + N * 3 + K)
    x = r.normal(0, 1, (M, K)).astype(np.float32)
    w = bf16(r.normal(0, 0.02, (N, K)))
    b = r.normal(0, 1, N).astype(np.float32)
    y0 = np.zeros((M + 1, N), np.float32)
    if accumulate:
        y0[:M] = r.normal(0, 1, (M, N))
    y = dev.upload(y0)
    Kr.linear(y, dev.upload(x), dev.upload(w), dev.upload(b), M, K, N, accumulate=accumulate)
    got = y.numpy()
    xd, wd = x.astype(np.float64), bf16f(w).astype(np.float64)
    exact = xd @ wd.T + b + y0[:M]
    # K + 2 roundings of partial sums no larger than sum |x w| + |b| + |y0|, each at most 2^-24
    bound = (K + 2) * 2.0 ** -24 * (np.abs(xd) @ np.abs(wd).T + np.abs(b) + np.abs(y0[:M]))
    assert (np.abs(got[:M] - exact) <= bound).all()
    assert (got[M] == 0).all()                       # nothing past the last row


# bias and += in every plain-row form with partial rows and columns: 8 slices (K >=
# 512) in 16 x 32 ... 48 x 128 tiles, 4 slices in 16 x 64, 32 x 64, 64 x 64
# (test_gemm_forms.py holds the list to the dispatch's rule)
EPILOGUE = [(45, 1003, 544), (135, 1010, 512), (404, 1000, 544), (600, 1000, 512), (900, 900, 544), (1300, 1030, 512),
            (45, 2050, 544), (200, 2303, 96), (700, 2310, 160), (300, 1990, 96)]


@pytest.mark.parametrize("M,N,K", EPILOGUE)
def test_linear_epilogue(dev, M, N, K):
    test_linear_ring(dev, M, N, K, False)
    test_linear_ring(dev, M, N, K, True)


# hidden, intermediate, row counts: the += GEMMs (o_proj, K = 2048, and down) take
# every fragment-major form, 8 slices at 1024 columns, 4 at 2048
ALIKE = [(1024, 576, (70, 200, 300, 600, 800, 1100)), (2048, 1088, (70, 200, 300, 400, 520, 600, 700))]


@pytest.mark.parametrize("hidden,inter,rows", ALIKE)
def test_prefill_rows_alike(dev, orc, hidden, inter, rows):
    """The fewest rows against the oracle; more rows (other forms) give the first
    ones the same bits."""
    from qwenasr_amd.model import Decoder
    from qwenasr_amd.synth import SynthDecoder
    cfg = dict(n_layers=2, hidden=hidden, n_heads=16, n_kv_heads=8, head_dim=128, intermediate=inter, vocab=1000,
               eps=1e-6, theta=1e6)
    w = SynthDecoder(cfg, seed=78)
    d = Decoder(dev, w, max_seq=1280)
    emb = rng(hidden).normal(0, 0.02, (rows[-1], hidden)).astype(np.float32)
    logits, kv = {}, {}
    for n in rows:
        print(f"prefill rows alike hidden={hidden} rows={n}", flush=True)
        d.kv_len = 0
        logits[n] = d.prefill_logits(emb[:n])
        kv[n] = d.kv_rows_download(0, n)
    d.close()
    n0 = rows[0]
    cpu = orc.OracleDecoder(w, max_seq=256)
    want = cpu.prefill_logits(emb[:n0])
    kc, vc = cpu.kv()
    cpu.close()
    for got, ref in ((kv[n0][0], kc[:, :, :n0]), (kv[n0][1], vc[:, :, :n0])):
        assert np.linalg.norm(got - ref) <= 1e-5 * np.linalg.norm(ref)
    assert np.linalg.norm(logits[n0] - want) <= 2e-4 * np.linalg.norm(want)
    for a, b in zip(rows, rows[1:]):
        assert (logits[b][:a] == logits[a]).all(), (a, b)
        assert all((kv[b][i][:, :, :a] == kv[a][i]).all() for i in range(2)), (a, b)


# conv_hidden, whole chunks: conv2 (800 rows a chunk, conv_hidden columns) takes every
# convolution form
CONV = [(96, 1), (96, 2), (96, 4), (96, 6), (96, 11), (480, 3)]


@pytest.mark.parametrize("conv_hidden,chunks", CONV)
def test_conv_forms(dev, orc, conv_hidden, chunks):
    from qwenasr_amd.model import Encoder
    from qwenasr_amd.synth import SynthEncoder
    cfg = dict(d_model=64, n_layers=1, n_heads=1, head_dim=64, ffn_dim=128, output_dim=128, chunk_size=100,
               n_window_infer=800, conv_hidden=conv_hidden)
    print(f"conv forms conv_hidden={conv_hidden} chunks={chunks}", flush=True)
    w = SynthEncoder(cfg, seed=60 + conv_hidden)
    enc, ore = Encoder(dev, w), orc.OracleEncoder(w)
    mel = rng(chunks).normal(0, 0.5, (128, 100 * chunks + 37)).astype(np.float32)
    got, want = enc.forward(mel), ore.forward(mel)
    enc.close()
    ore.close()
    # f32-class sums of up to 4320 terms through four convolutions and a layer; measured 2e-7
    assert got.shape == want.shape
    assert (np.linalg.norm(got - want, axis=1) <= 1e-5 * np.linalg.norm(want, axis=1).max()).all()
