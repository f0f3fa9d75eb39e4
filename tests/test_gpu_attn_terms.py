"""The prefill attention on bf16 terms against float64, at the edges of its
16-row and 16-key tiles and of its two block forms (one or two query heads per
block, the same bits)."""
import numpy as np
import pytest

from conftest import rng

pytestmark = pytest.mark.gpu


def attend(q, k, v, past):
    out = np.empty_like(q, dtype=np.float64)
    n, m = q.shape[0], k.shape[1]
    seen = np.arange(m)[None] <= np.arange(n)[:, None] + past
    for h in range(q.shape[1]):
        s = (q[:, h].astype(np.float64) @ k[h // 2].astype(np.float64).T) * 128 ** -0.5
        s = np.where(seen, s, -np.inf)
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, h] = (p / p.sum(1, keepdims=True)) @ v[h // 2].astype(np.float64)
    return out


@pytest.mark.parametrize("n,past", [(2, 0), (16, 0), (17, 1), (33, 127), (128, 15), (130, 0), (255, 600), (768, 3)])
def test_causal_rows(dev, n, past):
    from qwenasr_amd import kernels as Kr
    print(f"causal rows n={n} past={past}", flush=True)
    r = rng(n * 31 + past)
    m = n + past
    cap = m + 5                                       # rows past the context must not be read into the result
    q = r.normal(0, 1, (n, 16, 128)).astype(np.float32)
    k, v = (np.full((8, cap, 128), np.nan, np.float32) for _ in range(2))
    k[:, :m] = r.normal(0, 1, (8, m, 128))
    v[:, :m] = r.normal(0, 0.6, (8, m, 128))
    dq, dk, dv, out = dev.upload(q), dev.upload(k), dev.upload(v), dev.empty((n, 16, 128), np.float32)
    Kr.causal_attention(out, dq, dk, dv, cap * 128, n, m, 16, 8, 128, 128 ** -0.5, past)
    got = out.numpy()
    ref = attend(q, k[:, :m], v[:, :m], past)
    # f32-class: a score's error is at most 128 2^-24 sum |q k| / sqrt(128) (about 1e-5
    # relative in its probability), averaged over the keys; measured 1e-7 - 3e-7
    assert np.linalg.norm(got - ref) <= 1e-6 * np.linalg.norm(ref)
    assert np.abs(got - ref).max() <= 2e-5
    # the last rows alone (other row tiles; at 768 rows the other block form): the same bits
    k0 = max(0, n - 20)
    part = dev.empty((n - k0, 16, 128), np.float32)
    Kr.causal_attention(part, dev.upload(q[k0:]), dk, dv, cap * 128, n - k0, m, 16, 8, 128, 128 ** -0.5, past + k0)
    assert (part.numpy() == got[k0:]).all()


@pytest.mark.parametrize("n,past", [(33, 127), (768, 3)])
def test_far_scores(dev, n, past):
    """Finite scores up to 2^128 apart (their difference past f32's range): the
    keys below the best get weight 0, whatever the gap."""
    from qwenasr_amd import kernels as Kr
    print(f"far scores n={n} past={past}", flush=True)
    r = rng(n + past)
    m = n + past
    q, k = np.zeros((n, 16, 128), np.float32), np.zeros((8, m, 128), np.float32)
    q[:, :, 5] = 2.0 ** 64
    # scores -2^127 ... 2^127, exact in f32: gaps 8.5e37, 1.7e38, 2.55e38 and 3.4e38
    k[:, :, 5] = r.choice([-(2.0 ** 63), -(2.0 ** 62), 0.0, 2.0 ** 62, 2.0 ** 63], (8, m), p=[0.3, 0.3, 0.3, 0.05, 0.05])
    v = r.normal(0, 0.6, (8, m, 128)).astype(np.float32)
    out = dev.empty((n, 16, 128), np.float32)
    Kr.causal_attention(out, dev.upload(q), dev.upload(k), dev.upload(v), m * 128, n, m, 16, 8, 128, 1.0, past)
    got = out.numpy()
    for i in range(n):
        for h in range(8):
            seen = k[h, :past + i + 1, 5]
            ref = v[h, :past + i + 1][seen == seen.max()].astype(np.float64).mean(0)
            # equal weights: the sums of at most m products of 2^-24 relative error each
            assert (np.abs(got[i, 2 * h:2 * h + 2] - ref) <= 1e-5).all(), (i, h)


@pytest.mark.parametrize("n,past", [(33, 127), (768, 3)])
@pytest.mark.parametrize("what", ["v_large", "v_inf", "k_large", "k_minus_inf"])
def test_values_without_terms(dev, n, past, what):
    """One key holds a value that has no three bf16 terms (infinite, or finite and
    rounding up to infinity): rows that see it are f32's, the others keep their bits."""
    from qwenasr_amd import kernels as Kr
    print(f"values without terms n={n} past={past} {what}", flush=True)
    r = rng(n + past)
    m, j0 = n + past, past + n // 2                    # seen by the rows from n // 2 on
    q = r.normal(0, 1, (n, 16, 128)).astype(np.float32)
    k, v = r.normal(0, 1, (8, m, 128)).astype(np.float32), r.normal(0, 0.6, (8, m, 128)).astype(np.float32)
    if what == "k_large":
        q[:, :, 9] = 1e-37
    if what == "k_minus_inf":
        q[:, :, 9] = np.abs(q[:, :, 9]) + 0.1

    def run():
        out = dev.empty((n, 16, 128), np.float32)
        Kr.causal_attention(out, dev.upload(q), dev.upload(k), dev.upload(v), m * 128, n, m, 16, 8, 128, 128 ** -0.5,
                            past)
        return out.numpy()

    plain = run()
    if what[0] == "v":
        v[2, j0, 9] = 3.4e38 if what == "v_large" else np.inf
    else:
        k[2, j0, 9] = 3.4e38 if what == "k_large" else -np.inf
    got = run()
    tile = j0 // 16 * 16                               # the first of its 16 keys
    before = np.arange(n) + past < tile
    assert (got[before] == plain[before]).all()
    other = [h for h in range(16) if h // 2 != 2]
    assert (got[:, other] == plain[:, other]).all()
    for i in range(n):
        end = past + i + 1
        if j0 >= end > tile and what == "v_inf":
            continue                                   # the tile's masked key: weight 0 times infinity
        for h in (4, 5):
            s = (k[2, :end].astype(np.float64) @ q[i, h].astype(np.float64)) * 128 ** -0.5
            p = np.exp(s - s.max())
            ref = (p / p.sum()) @ v[2, :end].astype(np.float64)
            if what == "v_inf" and end > j0:
                assert got[i, h, 9] == np.inf
                ref[9] = got[i, h, 9] = 0.0
            # test_causal_rows' bound, relative for the large component
            assert (np.abs(got[i, h] - ref) <= 2e-5 * np.maximum(1.0, np.abs(ref))).all(), (i, h)


@pytest.mark.parametrize("n,past", [(33, 127), (768, 3)])
def test_small_values(dev, n, past):
    """v near the smallest normal f32, where bf16 has no three terms left."""
    from qwenasr_amd import kernels as Kr
    print(f"small values n={n} past={past}", flush=True)
    r = rng(n + past)
    m, scale = n + past, np.float32(2.0 ** -122)
    q, k = r.normal(0, 1, (n, 16, 128)).astype(np.float32), r.normal(0, 1, (8, m, 128)).astype(np.float32)
    v = r.normal(0, 0.6, (8, m, 128)).astype(np.float32) * scale
    out = dev.empty((n, 16, 128), np.float32)
    Kr.causal_attention(out, dev.upload(q), dev.upload(k), dev.upload(v), m * 128, n, m, 16, 8, 128, 128 ** -0.5, past)
    ref = attend(q, k, v, past)
    # f32's smallest step, 2^-149, is 2^-27 of the scale: test_causal_rows' bounds
    assert np.linalg.norm((out.numpy() - ref) / scale) <= 1e-6 * np.linalg.norm(ref / scale)
