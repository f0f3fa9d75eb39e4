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
