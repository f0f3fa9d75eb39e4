"""A single step's token and logit, reported to pinned host memory, against the
values the device keeps (read back after a run of steps)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graph", [True, False])
def test_step_report(dev, use_graph):
    from qwenasr_amd.model import Decoder
    from qwenasr_amd.synth import SynthDecoder
    cfg = dict(n_layers=2, hidden=1024, n_heads=16, n_kv_heads=8, head_dim=128, intermediate=3072, vocab=4096,
               eps=1e-6, theta=1e6)
    w = SynthDecoder(cfg, seed=9)
    d = Decoder(dev, w, max_seq=300)
    d.set_options(use_graph=use_graph)
    toks, logits, tok = [], [], 7
    for _ in range(6):
        tok = d.forward(token=tok)
        toks.append(tok)
        logits.append(d.last_logit())
    # the same steps as runs of 1, 2, ... 6 (graphs of 4 and 1): the last step's logit comes from the device
    for n in range(1, 7):
        d.kv_len = 0
        out = d.generate(n, first_token=7)
        assert out.tolist() == toks[:n]
        assert np.float32(d.last_logit()) == np.float32(logits[n - 1])
    # an embedding-fed step reports too
    d.kv_len = 0
    e = (w.embed[7].astype(np.uint32) << 16).view(np.float32)
    assert d.forward(embed=e) == toks[0] and d.last_logit() == logits[0]
    d.close()
