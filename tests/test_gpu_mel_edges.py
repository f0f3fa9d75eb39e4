"""The mel launch at the edges of its 16-frame blocks: shortest signals (whole
reflections), one frame more or less than a block, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [160, 200, 201, 399, 2559, 2560, 2561, 2720, 5120, 40123])
def test_mel_blocks(dev, orc, n):
    from qwenasr_amd.model import Encoder
    from qwenasr_amd.synth import ENC_0_6B, SynthEncoder, audio
    print(f"mel n={n}", flush=True)
    enc = Encoder(dev, SynthEncoder(dict(ENC_0_6B, n_layers=1, conv_hidden=32), seed=3))
    x = audio(n, 5)
    got, ref = enc.mel(x), orc.mel(x)
    assert got.shape == ref.shape
    # log10 of f32 sums of 400 products: 2e-4 absolute, the front end's bar
    np.testing.assert_allclose(got, ref, atol=2e-4, rtol=0)
    enc.close()
