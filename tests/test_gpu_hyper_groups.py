"""The hyper-connection's groups of tokens: at token counts that do not fill them evenly every token has the bits it has alone."""
import numpy as np
import pytest

from qwental_amd import synth
from test_gpu_hyper import Hyper

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,nb", [(2048, 3), (2048, 5), (1024, 6), (2048, 7), (2560, 9), (2048, 11), (2048, 13), (1024, 15)])
def test_tokens_alone(gpu, D, nb):
    rng = np.random.default_rng(D + nb)
    hy = Hyper(gpu, D, 16, rng)
    h, out, inj = synth.hyper_state(rng, nb, D)
    for three in (False, True):
        whole = hy.run(h, out, inj, 1, three=three)
        for t in range(nb):
            for a, b in zip(whole, hy.run(h[t:t + 1], out[t:t + 1], inj[t:t + 1], 1, three=three)):
                assert np.array_equal(a[t:t + 1].view(np.uint8), b.view(np.uint8)), t
    hy.free()
