"""The dense product as one workgroup per tile of 16 rows and one wave per 256 values of K, at the edges of its range:
one row, a tile's remainder, one wave and sixteen, one token up to sixteen, every weight format, mixed formats."""
import numpy as np
import pytest

import qwental_amd as q
from qwental_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmts,Ns,K,nb", [((21,), (48,), 256, 1), ((21,), (17,), 2560, 3), ((21,), (16,), 4096, 16), ((21,), (1,), 1024, 2), ((8,), (33,), 256, 2),
                                          ((8,), (4099,), 4096, 9), ((8,), (1,), 2304, 16), ((14, 12, 13, 30), (1, 50, 16, 31), 512, 5),
                                          ((23, 20, 1), (15, 33, 100), 4096, 16), ((20, 14), (512, 7), 768, 1)])
def test_small_product(gpu, oracle, fmts, Ns, K, nb):
    rng = np.random.default_rng(K + nb + sum(Ns))
    Ws = [synth.matrix(rng, f, n, K) for f, n in zip(fmts, Ns)]
    x = synth.activations(rng, nb, K)
    path = q.Path(gpu, 2048, 512, 512, 10, 16)
    wbs = [gpu.buf_from(w) for w in Ws]

    def run(x0, count):
        xb = gpu.buf_from(x[x0:x0 + count])
        ys = [gpu.buf(count * n * 4) for n in Ns]
        b = gpu.batch()
        if len(fmts) == 1:
            path.qmv_gg(b, q.Tensor(wbs[0], fmts[0]), Ns[0], K, xb, ys[0], count, fout=True)
        else:
            path.qmv_ggm(b, [q.Tensor(w, f) for w, f in zip(wbs, fmts)], Ns, K, xb, ys, count)
        assert b.end() >= 0, gpu.last_error()
        out = [y.view(np.float32)[:count * n].reshape(count, n).copy() for y, n in zip(ys, Ns)]
        for y in ys + [xb]:
            y.free()
        return out

    got = run(0, nb)
    for f, n, W, y in zip(fmts, Ns, Ws, got):
        ref = oracle.qmv(f, W, n, K, x, f64=True)
        err = np.abs(y - ref).max() / max(np.abs(ref).max(), 1e-30)
        assert err <= 1e-5, (f, err)
    for t in {0, nb - 1}:  # a token's row does not depend on the tokens beside it
        for y, one in zip(got, run(t, 1)):
            assert np.array_equal(one[0].view(np.uint32), y[t].view(np.uint32))
    for bb in wbs:
        bb.free()
    path.close()
