"""One path over many kernels (token counts, router formats): what it dispatches stays that of a path that has met only this one kernel."""
import numpy as np
import pytest

import qwental_amd as q
from helpers import DeviceLayer
from qwental_amd import synth

pytestmark = pytest.mark.gpu


def out_of(gpu, path, dl, x, nb, D):
    bufs = [q.Buf(gpu, n) for n in (nb * D * 2, path.logits_bytes(16), path.sel_bytes(16), nb * D * 2)]
    bufs[0].fill(x)
    b = gpu.batch()
    path.gg_moe(b, dl.layer, nb, *bufs)
    b.end()
    y = bufs[3].view(np.uint16).copy()
    for buf in bufs:
        buf.free()
    return y


@pytest.mark.parametrize("D,I", [(256, 256), (1024, 512)])
def test_many_kernels(gpu, D, I):
    rng = np.random.default_rng(D)
    dls, paths = [], []
    for gu, dn, sg, su, sd in ((21, 21, 21, 21, 21), (8, 8, 8, 8, 8), (21, 20, 12, 23, 20), (21, 21, 8, 8, 8)):
        m = synth.moe_layer(rng, D, I, 32, fgu=gu, fd=dn, fsh=sg, fshd=sd, **({} if sg == su else {"fshu": su}))
        m["topk"] = 4
        dls.append(DeviceLayer(gpu, m, device_only=True))
    shared = q.Path(gpu, D, I, 32, 4, 16)
    for _ in range(2):  # more kernels than the path keeps, in an order that brings each back after the others
        for nb in range(1, 17):
            x = synth.activations(rng, nb, D)
            for dl in dls:
                own = q.Path(gpu, D, I, 32, 4, 16)
                assert np.array_equal(out_of(gpu, shared, dl, x, nb, D), out_of(gpu, own, dl, x, nb, D))
                own.close()
    shared.close()
    for dl in dls:
        dl.free()
