"""Groups of a ragged step that go through the layer side by side (the _j kernels): the same rows, bit for bit, as the groups one after the
other (what a profiled device runs), over steps whose groups are not alike."""
import numpy as np
import pytest

import qwental_amd as q
from helpers import DeviceLayer
from qwental_amd import synth
from test_gpu_vstep_batch import table

pytestmark = pytest.mark.gpu

IQ3, IQ3_Q8, NL, K4, Q8 = (21, 21, 21, 21, 21), (21, 21, 8, 8, 8), (21, 20, 12, 23, 20), (12, 14, 12, 12, 14), (8, 8, 8, 8, 8)


# two groups; three, the smallest of them in another form of down + combine (one or two tokens); four, a full set; five to eight, where the
# second set starts on the scratch of the first; shares of one, two and four quarters side by side
@pytest.mark.parametrize("recipe,D,I,E,rows,size", [
    (IQ3, 2048, 512, 64, 32, 16), (IQ3, 2048, 512, 128, 33, 16), (IQ3, 1024, 256, 64, 61, 16), (IQ3_Q8, 2048, 512, 64, 45, 16), (IQ3_Q8, 1024, 256, 64, 37, 7),
    (IQ3, 1024, 512, 128, 64, 9), (NL, 2560, 640, 64, 45, 16), (NL, 2560, 640, 64, 18, 16), (Q8, 1024, 512, 64, 50, 16), (Q8, 2048, 256, 64, 19, 4), (K4, 1024, 512, 64, 40, 16), (K4, 1024, 256, 128, 35, 12)])
@pytest.mark.parametrize("router,host_out", [(1, True), (30, False)])
def test_groups_beside_each_other(gpu, recipe, D, I, E, rows, size, router, host_out):
    gu, dn, sg, su, sd = recipe
    K = 10 if E >= 128 else 4
    rng = np.random.default_rng(rows * 7 + D + E)
    m = synth.moe_layer(rng, D, I, E, fgu=gu, fd=dn, fsh=sg, fshd=sd, **({} if sg == su else {"fshu": su}))
    m["topk"] = K
    if router == 30:
        for k in ("Wr", "wsg"):
            m[k] = (m[k].astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    dl = DeviceLayer(gpu, m, router_type=router, device_only=True)
    path = q.Path(gpu, D, I, E, K, 16, device_scratch=True)
    xb, ob = q.Buf(gpu, rows * D * 2), q.Buf(gpu, rows * D * 2, device_only=not host_out)
    n = [1] * (rows - 5) + [2, 3]
    for step in range(3):
        xb.fill(synth.activations(rng, rows, D))
        got = []
        for profiled in (True, False, False):
            par = table(size)
            ob.fill(np.full(rows * D, 0x7E00, np.uint16))
            gpu.profile(profiled)
            info = path.par_vstep(par, dl.layer, n, xb, ob)
            gpu.profile(False)
            assert info.ngroups == -(-rows // size) and info.gpu_ms > 0 and par.group_cost(size) > 0
            got.append(ob.view(np.uint16).copy() if host_out else ob.read(dtype=np.uint16))
            assert np.array_equal(got[-1], ob.read(dtype=np.uint16))
            par.free()
        assert np.isfinite(got[0].view(np.float16)).all() and np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    dl.free()
    path.close()
    for o in (xb, ob):
        o.free()
