"""Q8_0 and Q4_K gate / up rows and Q8_0 and Q6_K down rows from their tile-major copies: the same bits as from the GGUF rows (one
arithmetic, in one order; Q4_K: another split of a weight, the difference bounded), at one token and at token counts that split evenly over the shares of the joint down + combine launch
and that do not, rows of one and two blocks, odd numbers of tiles a workgroup, with and without a shared expert of the same format."""
import numpy as np
import pytest

import qwental_amd as q
from qwental_amd import synth
from helpers import DeviceLayer, maxrel, run_moe

pytestmark = pytest.mark.gpu
TOL = 2e-3  # binary16 results of a layer (half an ulp is 4.9e-4 of a value) against the float64 layer


@pytest.mark.parametrize("nb", [1, 2, 3, 5, 8, 9, 16])
@pytest.mark.parametrize("fgu,fd,fsh,fshd,D,I,E,K", [
    (8, 8, 8, 8, 2048, 512, 16, 10), (8, 8, 8, 21, 512, 256, 4, 2), (8, 21, 8, 8, 2560, 512, 8, 4), (12, 8, 12, 8, 1024, 256, 33, 8),
    (12, 14, 12, 14, 2048, 512, 80, 10), (12, 14, 8, 8, 1536, 256, 208, 6), (12, 12, 12, 12, 512, 256, 8, 8)])
def test_tiled_rows_equal_gguf_rows(gpu, oracle, nb, fgu, fd, fsh, fshd, D, I, E, K):
    rng = np.random.default_rng(fgu * 100 + fd * 10 + D + nb)
    m = synth.moe_layer(rng, D, I, E, fgu=fgu, fd=fd, fsh=fsh, fshd=fshd)
    m["topk"] = K
    x = synth.activations(rng, nb, D)
    x[nb - 1] = x[0]
    dl = DeviceLayer(gpu, m, device_only=True)
    res = []
    for copies in (True, False):
        gpu.L.qw_hip_set_repack(gpu.g, copies)
        try:
            path = q.Path(gpu, D, I, E, K, 16)
            gpu.profile(True)
            out, lg, _, _ = run_moe(gpu, path, dl, x, nb)
            names = [n for n, _ in gpu.profile_entries()]
            gpu.profile(False)
            res.append((out, lg, path.scratch(3).view(np.float32)[:nb * K * D].copy(), names))
            path.close()
        finally:
            gpu.L.qw_hip_set_repack(gpu.g, True)
    a, b = res
    assert ("qwk_gu_f108_c2" if fgu == 8 else "qwk_gu_f112_c2") in a[3] and not any("108" in n or "112" in n or "114" in n for n in b[3]), (a[3], b[3])
    if fd == 8 and fshd in (8, 0):
        assert any(n.startswith("qwk_dn%s_f108" % ("c" if nb == 1 else "q")) for n in a[3]), a[3]
    if fd == 14 and E * D * (I // 256 * 210) >= 64 << 20:
        assert any(n.startswith("qwk_dn%s_f114" % ("c" if nb == 1 else "q")) for n in a[3]), a[3]
    if fgu == 12:  # sums of 2560 products and fewer in binary32: 3e-7 of a value to float64 either way, twice that apart, a few times over at the worst value
        assert maxrel(a[2], b[2]) <= 4e-6
    else:
        assert np.array_equal(a[0].view(np.uint16), b[0].view(np.uint16)) and np.array_equal(a[2].view(np.uint32), b[2].view(np.uint32))
    assert maxrel(a[0], oracle.moe_layer_f64(m, a[1], x)) <= TOL
    dl.free()
