"""Q8_0 and Q4_K gate / up rows and Q8_0 and Q6_K down rows from their tile-major copies: the same bits as from the GGUF rows (one
arithmetic, in one order), at one token and at token counts that split evenly over the shares of the joint down + combine launch
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
    assert np.array_equal(a[0].view(np.uint16), b[0].view(np.uint16)) and np.array_equal(a[2].view(np.uint32), b[2].view(np.uint32))
    assert maxrel(a[0], oracle.moe_layer_f64(m, a[1], x)) <= TOL
    dl.free()


@pytest.mark.parametrize("nb", [1, 3, 16])
@pytest.mark.parametrize("D,I,E,K,fsh", [(512, 256, 4, 2, 12), (2048, 512, 16, 10, 8), (2560, 256, 33, 8, 21)])
def test_q4k_bits_do_not_depend_on_the_copy(gpu, nb, D, I, E, K, fsh):
    """Q4_K gate / up rows from the copy, from GGUF rows, and from GGUF rows beside the shared expert's tiles: one set of bits."""
    rng = np.random.default_rng(D + nb)
    m = synth.moe_layer(rng, D, I, E, fgu=12, fd=8, fsh=fsh, fshd=8)
    m["topk"] = K
    x = synth.activations(rng, nb, D)
    dl = DeviceLayer(gpu, m, device_only=True)
    planes, names = [], []
    for copies, inside in ((True, None), (False, None), (False, "1")):
        gpu.L.qw_hip_set_repack(gpu.g, copies)
        try:
            with gpu.switches(shared_in_gu=inside):
                path = q.Path(gpu, D, I, E, K, 16)
                gpu.profile(True)
                run_moe(gpu, path, dl, x, nb)
                names.append([n for n, _ in gpu.profile_entries() if n.startswith("qwk_gu_")][0])
                gpu.profile(False)
                H = path.scratch(1).view(np.uint16)
                nbv = 1 << (nb - 1).bit_length() if nb < 9 else 16
                planes.append([H[p * nbv * (K + 1) * I:][:nb * (K + 1) * I].reshape(nb, K + 1, I)[:, :K].copy() for p in (0, 1)])
                path.close()
        finally:
            gpu.L.qw_hip_set_repack(gpu.g, True)
    beside = {12: "qwk_gu_rt", 8: "qwk_gu_rt_s8_c1", 21: "qwk_gu_rt_s21_c1"}[fsh]  # (IQ3_S shared rows without their copy stay in this launch)
    assert names == ["qwk_gu_f112_c2", beside if fsh == 21 else "qwk_gu_rt", beside], names
    for other in planes[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(planes[0], other))
    dl.free()
