"""K-quant and IQ4_XS rows in a layer. Down rows through the range kernel (H rows staged in LDS, a contiguous range of tiles a
workgroup) and, for one token, through the launch that combines too: rows of one and two blocks, no, equal and Q8_0 shared
rows, few experts (several rounds of ranges meet one expert) and many, and the line to the any-shape kernel."""
import numpy as np
import pytest

import qwental_amd as q
from qwental_amd import synth
from helpers import DeviceLayer, maxrel, run_moe

pytestmark = pytest.mark.gpu
TOL = 2e-3  # binary16 results of a layer (half an ulp is 4.9e-4 of a value) against the float64 layer


@pytest.mark.parametrize("fd,fshd,D,I,E,K,nb,want", [
    (14, 14, 2048, 512, 64, 10, 4, "qwk_dnr_f14_c1_s14_c1"), (14, 8, 256, 256, 8, 2, 16, "qwk_dnr_f14_c1_s8_c4"), (14, 14, 1280, 512, 16, 4, 1, "qwk_dnc_f14_c1_s14_c1"),
    (12, 12, 768, 256, 48, 6, 9, "qwk_dnr_f12_c1_s12_c1"), (12, 8, 2560, 512, 32, 10, 2, "qwk_dnr_f12_c1_s8_c4"), (13, 13, 1024, 512, 512, 10, 16, "qwk_dnr_f13_c1_s13_c1"),
    (13, 13, 512, 256, 16, 16, 1, "qwk_dnc_f13_c1_s13_c1"), (12, 12, 1024, 256, 16, 4, 1, "qwk_dnc_f12_c1_s12_c1"), (23, 23, 2048, 256, 128, 8, 3, "qwk_dnr_f23_c1_s23_c1"), (23, 8, 1536, 512, 16, 1, 1, "qwk_dnc_f23_c1_s8_c4"),
    (14, 12, 1024, 512, 16, 4, 4, "qwk_dn_rt"), (12, 12, 1024, 768, 16, 4, 4, "qwk_dn_rt")])
def test_kq_down_rows(gpu, oracle, fd, fshd, D, I, E, K, nb, want):
    rng = np.random.default_rng(fd * 1000 + fshd * 10 + D + I + nb)
    m = synth.moe_layer(rng, D, I, E, fgu=21, fd=fd, fsh=8, fshd=fshd)
    m["topk"] = K
    x = synth.activations(rng, nb, D)
    path = q.Path(gpu, D, I, E, K, 16)
    dl = DeviceLayer(gpu, m, device_only=True)
    gpu.profile(True)
    out, lg, _, _ = run_moe(gpu, path, dl, x, nb)
    names = [n for n, _ in gpu.profile_entries()]
    gpu.profile(False)
    assert want in names, names
    assert maxrel(out, oracle.moe_layer_f64(m, lg, x)) <= TOL
    with gpu.switches(dn_any="1"):  # the any-shape kernel: the same products in the same order, so the same bits
        other = run_moe(gpu, q.Path(gpu, D, I, E, K, 16), dl, x, nb)[0]
    assert np.array_equal(out.view(np.uint16), other.view(np.uint16))
    dl.free()
    path.close()


@pytest.mark.parametrize("fsh,fshu,D,I,nb", [(12, 12, 1024, 256, 3), (12, 13, 2048, 512, 16), (14, 30, 2048, 384, 1), (20, 1, 2048, 640, 7), (23, 12, 1536, 512, 2), (13, 14, 2560, 640, 16),
                                             (12, 12, 1792, 256, 5), (30, 20, 512, 512, 4)])
def test_kq_shared_gate_up(gpu, oracle, fsh, fshu, D, I, nb):
    """The shared expert's gate/up of the multi-format family in the front launch: K cut over two to six waves, one and two blocks each
    (and 1792, which has no such cut)."""
    rng = np.random.default_rng(fsh * 1000 + fshu * 10 + D + I + nb)
    m = synth.moe_layer(rng, D, I, 16, fgu=21, fd=8, fsh=fsh, fshd=8, fshu=fshu)
    m["topk"] = 4
    x = synth.activations(rng, nb, D)
    path = q.Path(gpu, D, I, 16, 4, 16)
    dl = DeviceLayer(gpu, m, device_only=True)
    out, lg, _, _ = run_moe(gpu, path, dl, x, nb)
    assert maxrel(out, oracle.moe_layer_f64(m, lg, x)) <= TOL
    dl.free()
    path.close()
