"""The front launch of a layer: router rows beside the shared expert's gate/up, a wave per 256 values of K. One wave, eight, and ten (of
which two take a second block of a router row); one token up to sixteen with odd counts between; binary16 and bfloat16 router rows,
expert counts off a multiple of sixteen; shared rows tile-major, Q8_0, of one and of two formats of the other family."""
import numpy as np
import pytest

import qwental_amd as q
from qwental_amd import synth
from helpers import DeviceLayer, maxrel, run_moe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [1, 2, 3, 6, 9, 16])
@pytest.mark.parametrize("rt,E,D,I,fsh,fshu,want", [
    (30, 512, 2048, 256, 21, 21, "qwk_pre_w30_s121"), (1, 33, 2560, 256, 21, 21, "qwk_pre_w1_s121"), (30, 17, 2560, 384, 8, 8, "qwk_pre_w30_s8"), (1, 16, 512, 256, 8, 8, "qwk_pre_w1_s8"),
    (30, 40, 256, 256, 12, 12, "qwk_pre_w30_kq"), (1, 64, 768, 256, 13, 13, "qwk_pre_w1_kq"), (30, 31, 2304, 128 * 3, 12, 23, "qwk_pre_w30_kq"), (1, 20, 2560, 256, 14, 30, "qwk_pre_w1_kq"),
    (30, 128, 1024, 256, 23, 23, "qwk_pre_w30_kq"), (1, 48, 1280, 256, 20, 20, "qwk_pre_w1_kq"), (30, 64, 1792, 256, 1, 12, "qwk_pre_w30_kq")])
def test_front_launch(gpu, oracle, nb, rt, E, D, I, fsh, fshu, want):
    rng = np.random.default_rng(E * 100 + D + nb)
    K = 4
    m = synth.moe_layer(rng, D, I, E, fgu=21, fd=8, fsh=fsh, fshd=8, fshu=fshu)
    m["topk"] = K
    if rt == 30:
        m["Wr"], m["wsg"] = [(np.asarray(w).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16) for w in (m["Wr"], m["wsg"])]
        rows = np.concatenate([m["Wr"].reshape(E, D), m["wsg"].reshape(1, D)]).astype(np.uint32)
        W = (rows << 16).view(np.float32).astype(np.float64)
    else:
        W = np.concatenate([m["Wr"].reshape(E, D), m["wsg"].reshape(1, D)]).astype(np.float64)
    x = synth.activations(rng, nb, D)
    path = q.Path(gpu, D, I, E, K, 16)
    dl = DeviceLayer(gpu, m, router_type=rt, device_only=True)
    gpu.profile(True)
    out, lg, _, _ = run_moe(gpu, path, dl, x, nb)
    names = [n for n, _ in gpu.profile_entries()]
    gpu.profile(False)
    assert want in names, names
    ref = x.view(np.float16).reshape(nb, D).astype(np.float64) @ W.T
    assert maxrel(lg, ref) <= 1e-6  # binary32 sums of up to 2560 products, a chain of at most 90 additions: 90 x 2^-24 = 5e-6 at worst, 2e-7 measured
    one, lg1, _, _ = run_moe(gpu, path, dl, x[nb - 1:nb], 1)  # a token's logits and shared expert do not depend on the others
    assert np.array_equal(lg1[0].view(np.uint32), lg[nb - 1].view(np.uint32)) and np.array_equal(one[0].view(np.uint16), out[nb - 1].view(np.uint16))
    run_moe(gpu, path, dl, x, nb)
    nbv = 1 if nb <= 1 else 2 if nb <= 2 else 4 if nb <= 4 else 8 if nb <= 8 else 16
    Hraw = path.scratch(1).view(np.float16)
    H = (Hraw[:nb * (K + 1) * I].astype(np.float32) + Hraw[nbv * (K + 1) * I:nbv * (K + 1) * I + nb * (K + 1) * I].astype(np.float32)).reshape(nb, K + 1, I)
    _, H32, _ = oracle.moe_layer_f32(m, lg, x, 8 if nb <= 8 else 16)
    assert maxrel(H[:, K], H32[:, K]) <= 1e-5
    dl.free()
    path.close()
