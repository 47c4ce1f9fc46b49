"""Which groups of a ragged step go out together, and that their rows are the same bits as one after the other: every kernel for several groups at
sizes where it can go wrong (tests/test_gpu_vstep_join.py has the cuts), and steps whose groups stay apart."""
import numpy as np
import pytest

import qwental_amd as q
from helpers import DeviceLayer
from qwental_amd import synth
from test_gpu_vstep_batch import table

pytestmark = pytest.mark.gpu

IQ3, IQ3_Q8, NL, K4, Q8 = (21, 21, 21, 21, 21), (21, 21, 8, 8, 8), (21, 20, 12, 23, 20), (12, 14, 12, 12, 14), (8, 8, 8, 8, 8)


def run(gpu, path, dl, size, n, xb, ob):
    par, since = table(size), gpu.L.qw_hip_joint_launches(gpu.g)
    info = path.par_vstep(par, dl.layer, n, xb, ob)
    par.free()
    assert max(info.groups[:info.ngroups]) <= size and sum(info.groups[:info.ngroups]) == sum(n)
    return ob.read(dtype=np.uint16).copy(), gpu.L.qw_hip_joint_launches(gpu.g) - since, gpu.joint_kernels(since)


# (recipe, D, I, experts, top-k, rows, size of a group, router; kernels of the first joint set and once every copy is there)
@pytest.mark.parametrize("recipe,D,I,E,K,rows,size,router,first,later", [
    # Q8_0: a pair of 136 MB, read in GGUF order until it has come 32 times; router in bfloat16
    (Q8, 2048, 512, 64, 8, 45, 16, 30, ["pre_w30_s8", "gu_f8_c16", "dnq_f108_c1_s108_c1"], ["pre_w30_s8", "gu_f108_c2", "dnq_f108_c1_s108_c1"]),
    # Q4_K and Q6_K: a pair of 108 MB; 79 MB of down rows, tile-major at once
    (K4, 1536, 512, 128, 10, 45, 16, 1, ["pre_w1_kq", "gu_rt", "dnq_f114_c1_s114_c1"], ["pre_w1_kq", "gu_f112_c2", "dnq_f114_c1_s114_c1"]),
    # the selection for other expert counts; two groups of unlike sizes
    (K4, 1024, 512, 160, 8, 17, 15, 30, ["pre_w30_kq", "gu_f112_c2", "dnq_f114_c1_s114_c1"], None),
    (IQ3, 1024, 256, 96, 6, 18, 16, 1, ["pre_w1_s121", "gu_f121_c2", "dnq_f121_c1_s121_c1"], None),
    # types as arguments of gate/up, four groups
    ((23, 21, 21, 21, 21), 1024, 512, 64, 4, 28, 7, 30, ["pre_w30_s121", "gu_rt", "dnq_f121_c2_s121_c2"], None),
    ((13, 21, 8, 8, 8), 1024, 512, 64, 4, 33, 11, 1, ["pre_w1_s8", "gu_rt", "dnq_f121_c2_s8_c4"], None),
    ((12, 21, 8, 8, 8), 1024, 256, 64, 4, 20, 10, 1, ["pre_w1_s8", "gu_f112_c2", "dnq_f121_c1_s8_c4"], None),
    # more experts than a group has workgroups: two rounds and three; top-16 of 256
    (NL, 1024, 640, 128, 10, 48, 16, 1, ["pre_w1_kq", "gu_f121_c2", "dnr_f120_c10_s120_c10", "cmb"], None),
    (NL, 512, 640, 256, 16, 64, 16, 30, ["pre_w30_kq", "gu_f121_c2", "dnr_f120_c10_s120_c10", "cmb"], None)])
def test_groups_that_go_out_together(gpu, recipe, D, I, E, K, rows, size, router, first, later):
    gu, dn, sg, su, sd = recipe
    rng = np.random.default_rng(rows + D + E)
    m = synth.moe_layer(rng, D, I, E, fgu=gu, fd=dn, fsh=sg, fshd=sd, **({} if sg == su else {"fshu": su}))
    m["topk"] = K
    if router == 30:
        for k in ("Wr", "wsg"):
            m[k] = (m[k].astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    dl = DeviceLayer(gpu, m, router_type=router, device_only=True)
    path = q.Path(gpu, D, I, E, K, 16, device_scratch=True)
    xb, ob = q.Buf(gpu, rows * D * 2), q.Buf(gpu, rows * D * 2)
    n, sets = [1] * rows, -(-rows // size) // 4 + (-(-rows // size) % 4 > 1)
    xb.fill(synth.activations(rng, rows, D))
    with gpu.switches(no_join=1):
        apart, count, _ = run(gpu, path, dl, size, n, xb, ob)
        assert count == 0
    together, count, made = run(gpu, path, dl, size, n, xb, ob)
    assert count == sets * len(first) and made == ["qwk_" + k for k in first]
    assert np.isfinite(apart.view(np.float16)).all() and np.array_equal(together, apart)
    if later:
        for _ in range(12):
            together, count, made = run(gpu, path, dl, size, n, xb, ob)
            assert np.array_equal(together, apart)
        assert count == sets * len(later) and made == ["qwk_" + k for k in later]
    dl.free()
    path.close()
    for o in (xb, ob):
        o.free()


# Q6_K rows of less than 64 MB, D not a multiple of 512, a group of two with down + combine of its own kind, scratch with shadows
@pytest.mark.parametrize("recipe,D,I,E,rows,size,scratch", [(K4, 1024, 512, 64, 40, 16, True), (IQ3, 1280, 256, 64, 30, 15, True), (NL, 2560, 640, 64, 18, 16, True), (IQ3, 1024, 256, 64, 30, 15, False)])
def test_groups_that_stay_apart(gpu, recipe, D, I, E, rows, size, scratch):
    gu, dn, sg, su, sd = recipe
    rng = np.random.default_rng(rows + D)
    m = synth.moe_layer(rng, D, I, E, fgu=gu, fd=dn, fsh=sg, fshd=sd, **({} if sg == su else {"fshu": su}))
    m["topk"] = 4
    dl = DeviceLayer(gpu, m, device_only=True)
    path = q.Path(gpu, D, I, E, 4, 16, device_scratch=scratch)
    xb, ob = q.Buf(gpu, rows * D * 2), q.Buf(gpu, rows * D * 2)
    xb.fill(synth.activations(rng, rows, D))
    gpu.profile(True)
    apart, _, _ = run(gpu, path, dl, size, [1] * rows, xb, ob)
    gpu.profile(False)
    got, count, _ = run(gpu, path, dl, size, [1] * rows, xb, ob)
    assert count == 0 and np.array_equal(got, apart)
    dl.free()
    path.close()
    for o in (xb, ob):
        o.free()
