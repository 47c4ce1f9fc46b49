"""A ragged step as one batch against a batch a group (what a profiled device still runs): the same rows bit for bit, over the
forms a group's last launch takes, and what the groups' launches write to the host themselves."""
import numpy as np
import pytest

import qwental_amd as q
from helpers import DeviceLayer
from qwental_amd import synth

pytestmark = pytest.mark.gpu


def table(size):
    """A planner whose cheapest cut has as few groups of at most `size` rows as can be."""
    p = q.Par()
    for b in range(1, 17):
        for _ in range(2):
            p.observe(b, 0.01 if b <= size else 50.0)
    return p


# (routed gate/up, down, shared gate, up, down), D, I, groups: down + combine by token shares, one token a group, a combine of its own
# (IQ4_NL), 64 groups (as many as a batch has parts)
@pytest.mark.parametrize("recipe,D,I,n,size", [((21, 21, 21, 21, 21), 1024, 512, [9, 1, 13], 8), ((21, 21, 8, 8, 8), 1024, 256, [1, 2], 1), ((21, 20, 12, 23, 20), 2560, 640, [5, 16, 3], 16),
                                               ((8, 8, 8, 8, 8), 1024, 512, [16, 4], 4), ((21, 21, 21, 21, 21), 1024, 256, [4] * 16, 1)])
@pytest.mark.parametrize("scratch,host_out", [(True, True), (False, True), (True, False)])
def test_rows(gpu, recipe, D, I, n, size, scratch, host_out):
    gu, dn, sg, su, sd = recipe
    E, K, R = 32, 4, sum(n)
    rng = np.random.default_rng(R + D)
    m = synth.moe_layer(rng, D, I, E, fgu=gu, fd=dn, fsh=sg, fshd=sd, **({} if sg == su else {"fshu": su}))
    m["topk"] = K
    dl = DeviceLayer(gpu, m, device_only=True)
    path = q.Path(gpu, D, I, E, K, 16, device_scratch=scratch)
    xb, got = q.Buf(gpu, R * D * 2), []
    for step in range(3):
        x = synth.activations(rng, R, D)
        xb.fill(x)
        for grouped in (False, True):
            ob = q.Buf(gpu, R * D * 2, device_only=not host_out)
            par = table(size)
            gpu.profile(grouped)
            info = path.par_vstep(par, dl.layer, n, xb, ob)
            gpu.profile(False)
            assert max(info.groups[:info.ngroups]) <= size and sum(info.groups[:info.ngroups]) == R
            assert info.gpu_ms > 0 and info.wall_ms >= 0.5 * info.gpu_ms and par.group_cost(size) > 0
            hbm = ob.read(dtype=np.uint16)
            if host_out:
                assert np.array_equal(hbm, ob.view(np.uint16))
            got.append(hbm.copy())
            par.free()
            ob.free()
        assert np.array_equal(got[-1], got[-2]) and (step == 0 or not np.array_equal(got[-1], got[-3]))
    dl.free()
    path.close()
    xb.free()


@pytest.mark.parametrize("second", [0, 512, 1024])
def test_two_writers_of_one_buffer(gpu, second):
    """Ranges that overlap are carried back once, after the batch; disjoint ones by the products themselves."""
    rng = np.random.default_rng(1)
    N = K = 1024
    w = [synth.matrix(rng, f, N, K) for f in (8, 12)]
    bufs = [q.Buf(gpu, r.nbytes, device_only=True) for r in w]
    for b, r in zip(bufs, w):
        b.fill(r)
    W, V = q.Tensor(bufs[0], 8), q.Tensor(bufs[1], 12)
    path = q.Path(gpu, 1024, 256, 64, 4, 16, device_scratch=True)
    x, y = q.Buf(gpu, K * 2), q.Buf(gpu, 2 * N * 4)
    for _ in range(4):
        x.fill(synth.activations(rng, 1, K))
        y.view()[:] = 0xEE
        b = gpu.batch()
        path.qmv_gg(b, W, N, K, x, y, 1)
        path.qmv_gg(b, V, N, K, x, y, 1, yoff=4 * second)
        assert b.end() > 0
        hbm = y.read(dtype=np.uint32)
        assert np.array_equal(y.view(np.uint32)[:N + second], hbm[:N + second])
    path.close()
    for o in (*bufs, x, y):
        o.free()


@pytest.mark.parametrize("rows", [(5,), (16, 17), (1, 100, 33), (4096, 16, 48, 7), (15, 1, 1, 16)])
@pytest.mark.parametrize("nb", [1, 4, 16])
def test_matrices_of_one_launch(gpu, rows, nb):
    """The matrix a workgroup of the dense launch takes: first and last tiles of one to four matrices, each against its own launch."""
    rng = np.random.default_rng(len(rows) + nb)
    K, fmts = 512, (12, 23, 14, 30)
    path = q.Path(gpu, 1024, 256, 64, 4, 16, device_scratch=True)
    ws, bufs = [], []
    for f, r in zip(fmts, rows):
        raw = synth.matrix(rng, f, r, K)
        bufs.append(q.Buf(gpu, raw.nbytes, device_only=True))
        bufs[-1].fill(raw)
        ws.append(q.Tensor(bufs[-1], f))
    x = q.Buf(gpu, nb * K * 2)
    x.fill(synth.activations(rng, nb, K))
    ys, zs = [[q.Buf(gpu, nb * r * 4) for r in rows] for _ in range(2)]
    b = gpu.batch()
    path.qmv_ggm(b, ws, list(rows), K, x, ys, nb)
    assert b.end() > 0
    for w, r, z in zip(ws, rows, zs):
        b = gpu.batch()
        path.qmv_gg(b, w, r, K, x, z, nb)
        assert b.end() > 0
    for y, z in zip(ys, zs):
        assert np.array_equal(y.view(np.uint32), z.view(np.uint32)) and y.view(np.uint32).any()
    path.close()
    for o in (*bufs, x, *ys, *zs):
        o.free()


def layer_at(g, path, b, dl, f, nb, x, lg, sel, H, psh, poff, pd, doff, out, ooff):
    """One layer by its four dispatches, Psh, Pg and out at byte offsets of buffers of the caller's (path has dispatched the layer before: its kernels exist)."""
    gu, dn, sg, su, sd = f
    T, tail = dl.layer.c, "_n%d_e%dk%dd%di%d" % (g.L.qw_path_nbv(nb), path.E, path.topk, path.D, path.I)
    tensor = lambda i, t: g.L.qw_batch_buf(b.b, i, t.buf, t.offset)
    scratch = lambda i, which: g.L.qw_batch_buf(b.b, i, g.L.qw_path_scratch(path.p, which), 0)
    nbr = np.array([nb], np.uint32)

    def begin(name):
        k = g.kernel(name + tail)
        assert k, name + tail
        b.kernel(k)

    begin("moe_pre_gg_%d_%d_r1_w%d" % (sg, su, T.router.type))
    for i, t in ((0, T.router), (1, T.sh_gate_w), (6, T.sh_gate), (7, T.sh_up)):
        tensor(i, t)
    for i, buf in ((2, x), (3, lg), (5, sel), (8, H)):
        b.buf(i, buf)
    scratch(13, 0)
    b.bytes(14, nbr)
    b.dispatch(1, 1, 1, 256, 1, 1)
    begin("moe_gu_gg_%d_%d_g1" % (gu, sd))
    for i, t in ((0, T.gate), (1, T.up), (2, T.sh_down)):
        tensor(i, t)
    b.buf(3, psh, poff)
    for i, buf in ((4, x), (5, sel), (6, H)):
        b.buf(i, buf)
    scratch(11, 0)
    b.bytes(12, nbr)
    b.dispatch(1, 1, 1, 256, 1, 1)
    begin("moe_dn_gg_%d_s4" % dn)
    tensor(0, T.down)
    b.buf(2, H)
    b.buf(3, sel)
    scratch(7, 0)
    b.buf(9, pd, doff)
    b.dispatch(1, 1, 1, 128, 1, 1)
    begin("moe_cmb_gg_%d_s4" % dn)
    b.buf(1, psh, poff)
    b.buf(3, sel)
    b.buf(4, out, ooff)
    b.bytes(8, nbr)
    b.buf(9, pd, doff)
    b.dispatch(1, 1, 1, 256, 1, 1)


# down + combine of one token (qwk_dnc_*) and by token shares (qwk_dnq_*), IQ3_S and Q8_0
@pytest.mark.parametrize("recipe,nb", [((21, 21, 21, 21, 21), 1), ((21, 21, 8, 8, 8), 2), ((8, 8, 8, 8, 8), 1), ((8, 8, 8, 8, 8), 4), ((21, 21, 21, 21, 21), 16)])
@pytest.mark.parametrize("product", [True, False])
def test_partial_results_of_two_layers_beside_each_other(gpu, recipe, nb, product):
    """Pg, Psh and out of two layers at two offsets of host-visible buffers, a dense product or the second layer last: every byte is in the shadow when the batch has ended."""
    D, I, E, K = 1024, 512, 64, 4
    rng = np.random.default_rng(nb)
    gu, dn, sg, su, sd = recipe
    m = synth.moe_layer(rng, D, I, E, fgu=gu, fd=dn, fsh=sg, fshd=sd)
    m["topk"] = K
    dl = DeviceLayer(gpu, m, device_only=True)
    path = q.Path(gpu, D, I, E, K, 16, device_scratch=True)
    nbv = gpu.L.qw_path_nbv(nb)
    x, lg, sel = q.Buf(gpu, nb * D * 2), q.Buf(gpu, path.logits_bytes(nb), device_only=True), q.Buf(gpu, path.sel_bytes(nb), device_only=True)
    H = q.Buf(gpu, nbv * (K + 1) * I * 4, device_only=True)
    psh, pd, out, y = q.Buf(gpu, 2 * nbv * D * 4), q.Buf(gpu, 2 * nbv * K * D * 4), q.Buf(gpu, 2 * nb * D * 2), q.Buf(gpu, nb * 4096 * 4)
    wb = q.Buf(gpu, 4096 * (D // 32) * 34, device_only=True)
    wb.fill(synth.matrix(rng, 8, 4096, D))
    b = gpu.batch()
    path.gg_moe(b, dl.layer, nb, x, lg, sel, out)
    b.end()
    for step in range(4):
        x.fill(synth.activations(rng, nb, D))
        for buf in (psh, pd, out, y):
            buf.view()[:] = 0xEE
        b = gpu.batch()
        for l in range(2):
            layer_at(gpu, path, b, dl, recipe, nb, x, lg, sel, H, psh, l * nbv * D * 4, pd, l * nbv * K * D * 4, out, l * nb * D * 2)
        if product:
            path.qmv_gg(b, q.Tensor(wb, 8), 4096, D, x, y, nb)
        assert b.end() > 0
        got = [buf.view().copy() for buf in (psh, pd, out)]  # (before anything else waits for the device)
        for v, buf in zip(got, (psh, pd, out)):
            assert np.array_equal(v, buf.read(dtype=np.uint8))
        for v, used in zip(got, (nb * D * 4, nb * K * D * 4, nb * D * 2)):
            half = v.size // 2
            assert np.array_equal(v[:used], v[half:half + used]) and np.isfinite(v[:used].view(np.float32 if v is not got[2] else np.float16)).all()
    path.close()
    dl.free()
    for o in (x, lg, sel, H, psh, pd, out, y, wb):
        o.free()
