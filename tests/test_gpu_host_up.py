"""Small uploads that the host writes into HBM itself, and batches whose first launch takes the start stamp: the same bits as
with uploads by a launch, step after step with other inputs, and the cases in which the rule leaves the upload to the launch."""
import numpy as np
import pytest

import qwental_amd as q
from qwental_amd import synth
from helpers import DeviceLayer, run_moe

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    g = q.Gpu()
    p = q.Path(g, 1024, 256, 64, 4, 16, device_scratch=True)
    yield g, p
    p.close()
    g.close()


def weights(g, rng, fmt, N, K):
    raw = synth.matrix(rng, fmt, N, K)
    buf = q.Buf(g, raw.nbytes, device_only=True)
    buf.fill(raw)
    return buf, q.Tensor(buf, fmt)


def host_bytes(g):
    """Bytes that the host has written itself; None where the device's memory is not in its window."""
    n = q.gpu.C.c_size_t()
    return n.value if g.L.qw_hip_host_uploads(g.g, q.gpu.C.byref(n)) else None


LIMIT = 256 << 10


# (type, rows, K, tokens): one and several waves a tile, the persistent kernels, K over the staged length; 512 bytes to 240 KB of
# activations, and more than the host writes: 256 KB and six bytes, and a whole buffer every time (behind the large offset)
@pytest.mark.parametrize("fmt,N,K,nb,off", [(8, 17, 256, 1, 0), (21, 4096, 2048, 1, 0), (21, 20000, 2816, 16, 0), (30, 30000, 768, 2, 0), (14, 40000, 512, 3, 0), (8, 1000, 8192, 15, 0), (8, 1000, 8192, 16, 0),
                                            (12, 300, 4096, 16, 1 << 18), (1, 9, 512, 5, 48)])
def test_steps(env, fmt, N, K, nb, off):
    g, p = env
    rng = np.random.default_rng(N + K)
    wb, W = weights(g, rng, fmt, N, K)
    x, y = q.Buf(g, off + nb * K * 2 + 6), q.Buf(g, nb * N * 4)
    for step in range(24):
        act = synth.activations(rng, nb, K)
        res = []
        for sw in (None, 1):
            x.view()[:] = 0
            x.view()[off:off + act.nbytes] = act.view(np.uint8).ravel()
            whole = off > LIMIT / 2 or (step == 0 and sw is None)
            if whole:
                g.L.qw_hip_buf_mark_dirty(x.ref())
            before = host_bytes(g)
            with g.switches(no_host_up=sw):
                b = g.batch()
                p.qmv_gg(b, W, N, K, x, y, nb, xoff=off)
                t = b.end()
            assert 0 < t < 1e-2
            up = x.size if whole else x.size - off  # (in units of sixteen bytes, which ends at the buffer's)
            assert before is None or host_bytes(g) - before == (up if sw is None and up <= LIMIT else 0)
            res.append(y.view(np.uint32).copy())
        assert np.array_equal(*res) and res[0].any()
        assert np.array_equal(x.read(dtype=np.uint8)[off:off + act.nbytes], act.view(np.uint8).ravel())
    for o in (wb, x, y):
        o.free()


@pytest.mark.parametrize("form", ["plain", "written", "address", "in flight"])
def test_left_to_the_launch(env, form):
    """What the host must not write: a buffer that a kernel has written, one whose address is known, and anything while another batch has not
    been waited for - that batch keeps the activations it was submitted with. (plain: none of these, the host writes.)"""
    g, p = env
    rng = np.random.default_rng(3)
    K = N = 1024
    wb, W = weights(g, rng, 8, N, K)
    x, y, z = q.Buf(g, 2 * K * 2), q.Buf(g, 2 * N * 4), q.Buf(g, 2 * N * 4)
    u = q.Buf(g, 2 * N * 4)

    def product(act):  # from a buffer of its own, which goes up by a launch
        ref = q.Buf(g, x.size)
        ref.fill(act)
        with g.switches(no_host_up=1):
            b = g.batch()
            p.qmv_gg(b, W, N, K, ref, u, 2)
            assert b.end() > 0
        ref.free()
        return u.view(np.uint32).copy()

    for step in range(6):
        old, act = synth.activations(rng, 2, K), synth.activations(rng, 2, K)
        x.fill(old if form == "in flight" else act)
        if form == "address":
            assert g.L.qw_hip_buf_devptr(x.ref())
        first = None
        if form == "in flight":
            first = g.batch()
            p.qmv_gg(first, W, N, K, x, z, 2)
            g.L.qw_batch_submit(first.b)
            while not g.L.qw_batch_poll(first.b):  # its upload reads the shadow: that may change once it has run
                pass
            x.fill(act)
        if form == "written":  # made on the device in an earlier step
            b = g.batch()
            p.qmv_gg(b, W, K, K, y, x if step == 0 else z, 1)
            b.end()
            x.fill(act)
        before = host_bytes(g)
        b = g.batch()
        p.qmv_gg(b, W, N, K, x, y, 2)
        assert b.end() > 0
        assert before is None or host_bytes(g) - before == (x.size if form == "plain" else 0)
        if first is not None:
            assert g.L.qw_batch_wait(first.b) > 0
            assert np.array_equal(z.view(np.uint32), product(old))
        assert np.array_equal(y.view(np.uint32), product(act))
    for o in (wb, x, y, z, u):
        o.free()


def test_layer(env):
    """A layer whose front launch is the first of its batch, over host-visible buffers, one to sixteen tokens in turn."""
    g, _ = env
    rng = np.random.default_rng(4)
    D, I, E, K = 2048, 512, 32, 10
    m = synth.moe_layer(rng, D, I, E)
    m["topk"] = K
    dl = DeviceLayer(g, m)
    path = q.Path(g, D, I, E, K, 16)
    for nb in (1, 2, 5, 16, 2, 1):
        x = synth.activations(rng, nb, D)
        res = []
        for sw in (None, 1):
            with g.switches(no_host_up=sw):
                out, lg, sel, t = run_moe(g, path, dl, x, nb)
            assert t > 0
            res.append((out.view(np.uint16).copy(), lg.view(np.uint32).copy()))
        assert np.array_equal(res[0][0], res[1][0]) and np.array_equal(res[0][1], res[1][1])
    dl.free()
    path.close()
