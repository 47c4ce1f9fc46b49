"""Results of a dense product that its kernel writes to the shadow itself (and, as the last launch of a batch, ends the batch
with): after every batch the shadow holds the bytes that HBM holds, over each kernel that does so, and where the rule sends
the results back by a launch of their own instead."""
import numpy as np
import pytest
import torch

import qwental_amd as q
from qwental_amd import synth
from helpers import DeviceLayer

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


def same(y):
    """Shadow and HBM, bit for bit."""
    return np.array_equal(y.view(np.uint32), y.read(dtype=np.uint32))


# (type, rows, K, tokens): a workgroup a tile with one and several waves; the persistent kernels over whole and cut rows;
# rows that do not fill a tile; IQ3_S beside the tile-major copy and past the staged K
SHAPES = [(8, 17, 256, 1), (8, 5127, 2560, 7), (12, 100, 4096, 16), (14, 20000, 1024, 4), (14, 40000, 512, 3), (1, 9, 512, 5), (30, 30000, 768, 2),
          (20, 24000, 1024, 16), (21, 4096, 2048, 1), (21, 100, 1024, 3), (21, 33000, 512, 2), (21, 20000, 2816, 16),
          (8, 8191, 256, 2), (8, 20000, 512, 1), (12, 32000, 512, 3), (14, 2047, 256, 1)]  # up to 2000 workgroups; 128 and more count in sixteen words first


@pytest.mark.parametrize("fmt,N,K,nb", SHAPES)
def test_shadow_is_hbm(env, fmt, N, K, nb):
    g, p = env
    rng = np.random.default_rng(N + K)
    wb, W = weights(g, rng, fmt, N, K)
    x, y = q.Buf(g, nb * K * 2), q.Buf(g, nb * N * 4)
    seen = []
    for step in range(3):  # other activations each time: nothing of the step before may be left
        x.fill(synth.activations(rng, nb, K))
        y.view()[:] = 0xEE
        b = g.batch()
        p.qmv_gg(b, W, N, K, x, y, nb)
        assert b.end() > 0
        assert same(y)
        seen.append(y.view(np.float32).copy())
    assert all(np.isfinite(v).all() for v in seen) and not np.array_equal(seen[0], seen[1])
    for o in (wb, x, y):
        o.free()


@pytest.mark.parametrize("form", ["two writers", "chain", "flush", "submit", "binary16", "device output", "graph"])
def test_rules(env, form):
    """What else may surround such a launch in a batch."""
    g, p = env
    rng = np.random.default_rng(5)
    K = N = 1024
    wb, W = weights(g, rng, 8, N, K)
    vb, V = weights(g, rng, 12, N, K)
    x, y, z, dev = q.Buf(g, 2 * K * 2), q.Buf(g, 4 * N * 4), q.Buf(g, 2 * N * 4), q.Buf(g, 2 * N * 4, device_only=True)
    g.L.qw_hip_set_graphs(g.g, form == "graph")
    try:
        for step in range(4):
            x.fill(synth.activations(rng, 2, K))
            y.view()[:] = 0xEE
            b = g.batch()
            if form == "two writers":  # one buffer, two ranges
                p.qmv_gg(b, W, N, K, x, y, 2)
                p.qmv_gg(b, V, N, K, x, y, 2, yoff=2 * N * 4)
            elif form == "binary16":
                p.qmv_gg(b, W, N, K, x, y, 2, fout=False)
            elif form == "device output":  # nothing at all is carried back; the reader takes HBM
                p.qmv_gg(b, W, N, K, x, dev, 2)
            else:
                for _ in range(10 if form == "graph" else 1):
                    p.qmv_gg(b, W, N, K, x, y, 2)
                    p.qmv_gg(b, V, N, K, x, dev, 2)
                    if form == "flush":
                        b.flush()
                p.qmv_gg(b, V, N, K, x, z, 2)
            if form == "submit":
                g.L.qw_batch_submit(b.b)
                assert g.L.qw_batch_wait(b.b) > 0
            else:
                assert b.end() > 0
            ref = q.Buf(g, 4 * N * 4, device_only=True)  # the same products, results read from HBM
            c = g.batch()
            p.qmv_gg(c, W, N, K, x, ref, 2, fout=form != "binary16")
            p.qmv_gg(c, V, N, K, x, ref, 2, yoff=2 * N * 4)
            assert c.end() > 0
            r = ref.read(dtype=np.uint32)
            first, second = r[:2 * N] if form != "binary16" else r[:N], r[2 * N:]
            if form == "device output":
                assert np.array_equal(dev.read(dtype=np.uint32), first)
            else:
                got = y.view(np.uint32)
                assert np.array_equal(got[:first.size], first)
                if form == "two writers":
                    assert np.array_equal(got[2 * N:], second)
                else:
                    assert (got[first.size:] == 0xEEEEEEEE).all()
                    if form != "binary16":
                        assert np.array_equal(z.view(np.uint32), second) and same(z) and np.array_equal(dev.read(dtype=np.uint32), second)
            ref.free()
    finally:
        g.L.qw_hip_set_graphs(g.g, False)
        torch.cuda.synchronize()
        for o in (wb, vb, x, y, z, dev):
            o.free()


@pytest.mark.parametrize("recipe,D,I,E,topk,nb", [((21, 21, 21, 21, 21), 1024, 256, 64, 4, 1), ((21, 21, 8, 8, 8), 2048, 512, 128, 10, 3), ((8, 8, 8, 8, 8), 1024, 512, 64, 8, 16),
                                                  ((21, 20, 12, 23, 20), 2560, 640, 64, 4, 1), ((21, 20, 12, 23, 20), 2560, 640, 64, 4, 5), ((12, 14, 12, 12, 14), 1024, 256, 64, 6, 2)])
@pytest.mark.parametrize("scratch", [False, True])
def test_layer(env, recipe, D, I, E, topk, nb, scratch):
    """One MoE layer over host-visible buffers: every shadow (its scratch buffers too, where they are host-visible) holds what
    HBM holds, the output what a batch ended by a launch of its own (submit, then wait) leaves."""
    g, _ = env
    rng = np.random.default_rng(D + nb)
    p = q.Path(g, D, I, E, topk, 16, device_scratch=scratch)
    layer = DeviceLayer(g, synth.moe_layer(rng, D, I, E, fgu=recipe[0], fd=recipe[1], fsh=recipe[2], fshd=recipe[4], fshu=recipe[3]), device_only=True)
    x, lg, sel, out = q.Buf(g, nb * D * 2), q.Buf(g, p.logits_bytes(nb)), q.Buf(g, p.sel_bytes(nb)), q.Buf(g, nb * D * 2)
    for step in range(3):
        x.fill(synth.activations(rng, nb, D))
        got = []
        for ended in (False, True):
            out.view()[:] = lg.view()[:] = sel.view()[:] = 0xEE
            if not scratch:  # what the layer overwrites need not go up: garbage in it changes nothing
                for i, lo, n in ((1, 0, nb * (topk + 1) * I * 2), (3, 0, nb * topk * D * 4)):
                    c = g.L.qw_path_scratch(p.p, i).contents
                    np.ctypeslib.as_array((q.gpu.C.c_uint8 * c.size).from_address(c.ptr))[lo:lo + n] = 0x7F
            b = g.batch()
            p.gg_moe(b, layer.layer, nb, x, lg, sel, out)
            if ended:
                assert b.end() > 0
            else:
                g.L.qw_batch_submit(b.b)
                assert g.L.qw_batch_wait(b.b) > 0
            for buf in (lg, sel, out):
                assert np.array_equal(buf.view(), buf.read())
            got.append([buf.view().copy() for buf in (out, lg, sel)])
            if not scratch:
                for i in (1, 2, 3):  # H, Psh, Pg
                    c = g.L.qw_path_scratch(p.p, i).contents
                    raw = np.ctypeslib.as_array((q.gpu.C.c_uint8 * c.size).from_address(c.ptr)).copy()
                    hbm = np.empty(c.size, np.uint8)
                    assert g.L.qw_hip_buf_read(q.gpu.C.byref(c), 0, hbm.ctypes.data, c.size) and np.array_equal(raw, hbm)
                    got[-1].append(raw)
        assert all(np.array_equal(a, b) for a, b in zip(*got))
        assert np.isfinite(out.view(np.float16)).all()
    p.close()
    layer.free()
    for o in (x, lg, sel, out):
        o.free()


def test_slot_passes_between_streams(env):
    """A batch that ends itself gives its slot and the counters in it back as it found them: the next batch, on the other stream, takes the
    same slot and ends itself too. Few and many workgroups (which count in sixteen words first), the persistent kernel, a layer."""
    g, _ = env
    rng = np.random.default_rng(9)
    p = q.Path(g, 1024, 256, 64, 4, 16, device_scratch=True)
    layer = DeviceLayer(g, synth.moe_layer(rng, 1024, 256, 64), device_only=True)
    x, lg, sel, out = q.Buf(g, 3 * 1024 * 2), g.buf(p.logits_bytes(3)), g.buf(p.sel_bytes(3)), q.Buf(g, 3 * 1024 * 2)
    shapes = [(8, 8000, 1024), (8, 64, 1024), (14, 40000, 512), (12, 2064, 256)]
    ws = [weights(g, rng, *s) for s in shapes]
    ys = [q.Buf(g, 3 * N * 4) for _, N, _ in shapes]
    want = None
    x.fill(synth.activations(rng, 3, 1024))
    try:
        for step in range(8):
            g.L.qw_gpu_set_stream(g.g, step % 2)
            got = []
            for (_, N, K), (_, W), y in zip(shapes, ws, ys):
                y.view()[:] = 0xEE
                b = g.batch()
                p.qmv_gg(b, W, N, K, x, y, 3)
                assert b.end() > 0 and same(y)
                got.append(y.view().copy())
                g.L.qw_gpu_set_stream(g.g, (step + len(got)) % 2)
            out.view()[:] = 0xEE
            b = g.batch()
            p.gg_moe(b, layer.layer, 3, x, lg, sel, out)
            assert b.end() > 0 and np.array_equal(out.view(), out.read())
            got.append(out.view().copy())
            want = want or got
            assert all(np.array_equal(a, c) for a, c in zip(got, want))
    finally:
        g.L.qw_gpu_set_stream(g.g, 0)
        p.close()
        layer.free()
        for o in [x, lg, sel, out] + ys + [w for w, _ in ws]:
            o.free()
