"""The copies between host shadows and HBM around a batch (qwk_io in front of the kernels and behind them): what the host
wrote goes up, what the kernels wrote comes back, and nothing else of a buffer changes on either side."""
import ctypes as C

import numpy as np
import pytest

import qwental_amd as q
from helpers import DeviceLayer, run_moe
from qwental_amd import synth

pytestmark = pytest.mark.gpu


def product(oracle, ft, W, N, K, x):
    return oracle.qmv(ft, W, N, K, x, f64=True)


@pytest.mark.parametrize("N,K,nb,yoff,slack", [(16, 256, 1, 0, 0), (33, 512, 3, 52, 7), (640, 256, 16, 16, 100), (9, 256, 2, 4, 1), (4096, 256, 5, 0, 20000)])
def test_rows_inside_a_larger_buffer_leave_the_rest_alone(gpu, oracle, N, K, nb, yoff, slack):
    """y at an offset of a buffer full of the host's own bytes: only the product's bytes change, on the host and in HBM."""
    rng = np.random.default_rng(N + K + nb)
    W = synth.matrix(rng, 8, N, K)
    path = q.Path(gpu, 2048, 512, 512, 10, 16)
    wb, y = gpu.buf_from(W, device_only=True), gpu.buf(yoff + nb * N * 4 + slack)
    xb = gpu.buf(nb * K * 2)
    for it in range(3):  # the input changes under the same address from call to call
        x = synth.activations(rng, nb, K)
        fence = rng.integers(0, 256, y.size, dtype=np.uint8)
        y.view()[:] = fence
        C.memmove(xb.c.ptr, x.ctypes.data, x.nbytes)  # straight into the shadow
        b = gpu.batch()
        path.qmv_gg(b, q.Tensor(wb, 8), N, K, xb, y, nb, yoff=yoff)
        assert b.end() > 0
        got = y.view().copy()
        res = got[yoff:yoff + nb * N * 4].view(np.float32).reshape(nb, N)
        ref = product(oracle, 8, W, N, K, x)
        assert np.abs(res - ref).max() <= 1e-5 * np.abs(ref).max()
        keep = np.ones(y.size, bool)
        keep[yoff:yoff + nb * N * 4] = False
        assert np.array_equal(got[keep], fence[keep])
        assert np.array_equal(y.read(), got)  # HBM holds what the host sees
    for bb in (wb, xb, y):
        bb.free()
    path.close()


def test_gaps_between_strided_rows_keep_the_hosts_bytes(gpu, oracle):
    N, K, nb, stride = 20, 256, 4, 37
    rng = np.random.default_rng(5)
    W, x = synth.matrix(rng, 21, N, K), synth.activations(rng, nb, K)
    ok, err = gpu.compile("#define qmv_gg qmv_gg_gaps\n#define GF 21\n#define KD %d\n#define RB %d\n#define NB %d\n#define YT float\n" % (K, synth.row_bytes(21, K), nb))
    assert ok, err
    wb, xb, y = gpu.buf_from(W, device_only=True), gpu.buf_from(x), gpu.buf(nb * stride * 4)
    v = y.view(np.float32).reshape(nb, stride)
    v[:] = -7.5
    b = gpu.batch()
    b.kernel(gpu.kernel("qmv_gg_gaps"))
    b.buf(0, wb)
    b.buf(3, xb)
    b.buf(4, y)
    b.bytes(5, np.array([N, K, stride, 0], np.uint32))
    b.dispatch(1)
    assert b.end() > 0
    ref = product(oracle, 21, W, N, K, x)
    assert np.abs(v[:, :N] - ref).max() <= 1e-5 * np.abs(ref).max() and (v[:, N:] == -7.5).all()
    for bb in (wb, xb, y):
        bb.free()


@pytest.mark.parametrize("nbuf", [3, 24, 25, 60])
def test_many_buffers_and_many_batches_in_flight(gpu, oracle, nbuf):
    """More pieces than one launch carries, more batches in flight than there are slots, polled and waited for out of order."""
    N, K = 48, 256
    rng = np.random.default_rng(nbuf)
    W = synth.matrix(rng, 8, N, K)
    path = q.Path(gpu, 2048, 512, 512, 10, 16)
    wb = gpu.buf_from(W, device_only=True)
    xs = [synth.activations(rng, 1, K) for _ in range(nbuf)]
    xb, yb = [gpu.buf_from(x) for x in xs], [gpu.buf(N * 4) for _ in xs]
    refs = [product(oracle, 8, W, N, K, x)[0] for x in xs]
    b = gpu.batch()
    for x, y in zip(xb, yb):
        path.qmv_gg(b, q.Tensor(wb, 8), N, K, x, y, 1)
    assert b.end() > 0
    for y, r in zip(yb, refs):
        assert np.abs(y.view(np.float32)[:N] - r).max() <= 1e-5 * np.abs(r).max()
        y.view()[:] = 0
    flight = []
    for x, y in zip(xb, yb):
        b = gpu.batch()
        path.qmv_gg(b, q.Tensor(wb, 8), N, K, x, y, 1)
        gpu.L.qw_batch_submit(b.b)
        flight.append(b)
    while not gpu.L.qw_batch_poll(flight[-1].b):
        pass
    for i in reversed(range(nbuf)):
        assert gpu.L.qw_batch_wait(flight[i].b) > 0
        assert np.abs(yb[i].view(np.float32)[:N] - refs[i]).max() <= 1e-5 * np.abs(refs[i]).max()
    for bb in [wb] + xb + yb:
        bb.free()
    path.close()


def tail_setup(gpu, oracle, rng):
    """A product whose result is the head of a 64 KB buffer that has been up and down once; (record a batch, buffer, tail, check of the head)."""
    N, K, off = 64, 256, 32768
    W, x = synth.matrix(rng, 8, N, K), synth.activations(rng, 1, K)
    path = q.Path(gpu, 2048, 512, 512, 10, 16)
    wb, xb, y = gpu.buf_from(W, device_only=True), gpu.buf_from(x), gpu.buf(65536)
    ref = product(oracle, 8, W, N, K, x)[0]

    def record():
        b = gpu.batch()
        path.qmv_gg(b, q.Tensor(wb, 8), N, K, xb, y, 1)
        return b

    def head_ok():
        return np.abs(y.view(np.float32)[:N] - ref).max() <= 1e-5 * np.abs(ref).max()

    def free():
        for bb in (wb, xb, y):
            bb.free()
        path.close()

    assert record().end() > 0
    return record, y, off, head_ok, free


@pytest.mark.parametrize("how", ["submit", "flush", "end", "dirty"])
def test_hbm_looked_at_holds_what_the_host_wrote_elsewhere(gpu, oracle, how):
    """The host writes the tail of a buffer whose head a batch computes. Read from HBM the tail holds those bytes, and a
    download leaves them alone: between submit and wait, while a flushed part runs, after qw_batch_end, and where the buffer
    was marked dirty in between."""
    rng = np.random.default_rng(9)
    record, y, off, head_ok, free = tail_setup(gpu, oracle, rng)
    for _ in range(3):
        mine = rng.integers(0, 256, y.size - off, dtype=np.uint8)
        y.view()[off:] = mine
        b = record()
        if how == "submit":
            gpu.L.qw_batch_submit(b.b)
            while not gpu.L.qw_batch_poll(b.b):
                pass
        elif how == "flush":
            b.flush()
        else:
            assert b.end() > 0
            if how == "dirty":
                gpu.L.qw_hip_buf_mark_dirty(y.ref())
        if how == "flush":  # (the copy up is behind the flush on the stream: wait for it without waiting for the batch)
            other = record()
            assert other.end() > 0
        assert np.array_equal(y.read(len(mine), off), mine)
        assert gpu.L.qw_hip_buf_download(y.ref(), off, len(mine)) and np.array_equal(y.view()[off:], mine)
        if how == "submit":
            assert gpu.L.qw_batch_wait(b.b) > 0
        elif how == "flush":
            assert b.end() > 0
        assert head_ok() and np.array_equal(y.view()[off:], mine)
    free()


def test_a_kept_device_address_sees_every_later_submit(gpu, oracle):
    """Whoever asked for the address once reads the whole buffer as it was at the last submit, not the bytes of its batch only."""
    rng = np.random.default_rng(10)
    record, y, off, head_ok, free = tail_setup(gpu, oracle, rng)
    addr = gpu.L.qw_hip_buf_devptr(y.ref())
    got = np.empty(y.size - off, np.uint8)
    for _ in range(3):
        mine = rng.integers(0, 256, len(got), dtype=np.uint8)
        y.view()[off:] = mine
        assert record().end() > 0
        assert gpu.L.hipMemcpy(C.c_void_p(got.ctypes.data), C.c_void_p(addr + off), C.c_size_t(len(got)), 2) == 0  # 2: device to host
        assert np.array_equal(got, mine) and head_ok()
    free()


def test_a_result_left_to_a_later_dispatch_keeps_the_hosts_bytes(gpu):
    """moe_gu_gg binds the shared expert's down rows as a result, but the moe_dn_gg of the same batch writes them. A batch
    that ends before it leaves them as the host had them."""
    D, I, E, K, nb = 512, 256, 8, 2, 2
    rng = np.random.default_rng(11)
    m = synth.moe_layer(rng, D, I, E, 8, 8, 8)
    x = synth.activations(rng, nb, D)
    path = q.Path(gpu, D, I, E, K, 16)
    dl = DeviceLayer(gpu, m)
    sel = run_moe(gpu, path, dl, x, nb)[2]  # registers the kernels; its selection record
    k = gpu.kernel("moe_gu_gg_8_8_g1_n2_e%dk%dd%di%d" % (E, K, D, I))
    assert k
    xb, sb, H, psh = gpu.buf_from(x), gpu.buf_from(sel), gpu.buf(2 * (K + 1) * I * 4), gpu.buf(nb * D * 4)
    for _ in range(3):
        mine = rng.standard_normal(nb * D).astype(np.float32)
        psh.view(np.float32)[:] = mine
        b = gpu.batch()
        b.kernel(k)
        for i, bb in ((0, dl.bufs["Wg"]), (1, dl.bufs["Wu"]), (2, dl.bufs["Wsd"]), (3, psh), (4, xb), (5, sb), (6, H)):
            b.buf(i, bb)
        b.bytes(12, np.array([nb], np.uint32))
        b.dispatch(1)
        assert b.end() > 0, gpu.last_error()
        assert np.array_equal(psh.view(np.float32), mine) and np.array_equal(psh.read(dtype=np.float32), mine)
    # with moe_dn_gg and moe_cmb_gg behind it: written for the tokens of the combine, the rows of others computed or left alone
    dn, cmb = (gpu.kernel("%s_8_s4_n2_e%dk%dd%di%d" % (n, E, K, D, I)) for n in ("moe_dn_gg", "moe_cmb_gg"))
    pg, out = gpu.buf(nb * K * D * 4), gpu.buf(nb * D * 2)
    got = {}
    for tokens in (2, 1):
        H.view(np.float16)[:] = np.random.default_rng(12).standard_normal(H.size // 2).astype(np.float16)  # (the shared expert's part is moe_pre_gg's)
        mine = rng.standard_normal(nb * D).astype(np.float32)
        psh.view(np.float32)[:] = mine
        b = gpu.batch()
        b.kernel(k)
        for i, bb in ((0, dl.bufs["Wg"]), (1, dl.bufs["Wu"]), (2, dl.bufs["Wsd"]), (3, psh), (4, xb), (5, sb), (6, H)):
            b.buf(i, bb)
        b.bytes(12, np.array([nb], np.uint32))
        b.dispatch(1)
        b.kernel(dn)
        for i, bb in ((0, dl.bufs["Wd"]), (2, H), (3, sb), (9, pg)):
            b.buf(i, bb)
        b.dispatch(1)
        b.kernel(cmb)
        for i, bb in ((1, psh), (3, sb), (4, out), (9, pg)):
            b.buf(i, bb)
        b.bytes(8, np.array([tokens], np.uint32))
        b.dispatch(1)
        assert b.end() > 0, gpu.last_error()
        got[tokens] = psh.view(np.float32).copy()
        psh.view(np.float32)[:] = rng.standard_normal(nb * D)  # other bytes in HBM before the next one
        b = gpu.batch()
        b.kernel(k)
        for i, bb in ((0, dl.bufs["Wg"]), (1, dl.bufs["Wu"]), (2, dl.bufs["Wsd"]), (3, psh), (4, xb), (5, sb), (6, H)):
            b.buf(i, bb)
        b.bytes(12, np.array([nb], np.uint32))
        b.dispatch(1)
        assert b.end() > 0, gpu.last_error()
    assert np.abs(got[2]).min() > 0 and np.array_equal(got[1][:D], got[2][:D])
    assert np.array_equal(got[1][D:], mine[D:]) or np.array_equal(got[1][D:], got[2][D:])
    for bb in (xb, sb, H, psh, pg, out):
        bb.free()
    dl.free()
    path.close()
