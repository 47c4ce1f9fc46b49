"""The blocked grouped product (qwk_pfg_*) and the preparation by slices at the sizes where they can go wrong: row counts around
the groups of 16 and the blocks of 64, tables of every entry size, one and several steps of K, tile counts that do not fill
the last block, tables a caller made by itself."""
import numpy as np
import pytest

import qwental_amd as q
from helpers import DeviceLayer, maxrel
from qwental_amd import synth
from test_gpu_packing import run_case

pytestmark = pytest.mark.gpu
TOL = 2e-3
EDGES = [1, 15, 16, 17, 0, 32, 33, 47, 48, 49, 63, 64, 65, 0, 80, 129]


def edge_ids(rng, topk=1):
    """Token t's first pick so that expert e receives EDGES[e] rows; further picks from experts behind the list."""
    first = rng.permutation(np.repeat(np.arange(len(EDGES)), EDGES))
    rest = [len(EDGES) + np.arange(topk - 1)] * len(first)
    return np.concatenate([first[:, None], np.array(rest).reshape(len(first), topk - 1)], axis=1), len(EDGES) + topk - 1


@pytest.mark.parametrize("tm", [32, 64])
@pytest.mark.parametrize("D,I,fd", [(256, 256, None), (768, 512, None), (512, 640, 20), (1280, 640, 20)])
def test_rows_around_the_blocks(gpu, oracle, tm, D, I, fd):
    """K of one step (256) to three, gate / up tiles of an even and an uneven number of blocks, IQ4_NL down rows."""
    ids, E = edge_ids(np.random.default_rng(D + tm))
    run_case(gpu, oracle, len(ids), ids, E, 1, D, I, 21, tm, D + I + tm, device_only=True, fd=fd)


def test_entries_of_sixteen_rows_taken_together(gpu, oracle):
    """More than 5000 pairs with entries of 16 rows: the blocked kernel takes an expert's entries four at a time."""
    rng = np.random.default_rng(3)
    T, E, K = 640, 24, 8
    ids = synth.zipf_ids(rng, T, E, K)
    assert T * K > 5000
    run_case(gpu, oracle, T, ids, E, K, 256, 256, 21, 16, 33, device_only=True)


@pytest.mark.parametrize("D,I,E,K,T,blocked", [(256, 256, 128, 10, 512, (False, False)), (256, 256, 128, 10, 600, (True, True)), (256, 256, 16, 4, 500, (False, False)),
                                               (256, 256, 16, 4, 520, (True, True)), (256, 2816, 4, 1, 20, (False, True))])
def test_which_kernel_takes_entries_of_sixteen_rows(gpu, oracle, D, I, E, K, T, blocked):
    """The line between the two kernels, (pairs / experts) x (pairs x I) = 2^26, from both sides, with more and with less than
    5000 pairs; rows of more than 2560 values have the blocked kernel alone. The two add up K in different orders, after which
    gate, up, H and the down rows are rounded to binary16: four roundings of 2^-11, TOL."""
    rng = np.random.default_rng(T)
    assert I > 2560 or ((T * K) ** 2 * I >= E << 26) == blocked[0]
    ids = synth.zipf_ids(rng, T, E, K)
    m = synth.moe_layer(rng, D, I, E)
    x = synth.activations(rng, T, D)
    out = []
    dl = DeviceLayer(gpu, m, device_only=True)
    xb, ib = gpu.buf_from(x), gpu.buf_from(ids.ravel())
    wb, ob = gpu.buf_from(np.full(T * K, 1.0 / K, np.float32)), gpu.buf(T * D * 2)
    for tm in (16, 32):  # (from entries of 32 rows on it is always the blocked kernel)
        path = q.Path(gpu, D, I, E, K, 16, device_scratch=True)
        path.pf_reserve(T, tm)
        gpu.profile(True)
        b = gpu.batch()
        path.pf_moe(b, dl.layer, T, xb, ib, wb, ob)
        assert b.end() > 0
        gpu.profile(False)
        ran = [n.startswith("qwk_pfg") for n, _ in gpu.profile_entries() if n.startswith("qwk_pf")]
        assert ran == list(blocked if tm == 16 else (True, True))
        out.append(ob.view(np.float16).astype(np.float64))
        path.close()
    assert maxrel(out[0], out[1]) <= TOL
    for bb in (xb, ib, wb, ob):
        bb.free()
    dl.free()


@pytest.mark.parametrize("T,K", [(1024, 1), (1025, 1), (128, 8), (257, 5), (3000, 1), (513, 16)])
def test_prepared_rows_by_pair_and_by_slice(gpu, oracle, T, K):
    """The preparation on both sides of its limit, with hot experts and experts without a row (values are the other tests')."""
    rng = np.random.default_rng(T + K)
    E, D, I, tm = 40, 256, 256, 16
    ids = synth.zipf_ids(rng, T, E, K)
    m = synth.moe_layer(rng, D, I, E)
    x = synth.activations(rng, T, D)
    path = q.Path(gpu, D, I, E, K, 16, device_scratch=True)
    path.pf_reserve(T, tm)
    dl = DeviceLayer(gpu, m, device_only=True)
    xb, ib = gpu.buf_from(x), gpu.buf_from(ids.ravel())
    wb, ob = gpu.buf_from(np.full(T * K, 1.0 / K, np.float32)), gpu.buf(T * D * 2)
    b = gpu.batch()
    path.pf_moe(b, dl.layer, T, xb, ib, wb, ob)
    assert b.end() > 0
    mt, P = path.pf_max_tiles(), T * K
    counts, offs, _, tiles, _ = oracle.moe_pack(ids.ravel(), E, tm, mt)
    assert np.array_equal(path.pf_scratch(0, np.uint32)[:E], counts) and np.array_equal(path.pf_scratch(1, np.uint32)[:E], offs)
    assert np.array_equal(path.pf_scratch(2, np.uint32)[:4 * mt].reshape(mt, 4), tiles.reshape(mt, 4))
    pos, flat = path.pf_scratch(3, np.uint32)[:P], ids.ravel()
    assert np.array_equal(pos[np.argsort(flat, kind="stable")], np.arange(P))  # experts in order, pairs in order inside
    Xs = path.pf_scratch(4, np.float16)[:P * D].reshape(P, D)
    assert np.array_equal(Xs[pos].view(np.uint16), np.repeat(x, K, axis=0).view(np.uint16))
    for bb in (xb, ib, wb, ob):
        bb.free()
    dl.free()
    path.close()


def test_a_callers_own_table(gpu, oracle):
    """Entries that do not follow each other (a gap between an expert's rows, short entries in the middle, the same expert
    twice, an empty entry): every row of an entry is computed, no other row is touched."""
    E, N, K, M, tm = 5, 272, 512, 300, 32
    entries = [(0, 0, 32), (0, 32, 64), (0, 70, 102), (1, 110, 115), (1, 115, 147), (2, 150, 150), (3, 160, 192), (3, 192, 224), (3, 224, 256), (4, 256, 257), (3, 260, 292)]
    rng = np.random.default_rng(8)
    W, X = synth.matrix(rng, 21, E * N, K), synth.activations(rng, M, K)
    ok, err = gpu.compile("#define IQ_DQ_ONLY\n#define E %d\n#define TOPK 1\n#define D %d\n#define I 256\n#define NB 1\n#define GG_PART 5\n#define PFF 21\n#define KD %d\n#define TM %d\n#define moe_pf_gg pf_own_table\n" % (E, K, K, tm))
    assert ok, err
    wb, xb = gpu.buf_from(W, device_only=True), gpu.buf_from(X)
    table = np.zeros((len(entries) + 3, 4), np.uint32)
    table[:len(entries), :3] = entries
    tb, y = gpu.buf_from(table), gpu.buf(M * N * 2)
    y.view(np.uint16)[:] = 0x7e11  # a NaN of its own
    b = gpu.batch()
    b.kernel(gpu.kernel("pf_own_table"))
    b.buf(0, xb)
    b.buf(1, wb)
    b.buf(4, y)
    b.bytes(5, np.array([M, N], np.uint32))
    b.buf(6, tb)
    b.dispatch((N + 63) // 64, len(table))
    assert b.end() > 0, gpu.last_error()
    got = y.view(np.float16).reshape(M, N)
    rb = synth.row_bytes(21, K)
    ref, on = np.zeros((M, N)), np.zeros(M, bool)
    for e, r0, r1 in entries:
        if r1 > r0:
            ref[r0:r1] = oracle.qmv(21, W.reshape(E, N * rb)[e], N, K, X[r0:r1], f64=True)
            on[r0:r1] = True
    assert maxrel(got[on], ref[on]) <= TOL
    assert (y.view(np.uint16).reshape(M, N)[~on] == 0x7e11).all()
    for bb in (wb, xb, tb, y):
        bb.free()
