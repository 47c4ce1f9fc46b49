"""The blocked grouped product's list of row groups, longest first: every size of group, experts of several groups, more groups than
workgroups, against the product over the GGUF rows (another kernel, another order of sums). Both round G, U and H to binary16
(2^-11); a value that rounds the other way moves an output by no more than that of the largest: within 2e-3, as everywhere."""
import numpy as np
import pytest

import qwental_amd as q
from qwental_amd import synth
from helpers import DeviceLayer, maxrel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,T,K,tm", [("every size", 0, 1, 64), ("every size", 0, 1, 32), ("one expert", 700, 1, 64), ("skewed", 600, 4, 32), ("skewed", 1100, 4, 64)])
@pytest.mark.parametrize("fd,D,I", [(21, 1024, 512), (20, 2560, 640)])
def test_against_gguf_rows(gpu, rows, T, K, tm, fd, D, I):
    E = 128
    rng = np.random.default_rng(T + tm + fd)
    if rows == "every size":  # experts with 1 .. 128 rows
        ids = rng.permutation(np.repeat(np.arange(E), np.arange(1, E + 1)))
        T = ids.size
    elif rows == "one expert":
        ids = np.full(T, 77)
    else:
        ids = synth.zipf_ids(rng, T, E, K)
    m = synth.moe_layer(rng, D, I, E, fgu=21, fd=fd, fsh=21)
    x, w = synth.activations(rng, T, D), rng.uniform(0.1, 1.0, T * K).astype(np.float32)
    out = {}
    for tiled in (True, False):
        gpu.L.qw_hip_set_repack(gpu.g, tiled)
        try:
            dl, path = DeviceLayer(gpu, m, device_only=True), q.Path(gpu, D, I, E, K, 16)
            path.pf_reserve(T, tm)
            xb, ib, wb, ob = gpu.buf_from(x), gpu.buf_from(np.asarray(ids, np.uint32).ravel()), gpu.buf_from(w), gpu.buf(T * D * 2)
            for _ in range(2):
                b = gpu.batch()
                path.pf_moe(b, dl.layer, T, xb, ib, wb, ob)
                assert b.end() >= 0, gpu.last_error()
                got = ob.view(np.float16)[:T * D].reshape(T, D).astype(np.float64)
                assert tiled not in out or np.array_equal(out[tiled], got)
                out[tiled] = got
            for o in (xb, ib, wb, ob):
                o.free()
            path.close()
            dl.free()
        finally:
            gpu.L.qw_hip_set_repack(gpu.g, True)
    assert maxrel(out[True], out[False]) <= 2e-3
