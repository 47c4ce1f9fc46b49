"""The packing of larger steps (qwk_moe_prep_slices): places and packed rows against a stable sort of the pairs, where a token's
pairs fall into several workgroups' slices, where a slice holds many tokens, and with ids outside the table."""
import numpy as np
import pytest

import qwental_amd as q
from qwental_amd import synth
from helpers import DeviceLayer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,D,I,E,bad", [(206, 5, 1024, 256, 32, 0), (333, 7, 2048, 256, 16, 9), (1000, 10, 2048, 256, 64, 0), (4000, 16, 512, 256, 32, 100), (12000, 2, 2048, 256, 16, 5), (1100, 1, 2560, 256, 16, 0)])
def test_places_and_rows(gpu, T, K, D, I, E, bad):
    rng = np.random.default_rng(T + K)
    dl = DeviceLayer(gpu, synth.moe_layer(rng, D, I, E), device_only=True)
    path = q.Path(gpu, D, I, E, K, 16)
    path.pf_reserve(T, 64)
    x = synth.activations(rng, T, D)
    ids = np.argsort(rng.random((T, E)), axis=1)[:, :K].astype(np.uint32).ravel()
    P = T * K
    ids[rng.choice(P, bad, replace=False)] = E + 7  # dropped
    w = rng.uniform(0.1, 1.0, P).astype(np.float32)
    xb, ib, wb, ob = gpu.buf_from(x), gpu.buf_from(ids), gpu.buf_from(w), gpu.buf(T * D * 2)
    b = gpu.batch()
    path.pf_moe(b, dl.layer, T, xb, ib, wb, ob)
    assert b.end() >= 0, gpu.last_error()
    keep = np.flatnonzero(ids < E)
    order = keep[np.argsort(ids[keep], kind="stable")]
    want = np.full(P, 0xFFFFFFFF, np.uint32)
    want[order] = np.arange(order.size)
    assert np.array_equal(path.pf_scratch(3, np.uint32)[:P], want)
    assert np.array_equal(path.pf_scratch(0, np.uint32)[:E], np.bincount(ids[keep], minlength=E))
    rows = path.pf_scratch(4, np.uint16)[:P * D].reshape(P, D)
    assert np.array_equal(rows[:order.size], x.view(np.uint16).reshape(T, D)[order // K])
    for o in (xb, ib, wb, ob):
        o.free()
    path.close()
    dl.free()
