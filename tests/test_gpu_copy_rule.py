"""When the tile-major copies that stay beside their source (Q8_0 and Q4_K gate / up rows, Q8_0 and Q6_K down rows) are made: small ones at
the first dispatch, large ones once the matrix has come often enough; the layer's bits are the same before and after."""
import numpy as np
import pytest

import qwental_amd as q
from qwental_amd import synth
from helpers import DeviceLayer

pytestmark = pytest.mark.gpu
D, I, K = 2048, 512, 10


class Layer:
    """A Q8_0 layer of E experts on a device handle of its own; step() gives its output and what it ran."""

    def __init__(self, E):
        self.g = q.Gpu()
        rng = np.random.default_rng(E)
        m = synth.moe_layer(rng, D, I, E, fgu=8, fd=8, fsh=8, fshd=8)
        self.dl, self.path = DeviceLayer(self.g, m, device_only=True), q.Path(self.g, D, I, E, K, 16)
        self.x = self.g.buf_from(synth.activations(rng, 3, D))
        self.lg, self.sel, self.out = self.g.buf(self.path.logits_bytes(3)), self.g.buf(self.path.sel_bytes(3)), self.g.buf(3 * D * 2)

    def step(self):
        b = self.g.batch()
        self.path.gg_moe(b, self.dl.layer, 3, self.x, self.lg, self.sel, self.out)
        assert b.end() > 0
        return self.out.view(np.uint16).copy()

    def copied(self):
        return self.g.L.qw_hip_packed_bytes(self.g.g)

    def close(self):
        for o in (self.x, self.lg, self.sel, self.out):
            o.free()
        self.dl.free()
        assert self.copied() == 0
        self.path.close()
        self.g.close()


def experts_bytes(E, down_only=False):
    return E * I * D // 32 * 34 * (1 if down_only else 3)


def test_a_large_matrix_is_copied_when_it_has_come_often():
    E = 64  # gate and up together 143 MB: over the line; the down rows, 71 MB, are not
    L = Layer(E)
    one = D * I // 32 * 34  # the shared expert's down rows
    first = L.step()
    assert L.copied() == experts_bytes(E, True) + one  # a layer that is touched once does not pay for a copy of its large matrices
    for _ in range(30):
        assert np.array_equal(L.step(), first)
    assert L.copied() == experts_bytes(E, True) + one
    assert np.array_equal(L.step(), first) and L.copied() == experts_bytes(E) + one  # the thirty-second
    assert np.array_equal(L.step(), first)
    w = L.dl.bufs["Wg"]  # other weights: counted from the start
    w.fill(w.read())
    assert L.copied() == experts_bytes(E, True) + one
    assert np.array_equal(L.step(), first) and L.copied() == experts_bytes(E, True) + one
    L.g.L.qw_hip_set_copy_uses(L.g.g, 1)  # a caller that wants them now
    assert np.array_equal(L.step(), first) and L.copied() == experts_bytes(E) + one
    L.close()


def test_copies_stop_at_their_budget():
    E = 16  # gate and up 36 MB, down 18 MB
    L = Layer(E)
    one = D * I // 32 * 34
    budget = L.g.L.qw_hip_copy_budget(L.g.g, None)
    assert budget == L.g.L.qw_gpu_max_working_set(L.g.g) // 3
    L.g.L.qw_hip_set_copy_budget(L.g.g, experts_bytes(E) - 1)  # all but one byte of the layer
    first = L.step()
    used = q.gpu.C.c_size_t()
    assert L.copied() == experts_bytes(E) - experts_bytes(E, True)
    assert L.g.L.qw_hip_copy_budget(L.g.g, q.gpu.C.byref(used)) == experts_bytes(E) - 1 and used.value == L.copied()
    for _ in range(40):
        assert np.array_equal(L.step(), first)
    assert L.copied() == experts_bytes(E) - experts_bytes(E, True)
    L.g.L.qw_hip_set_copy_budget(L.g.g, budget)
    assert np.array_equal(L.step(), first) and L.copied() == experts_bytes(E) + one
    L.dl.bufs["Wd"].fill(L.dl.bufs["Wd"].read())  # the room of a copy that is dropped is given back
    L.g.L.qw_hip_copy_budget(L.g.g, q.gpu.C.byref(used))
    assert used.value == L.copied() == experts_bytes(E) - experts_bytes(E, True) + one
    L.close()


def test_buffers_may_outlive_the_device():
    """Weights that were counted, and weights that were copied: the device goes first."""
    L = Layer(64)
    L.step()
    L.path.close()
    L.g.close()
    for o in (L.x, L.lg, L.sel, L.out):
        o.free()
    L.dl.free()
