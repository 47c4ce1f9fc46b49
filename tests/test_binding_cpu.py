"""The packed form in which the binding hands a tensor to the dense products."""
import ctypes as C

import numpy as np

import qwental_amd as q
from qwental_amd import gpu


class Holder:  # a buffer's C record, without a device
    def __init__(self):
        self.c = gpu.QwBuf()


def test_packed_tensor():
    for ftype, offset in ((1, 0), (30, 16), (21, 2**33 + 110), (np.int64(14), np.int64(4096))):
        t = q.Tensor(Holder(), ftype, offset)
        want = gpu.QwTensor(C.pointer(t.buf.c), int(offset), int(ftype))
        assert gpu._packed(t, []) == bytes(want)

        class Other:  # anything with a c() of its own
            def c(self):
                return want

        keep = []
        assert gpu._packed(Other(), keep) == bytes(want) and keep == [want]
