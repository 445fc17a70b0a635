"""What a caller gets from a Spectrometer keeps the Spectrometer: its buffers
are freed when it is collected, and a view of them read afterwards faults."""
import gc
import weakref

import numpy as np

import rawspec_amd as R


class _Stub(R.Spectrometer):
    """A Spectrometer over plain host memory, without a device."""

    def __init__(self):
        super().__init__(Nc=1, Ntpb=8, Nts=[8], Nas=[1], init=False)
        self.mem = np.arange(64, dtype=np.float32)
        for i in range(1):
            self.ctx.h_pwrbuf[i] = R.C.cast(self.mem.ctypes.data, R.C.POINTER(R.C.c_float))
            self.ctx.h_pwrbuf_size[i] = 32


def test_device_pointer_is_an_int_that_keeps_its_owner():
    sp = _Stub()
    p = R.DevicePointer(4096, sp)
    assert p == 4096 and p + 1 == 4097 and isinstance(p, int)
    ref = weakref.ref(sp)
    del sp
    gc.collect()
    assert ref() is not None
    del p
    gc.collect()
    assert ref() is None


def test_numpy_view_keeps_its_owner():
    sp = _Stub()
    v = sp.pwrbuf(0).reshape(2, 4)
    ref = weakref.ref(sp)
    del sp
    gc.collect()
    assert ref() is not None and v[1, 3] == 7
    del v
    gc.collect()
    assert ref() is None
