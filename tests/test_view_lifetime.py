"""Buffers of a Spectrometer that was dropped while they are read: a numpy view
holds it; a device address does not (an array library may keep the address for
good), so the newest context that handed one out and was collected stays until
the next is made, and close() frees at once."""
import gc
import weakref

import numpy as np

import rawspec_amd as R


class _Stub(R.Spectrometer):
    """A Spectrometer over plain host memory, without a device."""

    def __init__(self, closed=None):
        super().__init__(Nc=1, Ntpb=8, Nts=[8], Nas=[1], init=False)
        self.mem = np.arange(64, dtype=np.float32)
        self.closed = closed
        self.ctx.h_pwrbuf[0] = R.C.cast(self.mem.ctypes.data, R.C.POINTER(R.C.c_float))
        self.ctx.h_pwrbuf_size[0] = 32

    def close(self):
        if self.closed is not None:
            self.closed.append(self._serial)


def test_context_with_device_addresses_outlives_its_collection():
    closed = []
    a, b, c = _Stub(closed), _Stub(closed), _Stub(closed)
    for sp in (a, b):
        sp.initialized = sp._lent = True      # as device_pwrbuf() leaves it
    serials = [sp._serial for sp in (a, b, c)]
    del sp, a, b, c
    gc.collect()
    # the one that lent nothing and the older of the two are closed
    assert sorted(closed) == [serials[0], serials[2]]
    gc.collect()
    assert len(closed) == 2 and [s._serial for s in R._kept] == [serials[1]]
    d = _Stub(closed)                         # the next context: the kept one goes
    assert closed[-1] == serials[1] and not R._kept and len(closed) == 3
    del d


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
