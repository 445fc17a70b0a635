"""Groups split into 64 and more partial sums, which several threads of the
reduction share: 64 to 512 partials and counts that leave threads without any or
with fewer than eight, outputs that do not fill a workgroup's 32, stores and
additions to the integration; against the FP64 oracle at the FP32 bar."""
import pytest

from tests.spectro_cases import PLAIN_TOL
from tests.test_gpu_hybrid import run

pytestmark = pytest.mark.gpu


# units of 1024 samples in a group: 64, 113, 127, 128 and 231 partials
@pytest.mark.parametrize("units", [256, 449, 505, 509, 923])
@pytest.mark.parametrize("nt, mode, bits", [(128, 1, 8), (128, 4, 16), (1024, -4, 8)])
def test_split_units(nt, mode, bits, units):
    na = units * (1024 // nt)
    assert run(Nc=1, Ntpb=1024 * units, Nts=[nt, nt], Nas=[na, 2 * na], Np=2, bits=bits, pols=[mode] * 2,
               fwd=units % 2 == 0, conj=0, nbuf=2) <= PLAIN_TOL


# points, spectra, channels: few outputs of the vector kernels, odd numbers of them
@pytest.mark.parametrize("nt, na, nc", [(1, 1 << 20, 3), (2, 1 << 18, 1), (10, 4096, 3), (64, 16384, 1), (1000, 1024, 3)])
def test_few_outputs(nt, na, nc):
    assert run(Nc=nc, Ntpb=nt * na, Nts=[nt, nt], Nas=[na, 2 * na], Np=2, bits=16, pols=[1, -4], fwd=True, conj=0,
               nbuf=2) <= PLAIN_TOL
