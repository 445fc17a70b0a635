"""Short transforms in long dumps on both sides of the lines where a group takes
32 or 64 of a workgroup's slots instead of 16 (few wavefronts; a slot keeps 4
spectra, or 8 with a quarter of the device's wavefronts), with ragged last rounds
and groups that leave slots without one; against the FP64 oracle at the FP32
bar."""
import pytest

from tests.spectro_cases import PLAIN_TOL
from tests.test_gpu_hybrid import run

pytestmark = pytest.mark.gpu


# points, spectra per dump, dumps, channels
CASES = [(1, 127, 96, 3), (1, 128, 2048, 3), (1, 512, 512, 3), (2, 255, 64, 4), (4, 256, 33, 5), (4, 1024, 8, 4),
         (8, 128, 512, 4), (8, 130, 64, 2), (8, 1000, 16, 3), (16, 128, 512, 16), (16, 509, 7, 2), (32, 512, 16, 8)]


@pytest.mark.parametrize("np_, mode, bits", [(1, 1, 8), (2, -4, 8), (2, 4, 16)])
@pytest.mark.parametrize("nt, na, ng, nc", CASES)
def test_slots_of_a_group(nt, na, ng, nc, np_, mode, bits):
    assert run(Nc=nc, Ntpb=nt * na * ng, Nts=[nt], Nas=[na], Np=np_, bits=bits, pols=[mode], fwd=na % 2 == 0,
               conj=0) <= PLAIN_TOL
