"""Dump groups of the kernel that begins on the matrix cores (64 to 1024 points)
whose units of 1024 samples no halving divides: the chunks cover the group, the
last one with fewer units than the others (one to three workgroup rounds, idle
wavefronts), and k_reduce adds a number of partial sums that is no multiple of
eight.  Against the FP64 oracle at the bar of test_gpu_hybrid.py, integrations
over two buffers among them; and that the group was split."""
import re

import pytest

from tests.spectro_cases import PLAIN_TOL
from tests.test_gpu_hybrid import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [8, 16])
@pytest.mark.parametrize("np_, mode", [(1, 1), (2, 1), (2, 4), (2, -4)])
@pytest.mark.parametrize("nt, units", [(128, 9), (256, 41), (512, 75), (1024, 131)])
def test_uneven_chunks(nt, units, np_, mode, bits):
    unit = 1024 // nt
    fwd = (units + bits // 8) % 2 == 0
    # one group a buffer; two groups; one over two buffers
    assert run(Nc=2, Ntpb=1024 * units * 2, Nts=[nt, nt, nt], Nas=[2 * units * unit, units * unit, 4 * units * unit],
               Np=np_, bits=bits, pols=[mode] * 3, fwd=fwd, conj=0, nbuf=2) <= PLAIN_TOL


@pytest.mark.parametrize("nt, units", [(64, 923), (256, 923), (1024, 61)])
def test_long_odd_groups_are_split(nt, units):
    import torch
    import rawspec_amd as R
    print("case:", nt, units, flush=True)
    with R.Spectrometer(Nc=1, Ntpb=1024 * units, Nts=[nt], Nas=[1024 // nt * units], Np=1) as sp:
        d = torch.zeros(sp.device_input_size(), dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        rep = sp.autotune(d.data_ptr(), 1, 1)
    print(" ", rep.strip(), flush=True)
    m = re.search(r"hybrid target .*\(chunk (\d+), ", rep)
    # at most 16 units a chunk, whichever target was fastest
    assert m and int(m.group(1)) <= 16 * 1024 // nt
