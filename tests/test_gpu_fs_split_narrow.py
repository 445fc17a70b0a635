"""Split four-step pass B where its tiles are narrow: 4 columns at N1 = 1024
(2^19 and 2^20 points), 2 at N1 = 2048 (2^21 points, one polarisation: the
only length beyond 2^20 that a 256-CU device splits).  Every finish mode
against the FP64 oracle at the rule of the other four-step products: a dump
within one call, within a batch, from held buffers, and integrations over
several batches (first, middle, last); runs of equal length and a shorter
last one; and that the reduction ran.
"""
import pytest

from tests.spectro_cases import PLAIN_TOL, check_results, run_device_case

pytestmark = pytest.mark.gpu


def _reduced(Ntpb, nt, na, nbuf):
    """Whether nbuf one-buffer calls launch k_fs_b_reduce."""
    import torch
    import rawspec_amd as R
    with R.Spectrometer(Nc=1, Ntpb=Ntpb, Nts=[nt], Nas=[na], Np=1, Nbps=8) as sp:
        d = torch.zeros(sp.device_input_size(), dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        sp.profile(True)
        for _ in range(nbuf):
            assert sp.start_processing_device(d.data_ptr(), 1) == 0
        return "k_fs_b_reduce" in {k.split(".")[1] for k in sp.profile_report()}


# points, spectra per buffer, spectra per dump, buffers, batches
CASES = {
    "2^21 one call": (21, 8, 8, 1, None),
    "2^21 one call, runs of 5 and 4": (21, 9, 9, 1, None),
    "2^21 batch": (21, 1, 8, 8, [8]),
    "2^21 held": (21, 1, 8, 8, None),
    "2^21 first, middle, last": (21, 1, 24, 24, [8, 8, 8]),
    "2^20 runs of 3 and 2": (20, 5, 5, 1, None),
    "2^20 held": (20, 1, 8, 8, None),
    "2^19 two dumps": (19, 16, 8, 1, None),
}


@pytest.mark.parametrize("name", list(CASES))
def test_narrow_tiles(name):
    lg, per, na, nbuf, batches = CASES[name]
    nt = 1 << lg
    print("case:", name, flush=True)
    assert _reduced(nt * per, nt, na, nbuf)
    res, cfg = run_device_case(Nc=1, Ntpb=nt * per, Nts=[nt], Nas=[na], Np=1, nbuf=nbuf, batches=batches,
                               tone=(0, 20.0, 300.0, 1024.0))
    assert len(res) == 1
    check_results(res, cfg, tol=PLAIN_TOL)
