"""The autotuner times every launch plan that differs, and its report names the
kernel that a small product runs on: the vector kernel, the one that begins on
the matrix cores (hybrid), the mixed-radix kernel, Bluestein's identity or the
matrix-core kernel of levels 1 and 2."""
import re

import pytest

pytestmark = pytest.mark.gpu

LINE = re.compile(r"small( [A-Za-z-]+)? target .*: [\d.]+ ms \(default [\d.]+ ms, (\d+) candidates\)")


def report(level=0, **kw):
    """(kernel, plans timed) per product."""
    import torch
    import rawspec_amd as R
    print("case:", kw, flush=True)
    with R.Spectrometer(**kw) as sp:
        assert sp.set_mfma(level) == 0
        d = torch.zeros(sp.device_input_size(), dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        rep = sp.autotune(d.data_ptr(), 1, 1)
    print("  " + "\n  ".join(rep.strip().splitlines()), flush=True)
    return [((m.group(1) or "").strip(), int(m.group(2))) for m in map(LINE.search, rep.strip().splitlines())]


def test_wavefronts_of_a_workgroup_make_a_plan():
    """256 groups of 8 spectra of 1024 points: one workgroup of 4 wavefronts per
    group (512 and 1024 workgroups wanted), or one of 8 (2048 and more, the
    default).  Both have chunks of the whole group."""
    assert report(Nc=32, Ntpb=1024 * 64, Nts=[1024], Nas=[8], Npolout=[-4]) == [("hybrid", 2)]


KERNELS = {
    # 256-point search products, long and single-spectrum dumps of 1024 points
    "hybrid": (dict(Nc=16, Ntpb=1 << 16, Nts=[256, 1024, 1024], Nas=[4, 64, 1], Npolout=[1, -4, -4]),
               ["hybrid", "hybrid", ""]),
    "int16": (dict(Nc=16, Ntpb=1 << 16, Nbps=16, Nts=[64, 128, 512], Nas=[64, 64, 64], Npolout=[-4, -4, -4]),
              ["", "hybrid", "hybrid"]),
    # from 2^18 points a polarisation and multiples of 10, 20 or 24
    "decimal": (dict(Nc=8, Ntpb=1000000, Nts=[1000, 250, 125], Nas=[1, 4, 1], Npolout=[1, -4, 1]),
                ["mixed-radix", "mixed-radix", "Bluestein"]),
    "tripled": (dict(Nc=8, Ntpb=1536 * 350, Nts=[1536, 12], Nas=[1, 4], Npolout=[1, -4]), ["mixed-radix", "Bluestein"]),
    # engine level 1: unsplit operands from 32 spectra per dump
    "level 1": (dict(level=1, Nc=16, Ntpb=1 << 16, Nts=[1024, 1024, 256], Nas=[64, 8, 4], Npolout=[-4, -4, 1]),
                ["matrix-core", "hybrid", "hybrid"]),
    "short decimal": (dict(Nc=2, Ntpb=16000, Nts=[1000], Nas=[1], Npolout=[1]), ["Bluestein"]),
}


@pytest.mark.parametrize("name", list(KERNELS))
def test_report_names_the_kernel(name):
    kw, kernels = KERNELS[name]
    assert [k for k, _ in report(**kw)] == kernels
