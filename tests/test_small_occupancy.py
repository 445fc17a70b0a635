"""Wavefronts per SIMD of the vector kernel's short transforms (no GPU needed: the
compiler's figures of the built library).  They are bound by loads in flight, so
a write-out that holds many partial sums at once must not cost a wavefront."""
import csv
import os

import pytest

TSV = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rawspec_amd", "_build",
                   "kernel_resources.tsv")


@pytest.mark.parametrize("n, bits, waves", [(8, 8, 7), (32, 8, 5), (32, 16, 5)])
@pytest.mark.parametrize("mode", [4, -4])
def test_short_stokes_transforms(n, bits, waves, mode):
    if not os.path.exists(TSV):
        pytest.skip("the library was not built here")
    m = f"Li{mode}" if mode > 0 else f"Lin{-mode}"
    name = f"7k_smallILi{n}ELi{bits}ELi2E{m}ELb0EE"
    with open(TSV) as f:
        rows = [r for r in csv.DictReader(f, delimiter="\t") if name in r["kernel"]]
    assert len(rows) == 1
    assert int(rows[0]["Occupancy [waves/SIMD]"]) >= waves
