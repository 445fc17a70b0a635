"""GPU parity of the mixed-radix small kernel (lengths 2^a 3^b and 2^a 5^b, the
lengths the reference plans with cuFFT, rawspec_gpu.cu:1182-1195), against the
FP64 oracle at the FP32 bar of the other lengths.  A transform of N points
rounds about log2 N times, as Bluestein's and the power-of-two kernels do, so
their tolerance holds unchanged.  Each buffer holds enough points for this
kernel to take the product (2^18 a polarisation); the lengths take every radix of all
families first, in the middle and last, workgroups of 1 to 16 spectra that
are not full wavefronts, dumps of one spectrum (sums from registers), of a few,
and split over workgroups.
"""
import pytest

from tests.spectro_cases import PLAIN_TOL, check_results, run_case

pytestmark = pytest.mark.gpu

CASES = {
    # stages 5,20,20 / 10,10,10 / 20,20: one and several spectra per workgroup
    "2000_stokes": dict(Nc=4, Ntpb=2000 * 136, Nts=[2000, 1000, 400], Nas=[1, 34, 680], Npolout=[-4, -4, -4]),
    # 4,20,20 / 2,20,20 / 4,20
    "1600_full_int16": dict(Nc=3, Ntpb=1600 * 220, Nts=[1600, 800, 80], Nas=[20, 440, 2], Npolout=[4, 1, 4], Nbps=16),
    # 4,4,4,20 / 2,4,4,20 / 2,4,20 / 2,20
    "1280_power": dict(Nc=5, Ntpb=1280 * 96, Nts=[1280, 640, 160, 40], Nas=[96, 3, 64, 1], Npolout=[1, 1, 1, 1]),
    # 8,8,24 / 2,8,24 / 4,24
    "1536_stokes": dict(Nc=7, Ntpb=1536 * 100, Nts=[1536, 384, 96], Nas=[50, 1, 1600], Npolout=[-4, 4, -4]),
    # 3,3,3,3,24 / 3,3,3,24 / 3,3,24 / 3,24
    "1944_power_inverse": dict(Nc=4, Ntpb=1944 * 72, Nts=[1944, 648, 216, 72], Nas=[9, 1, 81, 1944], Npolout=[1] * 4,
                               fft_dir=-1),
    # 3,24,24 / 3,12,24 / 12,24 / 6,24 with four sums
    "1728_full_inverse": dict(Nc=6, Ntpb=1728 * 104, Nts=[1728, 864, 288, 144], Nas=[8, 208, 16, 1], Npolout=[4, -4, 4, -4],
                              fft_dir=-1),
    # 5,5,5,10 / 5,5,10 / 5,10
    "1250_stokes": dict(Nc=6, Ntpb=1250 * 160, Nts=[1250, 250, 50], Nas=[16, 1, 1000], Npolout=[-4, 4, 1]),
    # 10,10,10 / 5,10,10 / 10,10 / 10,20 of one polarisation, integrated over two buffers
    "500_one_pol": dict(Nc=3, Ntpb=1000 * 96, Nts=[1000, 500, 100, 200], Nas=[192, 4, 960, 1], Npolout=[1] * 4, Np=1),
}


@pytest.mark.parametrize("name", list(CASES))
def test_mixed_radix(name):
    print("case:", name, flush=True)
    kw = dict(CASES[name])
    res, cfg, _ = run_case(nbuf=2, tone=(1, 20.0, 33.0, float(kw["Nts"][0])), **kw)
    w = check_results(res, cfg, tol=PLAIN_TOL)
    print(f"  {name}: worst {w}", flush=True)
