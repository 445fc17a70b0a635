"""Error of long integrations at the FP32 level, against 64-bit transforms and
sums of the same samples (torch, in float64): the root mean square over all bins
of |gpu - ref| / max(bin, mean bin) of total power.

The bar: the constants' common rounding (2^-24 = 0.6e-7) and a chain of 64
additions of equal terms, whose roundings (2.4e-8 rms each, on sums that grow
evenly) leave sqrt(64 / 3) * 2.4e-8 = 1.1e-7, the transforms' own errors averaging
out over the 32 and more spectra: sqrt(0.6^2 + 1.1^2) = 1.3e-7, and an eighth for
the spread of constants and tones: 1.5e-7.  Chains of 256 additions (2.2e-7 and
more) miss it."""
import pytest

pytestmark = pytest.mark.gpu

TOL = 1.5e-7

# points, spectra per dump, dumps, channels, pols, bits
CASES = {
    # pass B over 32 spectra in one run: 32 terms, not the 128 products
    "2^17 two pols": (1 << 17, 32, 1, 12, 2, 8),
    # 128 runs of single spectra, added by k_fs_b_reduce
    "8192 one pol": (8192, 128, 1, 1, 1, 8),
    "8192 two pols": (8192, 128, 1, 1, 2, 8),
    # 256 partial sums of 4 spectra, added by k_reduce
    "1024 one channel": (1024, 1024, 1, 1, 2, 8),
    # long groups in plenty: whole ones of 8 units a wavefront, shared ones of 16,
    # 32 and 64; long groups in chunks
    "64 points, 64 units": (64, 1024, 32, 64, 1, 8),
    "64 points, 64 units, two pols": (64, 1024, 32, 64, 2, 8),
    "128 points, 32 units": (128, 256, 64, 32, 2, 8),
    "128 points int16, 32 units": (128, 256, 64, 32, 2, 16),
    "256 points, 8 units": (256, 32, 256, 8, 2, 8),
    "256 points, 64 units": (256, 256, 64, 32, 2, 8),
    "1024 points, 64 units": (1024, 64, 64, 32, 2, 8),
    "1024 points int16, 64 units": (1024, 64, 64, 32, 2, 16),
    "512 points, 256 units": (512, 512, 4, 128, 2, 8),
}


def rms_error(nt, na, ng, nc, npol, bits):
    import torch
    import rawspec_amd as R
    S, lim = nt * na * ng, 127 if bits == 8 else 32767
    g = torch.Generator(device="cuda")
    g.manual_seed(5 + nt)
    x = torch.randn((nc, S, npol, 2), generator=g, device="cuda") * (20.0 if bits == 8 else 3000.0)
    x = x.round_().clamp_(-lim, lim).to(torch.int8 if bits == 8 else torch.int16)
    torch.cuda.synchronize()
    with R.Spectrometer(Nc=nc, Ntpb=S, Nts=[nt], Nas=[na], Np=npol, Nbps=bits) as sp:
        assert sp.start_processing_device(x.data_ptr(), 1) == 0 and sp.wait_for_completion() == 0
        out = torch.from_numpy(sp.pwrbuf(0).copy()).to("cuda").reshape(ng, nc, nt).double()
    total = 0.0
    for c in range(nc):
        z = torch.view_as_complex(x[c].double()).reshape(ng, na, nt, npol)
        f = torch.fft.fftshift(torch.fft.fft(z, dim=2), dim=2)
        ref = (f.real ** 2 + f.imag ** 2).sum(dim=(1, 3)) / (lim * lim)
        r = (out[:, c] - ref) / torch.maximum(ref, ref.mean(dim=1, keepdim=True))
        total += float(r.square().sum())
    return (total / (ng * nc * nt)) ** 0.5


@pytest.mark.parametrize("name", list(CASES))
def test_long_integrations(name):
    print("case:", name, flush=True)
    e = rms_error(*CASES[name])
    print(f"  rms {e:.2e}", flush=True)
    assert e <= TOL
