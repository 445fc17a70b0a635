"""Transforms whose first 32 points run on the matrix cores, against the FP64
oracle on full-range random codes (the most negative one included) with a
strong tone: the fused small kernel of 64 to 1024 points at the edges of its
launch plans (many short groups per wavefront, a ragged last one, one to
several units per wavefront, chunks with partial sums, two chunks in one
workgroup, integrations over buffers) for both sample widths, one and two
pols, all modes, both directions.

The bar is the FP32 engine's: 1e-5 of the total power of the bin or of the
channel's mean, whichever is larger (four-step products: the rule of
spectro_cases.check_results, five times a single-precision reference's
error where that is more)."""
import numpy as np
import pytest

import oracle as O
from tests.spectro_cases import PLAIN_TOL, check_results, rel_err, run_device_case

pytestmark = pytest.mark.gpu


def codes(n, Nc, Np, bits, seed):
    """[Nc][n][Np][2] codes: uniform over the whole range in channel 0, noise
    with a tone in the others, and a scattering of the most negative code."""
    rng = np.random.default_rng(seed)
    lim = 1 << (bits - 1)
    x = rng.normal(0.0, lim / 16, (Nc, n, Np, 2))
    ph = 2 * np.pi * 0.1375 * np.arange(n)
    x[1:, :, 0, 0] += lim / 3 * np.cos(ph)
    x[1:, :, 0, 1] += lim / 3 * np.sin(ph)
    x[0] = rng.integers(-lim, lim, (n, Np, 2))
    x = np.clip(np.rint(x), -lim, lim - 1)
    x[rng.random(x.shape) < 1e-3] = -lim
    return x.astype(np.int16 if bits == 16 else np.int8)


def run(*, Nc, Ntpb, Nts, Nas, Np, bits, pols, fwd, conj, nbuf=1, seed=3):
    import torch
    import rawspec_amd as R
    No = len(Nts)
    cfg = O.make_cfg(No=No, Np=Np, Nc=Nc, Ntpb=Ntpb, Nbps=bits, Npolout=pols, Nts=Nts, Nas=Nas,
                     input_conjugated=conj)
    assert O.derive(cfg) == 0
    sp = R.Spectrometer(Nc=Nc, Ntpb=Ntpb, Nts=Nts, Nas=Nas, Np=Np, Nbps=bits, Npolout=pols,
                        input_conjugated=conj, record_events=False)
    n = sp.ctx.Nb * Ntpb
    st = O.State(cfg)
    worst = 0.0
    print(f"case: Nc {Nc} Ntpb {Ntpb} Nts {Nts} Nas {Nas} Np {Np} bits {bits} pols {pols} "
          f"fwd {fwd} conj {conj} nbuf {nbuf}", flush=True)
    last = {}
    for b in range(nbuf):
        h = codes(n, Nc, Np, bits, seed + b)
        d = torch.from_numpy(h.reshape(-1).view(np.uint8).copy()).to("cuda")
        assert sp.start_processing_device(d.data_ptr(), 1 if fwd else -1) == 0
        assert sp.wait_for_completion() == 0
        _, ref, _ = st.process(h.reshape(-1), 1 if fwd else -1)
        for i in ref:
            last[i] = 1
            e = rel_err(sp.pwrbuf(i), ref[i], cfg.Nds[i], abs(cfg.Npolout[i]), Nc, Nts[i],
                        cfg.Npolout[i])
            worst = max(worst, float(e.max()))
    sp.close()
    st.close()
    assert len(last) == No, "a product made no dump"
    print(f"  worst {worst:.2e}", flush=True)
    return worst


@pytest.mark.parametrize("bits", [8, 16])
@pytest.mark.parametrize("np_, mode", [(1, 1), (2, 1), (2, 4), (2, -4)])
@pytest.mark.parametrize("nt", [64, 128, 256, 512, 1024])
def test_lengths_and_plans(nt, np_, mode, bits):
    fwd = (nt // 64 + bits) % 2 == 0
    unit = 1024 // nt
    # one unit per group, groups in plenty (ragged over the wavefronts)
    assert run(Nc=3, Ntpb=nt * unit * 701, Nts=[nt], Nas=[unit], Np=np_, bits=bits, pols=[mode],
               fwd=fwd, conj=0) <= PLAIN_TOL
    # few long groups: chunks with partial sums over two buffers; a group of
    # an odd number of units, which no chunk halves; groups shorter than a
    # unit, which another kernel takes
    s = 1024 * 30
    assert run(Nc=2, Ntpb=s, Nts=[nt, nt, nt], Nas=[2 * (s // nt), 15 * unit, 1], Np=np_, bits=bits,
               pols=[mode] * 3, fwd=not fwd, conj=1, nbuf=2) <= PLAIN_TOL


def test_two_chunks_share_a_workgroup():
    # 256 groups of 8 units: two chunks each fill the device
    for mode, bits in ((-4, 8), (1, 16)):
        assert run(Nc=32, Ntpb=1024 * 64, Nts=[1024], Nas=[8], Np=2, bits=bits, pols=[mode], fwd=True,
                   conj=0) <= PLAIN_TOL


@pytest.mark.parametrize("bits", [8, 16])
@pytest.mark.parametrize("np_", [1, 2])
@pytest.mark.parametrize("lg", [13, 14, 15, 16, 17, 18])
def test_fourstep_first_pass(lg, np_, bits):
    nt = 1 << lg
    for level in (0, 1):
        fwd = 1 if (lg + bits // 8 + level) % 2 else -1
        modes = [-4, 4] if np_ == 2 else [1, 1]
        kw = dict(Nc=3, Ntpb=2 * nt, Nts=[nt, nt], Nas=[1, 6], Np=np_, Nbps=bits, Npolout=modes, nbuf=3,
                  batches=[1, 2], fft_dir=fwd, conj=level, seed=lg, sigma=8.0 if bits == 8 else 900.0,
                  tone=(1, 20.0, 300.0, 1024.0), mfma=level)
        print(f"case: {kw}", flush=True)
        res, cfg = run_device_case(**kw)
        check_results(res, cfg, tol_by_product={0: 1e-3, 1: 1e-3} if level else None)


@pytest.mark.parametrize("np_, mode", [(1, 1), (2, 1), (2, -4)])
@pytest.mark.parametrize("nt", [1, 2, 4, 8, 16, 32, 2048, 4096])
def test_int8_lengths_in_fp16_up_to_the_first_exchange(nt, np_, mode):
    # the vector kernel's int8 lengths: whole groups, one spectrum per dump
    s = 8192 * 3
    for fwd in (True, False):
        assert run(Nc=2, Ntpb=s, Nts=[nt, nt], Nas=[s // nt // 3, 1], Np=np_, bits=8,
                   pols=[mode] * 2, fwd=fwd, conj=0) <= PLAIN_TOL
