"""The work the spectrometer is timed on: what a user's program has it do,
through the public entry points of rawspec_amd.Spectrometer.

A case is one stream: its geometry (Nc coarse channels, Np polarisations,
bits per component, Ntpb samples per block), its output products (nts, nas,
pols: transform lengths, spectra per dump, detection modes), how buffers are
handed over (device buffers one or several per call, or host blocks) and the
engine level.  One pass takes `nbuf` device buffers through the context, a
whole number of integrations of every product, and returns the last dump of
each product (and of each incoherent sum), whole, as the consumer finds it.
"""
import math

import numpy as np
import torch

import rawspec_amd as R


def listed():
    return [
        # A narrow stream with short buffers (4 MiB), one call per buffer: the
        # smallest work a call does, where launches and latency count.
        case("power_8ch_1024_call", Nc=8, Ntpb=131072, nts=[1024], nas=[16], pols=[1]),
        # A two-channel stream of a mix of many small ones: few channels, one
        # mid-length transform, each buffer (2 MiB) dumped at once.
        case("crosspol_2ch_65536_call", Nc=2, Ntpb=262144, nts=[65536, 128], nas=[4, 256],
             pols=[4, 1]),
        # A decimal channelisation of a single-polarisation receiver with an
        # odd channel count, inverse transform (a flipped band).
        case("power_13ch_1pol_1000_inverse", Nc=13, Np=1, Ntpb=256000, nts=[1000], nas=[64],
             pols=[1], fwd=False),
        # Search mode: short transforms, short integrations, full Stokes, a
        # dump rate so high that the output is as large as the input.
        case("stokes_64ch_search_256_call", Nc=64, Ntpb=131072, nts=[256], nas=[4], pols=[-4]),
        # The usual three products (high frequency resolution, high time
        # resolution, mid resolution) in full Stokes over a whole 51-buffer
        # integration of 256 MiB buffers, one buffer per call: the granularity
        # of rawspec_start_processing.
        case("stokes_64ch_3products_calls", Nc=64, Ntpb=524288, nts=[1 << 20, 8, 1024],
             nas=[51, 128, 3072], pols=[-4, -4, -4], nbuf=51, tone=True),
        # The same run as a server feeds it: 8 buffers per call, engine level 1.
        case("stokes_64ch_3products_batches_l1", Nc=64, Ntpb=524288, nts=[1 << 20, 8, 1024],
             nas=[51, 128, 3072], pols=[-4, -4, -4], nbuf=51, batch=8, level=1, tone=True),
        # The same three products as total power, level 1, one call per buffer.
        case("power_64ch_3products_calls_l1", Nc=64, Ntpb=524288, nts=[1 << 20, 8, 1024],
             nas=[8, 128, 4096], pols=[1, 1, 1], nbuf=8, level=1),
        # A quarter of the band in the cross-polarised mode, 8 buffers per call.
        case("crosspol_16ch_3products_batch", Nc=16, Ntpb=524288, nts=[1 << 20, 8, 1024],
             nas=[16, 128, 4096], pols=[4, 4, 4], nbuf=16, batch=8),
        # An array: 16 antennas of 16 channels, 16-bit samples, four products,
        # each also summed incoherently over the antennas.
        case("power_16ant_int16_4products_ics", Nc=256, Nant=16, bits=16, Ntpb=262144,
             nts=[64, 4096, 131072, 8], nas=[2048, 32, 4, 16384], pols=[1, 1, 1, 1], nbuf=2,
             sigma=1000.0),
        # One stream of the serving mix: 16-bit, two products of unlike kinds.
        case("stokes_30ch_int16_262144_call", Nc=30, bits=16, Ntpb=262144, nts=[262144, 2048],
             nas=[1, 64], pols=[-4, 1], sigma=300.0),
        # A spectral-line stream: few channels, very long transforms.
        case("power_4ch_8388608_call", Nc=4, Ntpb=1 << 20, nts=[1 << 23], nas=[1], pols=[1]),
        # Blocks in host memory, 4-bit samples expanded on the device, dumps
        # back in host memory: the reference program's own calls.
        case("power_32ch_4bit_host", Nc=32, bits=4, Ntpb=524288, nts=[4096, 64], nas=[32, 2048],
             pols=[1, 1], host=True, sigma=2.5),
    ]


def case(name=None, *, Nc, Ntpb, nts, nas, pols, Np=2, bits=8, Nant=1, nbuf=1, batch=1, level=0,
         fwd=True, host=False, sigma=8.0, tone=False):
    c = dict(Nc=Nc, Np=Np, bits=bits, Nant=Nant, Ntpb=Ntpb, nts=_text(nts), nas=_text(nas),
             pols=_text(pols), nbuf=nbuf, batch=batch, level=level, fwd=fwd, host=host,
             sigma=sigma, tone=tone)
    if name is not None:
        c["name"] = name
    return c


def _text(values):
    return ",".join(str(v) for v in values)


def _ints(text):
    return [int(v) for v in text.split(",")]


def _samples(c):
    """Time samples per channel of one device buffer (Nb blocks)."""
    return max(c["Ntpb"], max(_ints(c["nts"])))


def _nss(c):
    return [_samples(c) // n for n in _ints(c["nts"])]


def _buffer_bytes(c):
    return c["Nc"] * _samples(c) * c["Np"] * 2 * max(c["bits"], 8) // 8


def _dump_floats(c, i):
    nt, na, po, nss = _ints(c["nts"])[i], _ints(c["nas"])[i], _ints(c["pols"])[i], _nss(c)[i]
    q = 4 if c["Np"] == 2 and abs(po) == 4 else 1
    return max(1, nss // na), q, c["Nc"], nt


def draw(rng):
    """A stream of the listed ranges: 1 to 64 channels (odd ones too), buffers
    of 0.5 to 256 MiB, 1 to 3 products of 8 to 2^20 points or a decimal
    length, one or two polarisations, 8 or 16 bits (4 from the host), all
    detection modes, both directions, one or several buffers per call."""
    while True:
        Nc = int(round(2.0 ** rng.uniform(0.0, 6.0)))
        Np = rng.choice([1, 2, 2, 2, 2])
        host = rng.random() < 0.08
        bits = rng.choice([4, 8]) if host else rng.choice([8, 8, 8, 16])
        Nant = rng.choice([1, 1, 1, 1, 2, 4])
        if Nc % Nant:
            continue
        if rng.random() < 0.12:
            big = rng.choice([1000, 1536, 2000])
            nts = [big] + [big // rng.choice([2, 4, 5, 8]) for _ in range(rng.choice([0, 1]))]
            if any(big % n for n in nts):
                continue
        else:
            top = rng.choice([rng.uniform(3.0, 13.0), rng.uniform(12.0, 20.99), 20.0])
            big = 1 << int(top)
            nts = [big] + [1 << rng.randint(3, int(top)) for _ in range(rng.choice([0, 1, 1, 2]))]
        sample = Nc * Np * 2 * max(bits, 8) // 8
        mult = 1 << rng.randint(0, 16)
        if rng.random() < 0.3:
            mult = mult * 3 // 2 if mult > 1 else 3
        Ntpb = big * mult
        size = Ntpb * sample
        if not (1 << 19) <= size <= (1 << 28):
            continue
        nas, nis = [], []
        for n in nts:
            nss = Ntpb // n
            # a host pass is one buffer: its dumps complete within it
            na = rng.choice([k for k in (1, 3, 4, 16, 48, 128, 1024) if nss % k == 0] +
                            ([nss] if host else [nss, 2 * nss, 4 * nss]))
            nas.append(na)
            nis.append(max(1, na // nss))
        nbuf = math.lcm(*nis)
        batch = 1 if host or nbuf == 1 else rng.choice([1, nbuf, 8])
        pols = [rng.choice([1, 4, -4]) if Np == 2 else 1 for _ in nts]
        c = case(Nc=Nc, Np=Np, bits=bits, Nant=Nant, Ntpb=Ntpb, nts=nts, nas=nas, pols=pols,
                 nbuf=nbuf, batch=batch, level=rng.choice([0, 0, 1]) if bits == 8 else 0,
                 fwd=rng.random() < 0.85, host=host,
                 sigma={4: 2.5, 8: 8.0, 16: 500.0}[bits], tone=rng.random() < 0.3)
        if sum(4 * math.prod(_dump_floats(c, i)) for i in range(len(nts))) > (1 << 30):
            continue
        return c


def _weights(c):
    return [0.5 + (a % 8) / 8.0 for a in range(c["Nant"])] if c["Nant"] > 1 else None


def _inputs(c, seed):
    """The device buffers [Nc][samples][Np][re,im] of one pass: Gaussian noise
    with, for some streams, a narrowband tone, in the sample format's range."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    lim = {4: 7, 8: 127, 16: 32767}[c["bits"]]
    S = _samples(c)
    for r in range(c["nbuf"]):
        x = torch.randn((c["Nc"], S, c["Np"], 2), generator=g, device="cuda")
        x.mul_(c["sigma"])
        if c["tone"]:
            t = torch.arange(S, device="cuda", dtype=torch.int64)
            ph = (((t + r * S) * 300) % 1024).to(torch.float64) * (2.0 * math.pi / 1024)
            x[c["Nc"] // 2, :, 0, 0] += (2.5 * c["sigma"] * torch.cos(ph)).to(torch.float32)
            x[c["Nc"] // 2, :, 0, 1] += (2.5 * c["sigma"] * torch.sin(ph)).to(torch.float32)
        x.round_().clamp_(-lim, lim)
        yield x.to(torch.int16 if c["bits"] == 16 else torch.int8)


class _View:
    """A dump in device memory, for torch.as_tensor."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (ptr, False),
                                         "version": 3}


class _State:
    """What the program has in hand: the context, its inputs, its outputs."""

    def __init__(self, c, seed):
        aws = _weights(c)
        extra = dict(incoherently_sum=1, Aws=aws) if aws else {}
        self.sp = R.Spectrometer(Nc=c["Nc"], Ntpb=c["Ntpb"], Nts=_ints(c["nts"]),
                                 Nas=_ints(c["nas"]), Np=c["Np"], Nbps=c["bits"],
                                 Npolout=_ints(c["pols"]), Nant=c["Nant"], record_events=False,
                                 **extra)
        self.host, self.expand4 = c["host"], c["bits"] == 4
        self.dir = R.RAWSPEC_FORWARD_FFT if c["fwd"] else R.RAWSPEC_INVERSE_FFT
        self.batch = c["batch"]
        if self.sp.set_mfma(c["level"]):
            raise RuntimeError("set_mfma")
        n = len(_ints(c["nts"]))
        shapes = [_dump_floats(c, i) for i in range(n)]
        if self.host:
            blocks = self.sp.ctx.Nb
            for x in _inputs(c, seed):
                h = x.cpu().numpy().reshape(c["Nc"], blocks, -1, 2)
                if self.expand4:
                    h = ((h[..., 0] << 4) | (h[..., 1] & 15)).astype(np.uint8)
                for b in range(blocks):
                    raw = np.ascontiguousarray(h[:, b]).reshape(-1).view(np.uint8)
                    self.sp.block(b)[:raw.size] = raw
            self.outputs = [self.sp.pwrbuf(i).reshape(shapes[i]) for i in range(n)]
            if aws:
                self.outputs += [self.sp.icsbuf(i) for i in range(n)]
            return
        self.sp.set_device_output(True)
        self.ring = [x.contiguous() for x in _inputs(c, seed)]
        self.ptrs = [x.data_ptr() for x in self.ring]
        self.outputs = [torch.as_tensor(_View(self.sp.device_pwrbuf(i), shapes[i]), device="cuda")
                        for i in range(n)]
        if aws:
            icsbuf = R.lib().rawspec_amd_device_icsbuf
            for i, (nd, q, nc, nt) in enumerate(shapes):
                self.outputs.append(torch.as_tensor(
                    _View(icsbuf(self.sp.ctx, i), (nd, q, nc // c["Nant"], nt)), device="cuda"))
        torch.cuda.synchronize()


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    sp = state.sp
    if state.host:
        if sp.copy_and_start(sp.ctx.Nb, expand4=state.expand4, fft_dir=state.dir):
            raise RuntimeError("copy_and_start")
        if sp.wait_for_completion():
            raise RuntimeError("wait_for_completion")
        return state.outputs
    p, b = state.ptrs, state.batch
    for k in range(0, len(p), b):
        if b == 1:
            rc = sp.start_processing_device(p[k], state.dir)
        else:
            rc = sp.start_processing_device_batch(p[k:k + b], state.dir)
        if rc:
            raise RuntimeError("start_processing")
    return state.outputs


def work(case):
    """Bytes: every input sample once, every dump that the pass writes once.
    Flops: 5 N log2 N per transform and the detection's sums."""
    c = case
    nbuf = c["nbuf"]
    sample_bytes = 2 * c["Np"] * c["bits"] / 8
    points = float(c["Nc"]) * _samples(c) * nbuf
    moved, flops = points * sample_bytes, 0.0
    for i, (nt, na) in enumerate(zip(_ints(c["nts"]), _ints(c["nas"]))):
        shape = _dump_floats(c, i)
        dumps = nbuf * _samples(c) // nt / max(na, 1) / shape[0]
        moved += max(1.0, dumps) * 4 * math.prod(shape) * (1 + (1 / c["Nant"] if c["Nant"] > 1 else 0))
        flops += points * (c["Np"] * 5 * math.log2(nt) + (16 if shape[1] == 4 else 4 * c["Np"]))
    return {"bytes": moved, "flops": flops}


def _power(x, nt, po, fwd):
    """Detected spectra [Q][Nc][nss][nt] of x [Nc][samples][Np] in 64 bits."""
    nc, s, npol = x.shape
    v = x.reshape(nc, s // nt, nt, npol)
    f = torch.fft.fft(v, dim=2) if fwd else torch.fft.ifft(v, dim=2, norm="forward")
    f = torch.fft.fftshift(f, dim=2)
    p = f.real ** 2 + f.imag ** 2
    if npol == 1 or po == 1:
        return p.sum(dim=3)[None]
    xx, yy = p[..., 0], p[..., 1]
    xy = f[..., 0] * f[..., 1].conj()
    if po == 4:
        return torch.stack([xx, yy, xy.real, xy.imag])
    return torch.stack([xx + yy, xx - yy, xy.real, xy.imag])


def exact(case, seed):
    """The last dump of each product by torch's transforms in 64 bits."""
    c = case
    full = 32767.0 if c["bits"] == 16 else 127.0
    nts, nas, pols, nss = _ints(c["nts"]), _ints(c["nas"]), _ints(c["pols"]), _nss(c)
    out = []
    for i in range(len(nts)):
        nd, q, nc, nt = _dump_floats(c, i)
        out.append(torch.zeros((nd, q, nc, nt), dtype=torch.float64, device="cuda"))
    for r, x in enumerate(_inputs(c, seed)):
        step = max(1, (1 << 23) // (x.shape[1] * x.shape[2]))
        for i in range(len(nts)):
            nis = max(1, nas[i] // nss[i])
            if r < c["nbuf"] - nis:
                continue
            nd, q, nc, nt = _dump_floats(c, i)
            for c0 in range(0, nc, step):
                z = x[c0:c0 + step].to(torch.float64)
                p = _power(torch.view_as_complex(z), nt, pols[i] if c["Np"] == 2 else 1, c["fwd"])
                out[i][:, :, c0:c0 + step] += p.reshape(q, p.shape[1], nd, -1, nt).sum(dim=3).permute(2, 0, 1, 3)
    out = [o / (full * full) for o in out]
    if c["Nant"] > 1:
        w = torch.tensor(_weights(c), dtype=torch.float64, device="cuda")
        for i in range(len(nts)):
            nd, q, nc, nt = out[i].shape
            out.append((out[i].reshape(nd, q, c["Nant"], nc // c["Nant"], nt) *
                        w[None, None, :, None, None]).sum(dim=2))
    if c["host"]:
        out = [o.cpu().numpy() for o in out[:len(nts)]] + [o.cpu().numpy().reshape(-1) for o in out[len(nts):]]
    return out
