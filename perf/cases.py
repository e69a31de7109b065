"""Performance cases of the pulsar-search chain on one GPU.

Each case is one call (or one short sequence of calls) that a program built on
this package makes again and again: one dedispersion of a full buffer, one
chunk through the channeliser, one chunk through the front end, one whole
step of a beam or of several beams.  Sizes are those of the repository's tests
and benchmark: subbands of 195.3125 kHz below 150 MHz in 16, 64 or 256
channels, 8 taps, Stokes-I integrated over 4 blocks, 128 to 4096 trials up to
50..1000 pc/cm^3, buffers of 4096 to 131072 samples.
"""
import math

import numpy as np
import torch

import __graft_entry__ as entry

FCH1, SUBBAND, T_IN, INTEGRATE, SIGMA = 150.0, 0.1953125, 5.12e-6, 4, 64.0
KDM = 4148.741601
U8_SCALE = 127.0 / 10.0  # quantisation of the clipper's normalised range
MAX_ADDS = 4.3e11        # of the largest listed dedispersion (the LOFAR-size beam)


def listed():
    """The smallest calls first, then the ordinary and the largest ones."""
    return [
        # a quick look at a few subbands: launch latency is what counts
        dict(name="dedisp_small_f32", kind="dedisp", n_sub=8, n_ch=16, tdms=128, dm_hi=50.0, nsamp=4096, dtype="f32"),
        # one buffer of a full LOFAR-size beam, the reference's own workload
        dict(name="dedisp_beam_f32", kind="dedisp", n_sub=62, n_ch=64, tdms=2048, dm_hi=500.0, nsamp=65536,
             dtype="f32"),
        # the same beam from an 8-bit buffer, with the series its detector reads
        dict(name="dedisp_beam_u8", kind="dedisp", n_sub=62, n_ch=64, tdms=2048, dm_hi=500.0, nsamp=65536, dtype="u8"),
        # fine channels, few trials, half-precision buffer, odd trial count
        dict(name="dedisp_256ch_f16", kind="dedisp", n_sub=34, n_ch=256, tdms=517, dm_hi=300.0, nsamp=32768,
             dtype="f16"),
        # coarse channels and a long DM range: trials tens of samples apart
        dict(name="dedisp_wide_f32", kind="dedisp", n_sub=31, n_ch=16, tdms=512, dm_hi=1000.0, nsamp=65536,
             dtype="f32"),
        # module by module from packets, as the reference's pipeline runs it
        dict(name="modules_37x16", kind="modules", n_sub=37, n_ch=16, n_taps=8, n_blk=4096, n_stokes=4),
        # a streaming chunk of a beam through the fused channeliser
        dict(name="ppf_beam_fp32", kind="ppf", n_sub=62, n_ch=64, n_taps=8, n_spec=8192, dft="fp32"),
        # fine channels: plain and split-precision DFT
        dict(name="ppf_256ch_fp32", kind="ppf", n_sub=47, n_ch=256, n_taps=8, n_spec=2048, dft="fp32"),
        dict(name="ppf_256ch_bf16x3", kind="ppf", n_sub=47, n_ch=256, n_taps=8, n_spec=2048, dft="bf16x3"),
        # a streaming chunk through the whole front end: channeliser, clipper
        # in its steady state, buffer fill
        dict(name="front_beam", kind="front", n_sub=62, n_ch=64, n_spec=8192, nsamp=16384, dtype="f32"),
        # one whole step of a LOFAR-size beam with its detection
        dict(name="step_beam_f32", kind="step", n_sub=62, n_ch=64, tdms=2048, dm_hi=500.0, nsamp=65536, dtype="f32"),
        # several different beams stepped together, 8-bit buffers
        dict(name="beams_4_u8", kind="beams", beams=4, tdms=512, dm_hi=200.0, nsamp=16384, dtype="u8", dft="bf16x3"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dedisp"] * 5 + ["ppf"] * 3 + ["front", "step", "beams", "modules"])
    n_ch = rng.choice([16, 64, 256])
    if kind in ("dedisp", "step"):
        while True:
            c = dict(kind=kind, n_sub=_log(rng, 8, 62), n_ch=n_ch, tdms=_log(rng, 128, 4096),
                     dm_hi=float(rng.choice([50, 100, 200, 300, 500, 750, 1000])), nsamp=1 << rng.randint(12, 17),
                     dtype=rng.choice(["f32", "f32", "f16", "u8"]))
            if kind == "dedisp" and rng.random() < 0.25:  # buffers that are no power of two
                c["nsamp"] = c["nsamp"] - rng.randint(1, c["nsamp"] // 4)
            if kind == "step":
                c["nsamp"] = max(c["nsamp"], 16384)
            while c["nsamp"] < 1.25 * _maxshift(c) + 256:
                c["nsamp"] *= 2
            cost = _n_chan(c) * float(c["tdms"]) * _geometry(c)[1]
            # the chain's step also holds its input: at most the LOFAR beam's
            samples = c["n_sub"] * _geometry(c)[1] * float(c["n_ch"])
            if cost <= MAX_ADDS * (0.6 if kind == "step" else 1.0) and samples <= 62 * 52640 * 64:
                return c
    if kind == "ppf":
        c = dict(kind=kind, n_sub=rng.randint(8, 62), n_ch=n_ch, n_taps=rng.choice([4, 8, 8, 8, 16]),
                 n_spec=_log(rng, 16, 524288 // n_ch), dft="fp32")
        if n_ch > 16 and c["n_taps"] == 8:
            c["dft"] = rng.choice(["fp32", "bf16x3", "fp16x2"])
        return c
    if kind == "modules":
        return dict(kind=kind, n_sub=rng.randint(8, 62), n_ch=rng.choice([16, 64]), n_taps=8,
                    n_blk=_log(rng, 128, 8192), n_stokes=rng.choice([1, 4]))
    if kind == "front":
        return dict(kind=kind, n_sub=rng.randint(8, 62), n_ch=rng.choice([16, 64]), n_spec=_log(rng, 256, 8192),
                    nsamp=16384, dtype=rng.choice(["f32", "f16", "u8"]))
    return dict(kind="beams", beams=rng.randint(2, 6), tdms=_log(rng, 128, 1024),
                dm_hi=float(rng.choice([50, 100, 200])), nsamp=16384, dtype=rng.choice(["f32", "f16", "u8"]),
                dft=rng.choice(["fp32", "bf16x3"]))


# ------------------------------------------------------------------ geometry
def _n_chan(c):
    return c["n_sub"] * c["n_ch"]


def _tsamp(c):
    return T_IN * c["n_ch"] * INTEGRATE


def _foff(c):
    return -SUBBAND / c["n_ch"]


def _shifts(c):
    f = FCH1 + _foff(c) * np.arange(_n_chan(c), dtype=np.float64)
    return (KDM * (1.0 / f / f - 1.0 / FCH1 / FCH1)).astype(np.float32)


def _maxshift(c):
    step = np.float32(c["dm_hi"] / c["tdms"])
    return int(float(step * np.float32(c["tdms"] - 1) * _shifts(c)[-1]) / _tsamp(c))


def _geometry(c):
    """(samples that carry over to the next buffer, output samples)."""
    m = _maxshift(c)
    rem = (c["nsamp"] - m) % 224
    return m + rem, c["nsamp"] - m - rem


def _delays(c):
    """[tdms][channel] delays: float32 products, truncated."""
    step = np.float32(c["dm_hi"] / c["tdms"]) / np.float32(_tsamp(c))
    dm = np.arange(c["tdms"], dtype=np.float32) * step
    return (dm[:, None] * _shifts(c)[None, :]).astype(np.int32)


def _beam_cases(c):
    """The beams of a "beams" case: subbands and channels vary from beam to
    beam, each buffer long enough for its beam's delays."""
    out = []
    for k in range(c["beams"]):
        b = dict(c, n_sub=31 + (13 * k) % 32, n_ch=(64, 256, 16)[k % 3])
        while b["nsamp"] < 1.25 * _maxshift(b) + 256:
            b["nsamp"] *= 2
        out.append(b)
    return out


def _filter(c):
    """Prototype FIR, [tap][channel] float32: windowed sinc, centred channels."""
    n = c["n_taps"] * c["n_ch"]
    i = np.arange(n)
    h = np.sinc((i - (n - 1) / 2.0) / c["n_ch"]) * (0.5 - 0.5 * np.cos(2 * np.pi * i / (n - 1))) / c["n_ch"]
    return (h * (-1.0) ** (i % c["n_ch"])).astype(np.float32)


def _bandpass(c, h):
    e = float(np.sum(h.astype(np.float64) ** 2))
    level, std = 4 * INTEGRATE * SIGMA ** 2 * e, 2 * math.sqrt(2 * INTEGRATE) * SIGMA ** 2 * e
    n = _n_chan(c)
    return np.array([n, FCH1, FCH1 + _foff(c) * (n - 1), _foff(c), std, level], np.float64)


# -------------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _voltages(n_sub, n_ch, n_samp, g, impulses=False):
    """[sub][pol][sample][re, im] int16: noise with a narrowband carrier in a
    few subbands and, with impulses, 0.5 % of the integrated samples at 20 sigma."""
    out = torch.empty((n_sub, 2, n_samp, 2), dtype=torch.int16, device="cuda")
    spi = n_ch * INTEGRATE
    loud = torch.rand(n_samp // spi + 1, generator=g, device="cuda") < 0.005
    gain = (1.0 + 19.0 * loud.float()).repeat_interleave(spi)[:n_samp] * SIGMA
    for s in range(n_sub):
        x = torch.randn((2, n_samp, 2), generator=g, device="cuda")
        x *= gain[None, :, None] if impulses else SIGMA
        if s % 8 == 3:
            ph = (torch.arange(n_samp, device="cuda") % n_ch).float() * (2 * math.pi * ((s % n_ch) / n_ch - 0.5))
            x += 1.5 * SIGMA * torch.stack((ph.cos(), ph.sin()), -1)[None]
        out[s] = x.round_().clamp_(-32768, 32767).to(torch.int16)
    return out


def _series_input(c, g):
    """A full dedispersion buffer: the clipper's normalised spectra, a few of
    them rejected (far below), and for u8 the offsets of those rows."""
    n, ns = _n_chan(c), c["nsamp"]
    low = torch.rand(ns, generator=g, device="cuda") < 0.005
    if c["dtype"] == "u8":
        x = torch.empty((n, ns), dtype=torch.uint8, device="cuda")
        for a in range(0, n, 1024):
            b = min(a + 1024, n)
            y = torch.randn((b - a, ns), generator=g, device="cuda").mul_(U8_SCALE).round_().clamp_(-127, 127).add_(128)
            x[a:b] = y.masked_fill_(low[None, :], 128.0).to(torch.uint8)
        off = torch.where(low, -2500.0 - torch.rand(ns, generator=g, device="cuda"), torch.zeros(ns, device="cuda"))
        return x, off
    x = torch.randn((n, ns), generator=g, device="cuda")
    x.masked_fill_(low[None, :], -2500.0)
    return (x.half() if c["dtype"] == "f16" else x), None


# ----------------------------------------------------------------- the cases
def prepare(case, seed):
    ppl = entry.load_package()
    ppl.init(0)
    g = _generator(seed)
    c, k = case, case["kind"]
    s = dict(case=case, ppl=ppl)
    if k == "dedisp":
        s["plan"] = ppl.DedispPlan(_n_chan(c), c["nsamp"], c["tdms"], 0.0, c["dm_hi"] / c["tdms"], _tsamp(c), FCH1,
                                   _foff(c), dtype=c["dtype"])
        s["x"], s["off"] = _series_input(c, g)
        n_out = s["plan"].nout
        s["out"] = torch.empty((c["tdms"], n_out), dtype=s["plan"].out_dtype(), device="cuda")
        if c["dtype"] == "u8":
            s["series"] = torch.empty((c["tdms"], n_out), dtype=torch.float32, device="cuda")
    elif k == "ppf":
        n_blk = c["n_spec"] * INTEGRATE
        s["ppf"] = ppl.PPF(c["n_sub"], c["n_ch"], c["n_taps"], _filter(c), precision=c["dft"], integrate=INTEGRATE)
        s["volt"] = _voltages(c["n_sub"], c["n_ch"], n_blk * c["n_ch"], g)
        s["out"] = torch.empty((c["n_spec"], c["n_sub"], 1, c["n_ch"]), device="cuda")
        run(s)  # the stream goes on: the filter's history is the chunk's own end
    elif k == "modules":
        # packets of 16 samples: [packet][header | sub][t][pol][re, im]
        n_pkt = c["n_blk"] * c["n_ch"] // 16
        s["ppf"] = ppl.PPF(c["n_sub"], c["n_ch"], c["n_taps"], _filter(c))
        s["packets"] = (torch.randn((n_pkt, 8 + c["n_sub"] * 64), generator=g, device="cuda") * SIGMA).round_().to(
            torch.int16)
        run(s)
    elif k == "front":
        h = _filter(dict(c, n_taps=8))
        s["ppf"] = ppl.PPF(c["n_sub"], c["n_ch"], 8, h, integrate=INTEGRATE)
        s["clip"] = ppl.Clipper(_bandpass(c, h))
        s["buf"] = ppl.DDBuffer(_n_chan(c), c["nsamp"], 3000, c["dtype"], U8_SCALE)
        # past the clipper's first 10000 spectra, which fill its history
        n = 2560
        v = _voltages(c["n_sub"], c["n_ch"], n * INTEGRATE * c["n_ch"], g)
        for _ in range(4):
            s["clip"].run(s["ppf"].stokes_i16(v, n * INTEGRATE))
        s["volt"] = _voltages(c["n_sub"], c["n_ch"], c["n_spec"] * INTEGRATE * c["n_ch"], g, impulses=True)
        s["stokes"] = torch.empty((c["n_spec"], c["n_sub"], 1, c["n_ch"]), device="cuda")
    elif k == "step":
        h = _filter(dict(c, n_taps=8))
        s["chain"] = ppl.BeamChain(c["n_sub"], c["n_ch"], 8, h, INTEGRATE, _bandpass(c, h), c["nsamp"], c["tdms"],
                                   0.0, c["dm_hi"] / c["tdms"], _tsamp(c), FCH1, _foff(c), dtype=c["dtype"],
                                   inv_scale=U8_SCALE)
        n_prime = s["chain"].overlap * INTEGRATE * c["n_ch"]
        s["chain"].prime(_voltages(c["n_sub"], c["n_ch"], n_prime, g))
        s["volt"] = _voltages(c["n_sub"], c["n_ch"], s["chain"].samples_per_step(), g, impulses=True)
    else:
        specs = []
        for b in _beam_cases(c):
            h = _filter(dict(b, n_taps=8))
            specs.append(ppl.BeamSpec(b["n_sub"], b["n_ch"], 8, h, INTEGRATE, _bandpass(b, h), b["nsamp"], b["tdms"],
                                      0.0, b["dm_hi"] / b["tdms"], FCH1, _foff(b)))
        # a fresh buffer's worth of data per step; each chunk is fed as a continuous stream
        s["mb"] = ppl.MultiBeam(specs, dtype=c["dtype"], inv_scale=U8_SCALE, dft=c["dft"], max_chunk_samples=1 << 20)
        s["volt"] = [_voltages(sp.n_sub, sp.n_ch, s["mb"].chunk_samples(b), g) for b, sp in enumerate(specs)]
        s["mb"].prime(s["volt"])
        s["mb"].step(s["volt"])  # past most of the clippers' learning
    return s


def run(s):
    ppl, c = s["ppl"], s["case"]
    k = c["kind"]
    if k == "dedisp":
        s["plan"].run(s["x"], d_out=s["out"])
        if c["dtype"] != "u8":
            return s["out"]
        s["plan"].u8_series(s["out"], s["off"], 1.0 / U8_SCALE, d_out=s["series"])
        return s["out"], s["series"]
    if k == "ppf":
        return s["ppf"].stokes_i16(s["volt"], c["n_spec"] * INTEGRATE, d_out=s["out"])
    if k == "modules":
        n_pkt = s["packets"].shape[0]
        x = ppl.ingest(s["packets"], n_pkt, c["n_sub"], 16, header_bytes=16)
        spec = s["ppf"].spectra_c32(x, c["n_blk"])
        st = ppl.stokes(spec, c["n_stokes"])
        return x, spec, st, ppl.integrate(st, INTEGRATE)
    if k == "front":
        s["ppf"].stokes_i16(s["volt"], c["n_spec"] * INTEGRATE, d_out=s["stokes"])
        s["clip"].run(s["stokes"])
        rows = s["stokes"].view(c["n_spec"], _n_chan(c))
        done = 0
        while done < c["n_spec"]:
            used, full = s["buf"].add(rows, first=done)
            done += used
            if full:
                s["buf"].rotate()
        filled = s["buf"].tensor()
        filled.owner = s["buf"]  # the view does not keep the buffer's memory by itself
        return s["stokes"], filled
    if k == "step":
        s["chain"].step(s["volt"])
        ints, vals, count = s["chain"].detect()
        seen = s["chain"].series if c["dtype"] == "u8" else s["chain"].out
        return seen, ints, vals, count
    s["mb"].step(s["volt"])
    return list(s["mb"].series if c["dtype"] == "u8" else s["mb"].outs)


# ------------------------------------------------------- work and tolerances
def _ppf_work(n_sub, n_ch, n_taps, n_blk, in_bytes=4):
    """Samples in, and the FIR, DFT and power operations of the blocks."""
    n = 2 * n_sub * n_blk * n_ch
    return n * in_bytes, n * (4 * n_taps + 5 * math.log2(n_ch) + 4)


def work(case):
    c, k = case, case["kind"]
    elem = {"f32": 4, "f16": 2, "u8": 1}.get(c.get("dtype"), 4)
    if k == "dedisp":
        n_out = _geometry(c)[1]
        outs = 2 if c["dtype"] == "u8" else 1
        return {"bytes": _n_chan(c) * c["nsamp"] * elem + c["tdms"] * n_out * 4 * outs,
                "flops": _n_chan(c) * c["tdms"] * float(n_out)}
    if k == "ppf":
        b, f = _ppf_work(c["n_sub"], c["n_ch"], c["n_taps"], c["n_spec"] * INTEGRATE)
        return {"bytes": b + c["n_spec"] * _n_chan(c) * 4, "flops": f}
    if k == "modules":
        n = _n_chan(c) * c["n_blk"]
        b, f = _ppf_work(c["n_sub"], c["n_ch"], c["n_taps"], c["n_blk"])
        # packets in; samples, spectra, Stokes and integrated Stokes out
        return {"bytes": b + 2 * n * 16 + n * c["n_stokes"] * 4 * (1 + 1 / INTEGRATE), "flops": f}
    if k == "front":
        b, f = _ppf_work(c["n_sub"], c["n_ch"], 8, c["n_spec"] * INTEGRATE)
        return {"bytes": b + c["n_spec"] * _n_chan(c) * (4 + elem), "flops": f}
    total = {"bytes": 0.0, "flops": 0.0}
    for b in [c] if k == "step" else _beam_cases(c):
        n_out = _geometry(b)[1]
        by, fl = _ppf_work(b["n_sub"], b["n_ch"], 8, n_out * INTEGRATE)
        total["bytes"] += by + b["tdms"] * n_out * 4
        total["flops"] += fl + _n_chan(b) * b["tdms"] * float(n_out)
    return total


def tolerance(case):
    """Dedispersion sums channels in order: the same bits from every
    implementation.  The channeliser's filter and transform are 32-bit sums
    (or products of split 16-bit parts) whose order is free: 1.2e-7, 2.5e-6
    and 2e-4 from 64 bits.  What follows the clipper is normalised, so that
    difference grows (2.4e-6 between the plain and the three-product
    transform); in 8 bits a value now and then falls on the other side of a
    step, and a short series shows it (7e-4 at those two transforms)."""
    k = case["kind"]
    if k == "dedisp":
        return "exact"
    if k in ("ppf", "modules"):
        return {"rel": {"fp32": 5e-7, "bf16x3": 1e-5, "fp16x2": 8e-4}[case.get("dft", "fp32")]}
    return {"rel": 1e-3 if case["dtype"] == "u8" else 1e-5}


def _exact_spectra(x, h, n_ch, n_taps):
    """[sub][pol][block][channel] complex128 spectra of a periodic stream."""
    n_sub, _, n_samp, _ = x.shape
    z = torch.view_as_complex(x.double()).view(n_sub, 2, n_samp // n_ch, n_ch)
    h = torch.from_numpy(h.astype(np.float64)).to(x.device).view(n_taps, n_ch)
    y = torch.zeros_like(z)
    for t in range(n_taps):
        y += torch.roll(z, n_taps - 1 - t, dims=2) * h[t]
    return torch.fft.fft(y, dim=-1)


def exact(case, seed):
    c, k = case, case["kind"]
    g = _generator(seed)
    if k == "dedisp":
        n_out = _geometry(c)[1]
        if _n_chan(c) * c["tdms"] * float(n_out) > 4e10:
            return None  # over 20 seconds
        x, off = _series_input(c, g)
        d = torch.from_numpy(_delays(c).astype(np.int64)).cuda()
        t = torch.arange(n_out, device="cuda")
        out = torch.zeros((c["tdms"], n_out), dtype=torch.float64, device="cuda")
        extra = torch.zeros_like(out) if off is not None else None
        for ch in range(_n_chan(c)):
            at = t[None, :] + d[:, ch, None]
            out += x[ch].double()[at]
            if extra is not None:
                extra += off.double()[at]
        if extra is None:
            return out
        return out.to(torch.int64), (out - 128.0 * _n_chan(c)) / U8_SCALE + extra
    if k == "ppf":
        n_blk = c["n_spec"] * INTEGRATE
        x = _voltages(c["n_sub"], c["n_ch"], n_blk * c["n_ch"], g)
        h = _filter(c)
        out = torch.empty((c["n_spec"], c["n_sub"], 1, c["n_ch"]), dtype=torch.float64, device="cuda")
        for s in range(c["n_sub"]):
            z = _exact_spectra(x[s:s + 1], h, c["n_ch"], c["n_taps"])[0]
            p = (z.real ** 2 + z.imag ** 2).sum(0).view(c["n_spec"], INTEGRATE, c["n_ch"])
            out[:, s, 0] = p.sum(1)
        return out
    if k == "modules":
        n_pkt = c["n_blk"] * c["n_ch"] // 16
        pk = (torch.randn((n_pkt, 8 + c["n_sub"] * 64), generator=g, device="cuda") * SIGMA).round_()
        x = pk[:, 8:].view(n_pkt, c["n_sub"], 16, 2, 2).permute(1, 3, 0, 2, 4).reshape(c["n_sub"], 2, n_pkt * 16, 2)
        z = _exact_spectra(x, _filter(c), c["n_ch"], c["n_taps"]).permute(2, 0, 1, 3).contiguous()
        zx, zy = z[:, :, 0], z[:, :, 1]
        px, py = zx.abs() ** 2, zy.abs() ** 2
        st = [px + py]
        if c["n_stokes"] == 4:
            cross = zx * zy.conj()
            st += [px - py, 2 * cross.real, 2 * cross.imag]
        st = torch.stack(st, 2)
        n = c["n_blk"] // INTEGRATE
        integ = st[:n * INTEGRATE].view(n, INTEGRATE, c["n_sub"], c["n_stokes"], c["n_ch"]).sum(1)
        return x.double(), torch.view_as_real(z), st, integ
    # the clipper's decisions are a recurrence over every earlier spectrum: no
    # plain form of it in 64 bits is quick
    return None
