"""Performance cases of the correlator: sectors as its users run them.

A case is one call of a public entry point on one block of frames of two
stations: the ACF/XCF sector on device data (`spectra`), the phased-array sum
with its re-quantised series (`phased`), one chunk of the whole-scan cross
spectrum (`fringe`) and the sector on host buffers (`host`).  Sizes, bit
widths, rates and delay terms are those of bench.py and tests/: FFT
256..65536, 1/2/4/8 bits, 64..1024 Msps, both arithmetic forms, USB and LSB
stations, bit shuffles, band offsets, from a scan's short last sector up to a
full second of 1024 Msps.

Inputs are a correlated Gaussian pair, the second station delayed, quantised
as the station backends do and packed into the stations' words.  `exact`
re-computes a case in 64 bits from the same codes with torch alone.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("fx-corr_amd"))

import fxcorr as F  # noqa: E402

DEV = "cuda"
CHUNK = 1 << 26          # samples of one station generated at a time
MAX_DELAY = 64           # samples station 2 may lag station 1
CHAIN_MIN = 512          # plain form: overlaps above this follow the f32 recurrence

FFTS = (256, 512, 1024, 2048, 4096, 8192, 16384, 32768, 65536)


def _case(kind, form, fft, frames, bits1=2, bits2=2, msps=1024, lsb2=False, shuffle2=False, shift=0,
          delay=5.3, raw=False, first=0, name=None):
    """kind: entry point; form: arithmetic; shift: band offset in bins
    (station 2's bin minus station 1's); delay: residual in samples; raw:
    also write the phased series; first: the sector's first frame."""
    c = dict(kind=kind, form=form, fft=fft, frames=frames, bits1=bits1, bits2=bits2, msps=msps,
             lsb2=lsb2, shuffle2=shuffle2, shift=shift, delay=delay, raw=raw, first=first)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the last, short sector of a 64 Msps scan: launches and host work
        _case("spectra", "plain", 1024, 150, msps=64, delay=37.3, first=62500, name="short_plain_1024"),
        # one second of the 64 Msps survey shape from the reader's host buffers
        _case("host", "chosen", 1024, 62499, msps=64, delay=37.3, name="host_chosen_1024"),
        # one second of 1024 Msps, 2-bit, station 2 LSB with its bit shuffle, in each form
        _case("spectra", "chosen", 1024, 1000000, lsb2=True, shuffle2=True, delay=3.2, first=1000000,
              name="second_chosen_1024"),
        _case("spectra", "plain", 1024, 1000000, lsb2=True, shuffle2=True, delay=3.2, first=1000000,
              name="second_plain_1024"),
        # coarse channels, mixed recorders (8-bit and 1-bit)
        _case("spectra", "chosen", 256, 200001, 8, 1, 256, delay=-7.4, name="mixed_chosen_256"),
        # 4096 channels' worth of a mixed-width scan
        _case("spectra", "chosen", 4096, 50001, 8, 2, 512, shuffle2=True, delay=9.6, name="mixed_chosen_4096"),
        # fine channels in the reference-faithful form
        _case("spectra", "plain", 16384, 8001, 2, 4, 256, lsb2=True, delay=-2.7, name="fine_plain_16384"),
        # spectral-line second: 512 Msps, 4-bit and 1-bit, bands 16 MHz apart
        _case("spectra", "chosen", 65536, 7812, 4, 1, 512, shift=2048, delay=0.3, name="line_chosen_65536"),
        # fringe search over one chunk of the reader
        _case("fringe", "chosen", 8192, 8192, 2, 2, 1024, delay=11.1, name="fringe_chosen_8192"),
        # phased array, reference-faithful series
        _case("phased", "plain", 1024, 100001, 2, 2, 1024, raw=True, delay=2.3, name="phased_plain_1024"),
        # phased array of a mixed pair into an 8-bit series
        _case("phased", "chosen", 4096, 20001, 8, 2, 512, lsb2=True, raw=True, delay=-4.8,
              name="phased_chosen_4096"),
        # phased power of fine channels
        _case("phased", "chosen", 32768, 3001, 2, 1, 512, delay=1.6, name="phased_chosen_32768"),
    ]


def draw(rng):
    kind = rng.choices(("spectra", "phased", "fringe", "host"), (6, 3, 1, 1))[0]
    form = rng.choice(("plain", "chosen"))
    fft = rng.choice(FFTS)
    # samples of one station over their logarithm, up to an eighth of a second of 1024 Msps
    samples = 2.0 ** rng.uniform(17.3, 27.0)
    frames = max(3, int(samples / fft)) + rng.randrange(2)
    shift = 0
    if rng.random() < 0.3:   # another sky centre: whole multiples of 1/32 band, or any bin
        shift = rng.choice((-1, 1)) * rng.choice((fft // 32, rng.randrange(1, fft // 8)))
    return _case(kind, form, fft, frames, rng.choice((1, 2, 2, 4, 8)), rng.choice((1, 2, 2, 4, 8)),
                 rng.choice((64, 128, 256, 512, 1024)), rng.random() < 0.4, rng.random() < 0.4, shift,
                 round(rng.uniform(-12.0, 12.0), 2), kind == "phased" and rng.random() < 0.7,
                 rng.randrange(0, 200000))


# ------------------------------------------------------------------- inputs
def _levels(bits):
    if bits == 2:
        return np.array([-3.0, -1.0, 1.0, 3.0])
    return np.arange(1 << bits, dtype=np.float64) - ((1 << bits) - 1) / 2.0


def _shuffle(case, seed):
    """Station 2's map: decoded bit i is stored bit map[i]."""
    if not case["shuffle2"]:
        return np.arange(32, dtype=np.int32)
    return np.random.default_rng(seed).permutation(32).astype(np.int32)


def _quantise(x, bits):
    if bits == 1:
        return (x >= 0).to(torch.uint8)
    if bits == 2:
        return ((x >= -0.98).to(torch.uint8) + (x >= 0).to(torch.uint8) + (x >= 0.98).to(torch.uint8))
    n = 1 << bits
    return torch.clamp(torch.floor(x * (n / 8.0) + n / 2.0), 0, n - 1).to(torch.uint8)


def _codes(case, seed):
    """Both stations' codes (uint8, frames * fft each), LSB stations' odd
    samples negated before the quantiser.  Blocks hold whole frames."""
    n, total = case["fft"], case["frames"] * case["fft"]
    g = torch.Generator(device=DEV).manual_seed(seed)
    lag = int(abs(case["delay"]))
    rho = 0.1 if case["kind"] == "phased" else 0.02
    out = [torch.empty(total, dtype=torch.uint8, device=DEV) for _ in range(2)]
    for at in range(0, total, CHUNK):
        m = min(CHUNK, total - at)
        common = torch.randn(m + MAX_DELAY, generator=g, device=DEV)
        for st in range(2):
            late = lag if (case["delay"] >= 0) == (st == 1) else 0
            x = torch.randn(m, generator=g, device=DEV)
            x = math.sqrt(1 - rho) * x + math.sqrt(rho) * common[MAX_DELAY - late:MAX_DELAY - late + m]
            if st == 1 and case["lsb2"]:
                x.view(-1, 2)[:, 1].neg_()
            out[st][at:at + m] = _quantise(x, case["bits%d" % (st + 1)])
    return out


def _pack(codes, bits, bit_map):
    """Codes to bytes, first sample in the lowest bits of little-endian
    words; decoded bit i of a word is stored as bit bit_map[i]."""
    per = 8 // bits
    c = codes.view(-1, per)
    by = c[:, 0].clone()
    for j in range(1, per):
        by |= c[:, j] << (bits * j)
    if np.array_equal(bit_map, np.arange(32)):
        return by
    w = by.view(torch.int32)
    o = torch.zeros_like(w)
    for i in range(32):
        o |= ((w >> i) & 1) << int(bit_map[i])
    return o.view(torch.uint8)


def _band(case):
    """(shift, a1s, a1e, a2s) of the overlap of two equal bands."""
    m, sb = case["fft"] // 2, case["shift"]
    a1s = max(0, -sb)
    return sb, a1s, min(m, m - sb), a1s + sb


def _delay(case, seed):
    """Delay-model terms: a drifting geometric table, clocks, fringe rate."""
    rng = np.random.default_rng([seed, 7])
    fs, n = case["msps"] * 1e6, case["fft"]
    points = 2 + int((case["first"] + case["frames"]) * n / fs)
    table = 3e-7 + 4e-12 * np.arange(points) * rng.uniform(-1, 1) + 1e-16 * np.arange(points) ** 2
    seek = round(3e-7 * fs) / fs
    kw = dict(frame_dt=n / fs, fs=fs, time_offset_s=float(rng.integers(0, 60)),
              delay_user_samples=case["delay"] - (3e-7 - seek) * fs + float(rng.uniform(-0.1, 0.1)),
              extra_delay_rate_sps=float(rng.uniform(-1e-11, 1e-11)),
              clock2_delay_s=float(rng.uniform(-0.2, 0.2)) / fs, clock2_rate_sps=1e-13, d_seek=seek,
              lo1_hz=6.7e9, lo2_hz=6.7e9)
    return table, kw


def _products(case):
    if case["kind"] == "phased":
        return F.PRODUCT_PHASED | (F.PRODUCT_RAW_OUT if case["raw"] else 0)
    if case["kind"] == "fringe":
        return F.PRODUCT_XCF
    return F.PRODUCT_ACF | F.PRODUCT_XCF


def _bit_out(case):
    return max(case["bits1"], case["bits2"])


def prepare(case, seed):
    codes = _codes(case, seed)
    bit_map = _shuffle(case, seed)
    raw = [_pack(codes[0], case["bits1"], np.arange(32)), _pack(codes[1], case["bits2"], bit_map)]
    del codes
    n, h = case["fft"], case["fft"] // 2 + 1
    plan = F.Plan(n, bits=(case["bits1"], case["bits2"]),
                  levels=[_levels(case["bits1"]), _levels(case["bits2"])], shuffles=(None, bit_map),
                  lsb=(False, case["lsb2"]), band=_band(case), df_hz=case["msps"] * 1e6 / n,
                  products=_products(case), bit_out=_bit_out(case),
                  precision=F.PRECISION_CHOSEN if case["form"] == "chosen" else F.PRECISION_PLAIN_FP32)
    table, kw = _delay(case, seed)
    s = dict(case=case, plan=plan, cfg=F.make_delay_cfg(table, **kw), raw=raw)
    if case["kind"] == "host":
        s["raw"] = [r.cpu().numpy() for r in raw]
    elif case["kind"] == "fringe":
        s["ac"] = torch.zeros(h, dtype=torch.complex128, device=DEV)
    else:
        s["acc"] = torch.empty((F.N_PRODUCTS, h), dtype=torch.float64, device=DEV)
        if case["raw"]:
            s["series"] = torch.empty(case["frames"] * n * _bit_out(case) // 8, dtype=torch.uint8, device=DEV)
    return s


def run(s):
    case, plan = s["case"], s["plan"]
    nf, first, (raw1, raw2) = case["frames"], case["first"], s["raw"]
    if case["kind"] == "host":
        r = plan.sector_run(raw1, raw2, first, nf, s["cfg"])
        return dict(acf1=r["acc11"], acf2=r["acc22"], xcf=r["acc12"])
    stream = torch.cuda.current_stream().cuda_stream
    if case["kind"] == "fringe":
        ac = s["ac"].zero_()     # a scan's first chunk
        F.fringe_accumulate_device(plan, raw1.data_ptr(), raw2.data_ptr(), first, nf, s["cfg"],
                                   ac.data_ptr(), stream)
        return dict(xcf=ac)
    acc, series = s["acc"], s.get("series")
    plan.sector_run_device(raw1.data_ptr(), raw2.data_ptr(), first, nf, s["cfg"], acc.data_ptr(),
                           None if series is None else series.data_ptr(), stream)
    if case["kind"] == "phased":
        return dict(power=acc[0]) if series is None else dict(power=acc[0], series=series)
    return dict(acf1=acc[1], acf2=acc[2], xcf=acc[3:])


def work(case):
    n, nf = case["fft"], case["frames"]
    h = n // 2 + 1
    fft = 2.5 * n * math.log2(n)
    per_bin = {"phased": 30, "fringe": 20}.get(case["kind"], 26)   # rotations, products, sums
    out = {"phased": 1, "fringe": 2}.get(case["kind"], 4) * h * 8
    flops = nf * (2 * fft + per_bin * h)
    if case["raw"]:
        out += nf * n * _bit_out(case) // 8
        flops += nf * fft
    return {"bytes": nf * n * (case["bits1"] + case["bits2"]) // 8 + out, "flops": flops}


def tolerance(case):
    # FP32 FFTs with FP64 integration: up to 4.4e-7 (2-norm) and 1.2e-6 (one
    # bin) from `exact` over these ranges.  A code of the series may move to
    # its neighbour where a sample lies on a decision boundary: up to 8e-6 of
    # the bytes, or one byte of the shortest series (20 kB).
    return {"rel": 2e-6, "max": 1e-5, "differ": 1e-4}


# ------------------------------------------------------- the same in 64 bits
def _frame_delays(case, seed):
    """Per frame: both stations' integer shifts and fractional delays, and
    the delay that turns the fringe (main.rs:184-241)."""
    table, kw = _delay(case, seed)
    i = np.arange(case["first"], case["first"] + case["frames"], dtype=np.float64)
    local = (i + 0.5) * kw["frame_dt"]
    t = local + kw["time_offset_s"]
    last = len(table) - 1
    i0 = np.minimum(np.floor(local).astype(np.int64), last)
    i1 = np.minimum(i0 + 1, last)
    frac = np.where(i1 == i0, 0.0, np.clip(local - i0, 0.0, 1.0))
    net = (table[i0] * (1.0 - frac) + table[i1] * frac + 0.0 + kw["delay_user_samples"] / kw["fs"] +
           kw["extra_delay_rate_sps"] * t)
    full = net + (kw["clock2_delay_s"] + kw["clock2_rate_sps"] * t)
    tau = full - kw["d_seek"]
    v = tau * kw["fs"]
    shift = (np.sign(v) * np.floor(np.abs(v) + 0.5)).astype(np.int64)   # halves away from zero
    phase = -2.0 * np.pi * kw["lo1_hz"] * full
    phase = np.mod(phase + np.pi, 2.0 * np.pi) - np.pi
    as_dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    return as_dev(shift), as_dev(tau - shift / kw["fs"]), as_dev(phase)


def _polar32(theta):
    """exp(i theta) of an angle rounded to f32, rounded to f32 (as f64)."""
    t = theta.float().double()
    return torch.complex(torch.cos(t).float().double(), torch.sin(t).float().double())


def _phasors(case, start, step, count):
    """(frames, count) phasors start, start * step, ...: angles in 64 bits
    (chosen), or of the f32 start and step: the f32 recurrence of the plain
    form, up to CHAIN_MIN links its powers in 64 bits."""
    k = torch.arange(count, dtype=torch.float64, device=DEV)
    if case["form"] == "chosen":
        a = start[:, None] + step[:, None] * k
        return torch.complex(torch.cos(a), torch.sin(a))
    p, q = _polar32(start), _polar32(step)
    if count <= CHAIN_MIN and case["kind"] != "phased":
        a, r = torch.angle(q)[:, None] * k, torch.abs(q)[:, None] ** k
        return p[:, None] * torch.polar(r, a)
    out = torch.empty((count, len(start), 2), dtype=torch.float32, device=DEV)
    pr, pi, qr, qi = p.real.float(), p.imag.float(), q.real.float(), q.imag.float()
    for b in range(count):
        out[b, :, 0], out[b, :, 1] = pr, pi
        pr, pi = pr * qr - pi * qi, pr * qi + pi * qr
    return torch.view_as_complex(out.double()).T


def _spectrum(codes, bits, lsb, shift, n):
    lv = torch.from_numpy(_levels(bits)).to(DEV)
    x = lv[codes.long()].view(-1, n)
    if lsb:
        x[:, 1::2] *= -1
    if shift is not None:
        src = torch.arange(n, device=DEV)[None, :] - shift[:, None]
        x = torch.where((src >= 0) & (src < n), torch.gather(x, 1, src.clamp(0, n - 1)), 0.0)
    return torch.fft.rfft(x)


def exact(case, seed):
    n, nf, m = case["fft"], case["frames"], case["fft"] // 2
    codes = _codes(case, seed)
    bit_map = np.arange(32)   # the series goes out through station 1's map
    shift, frac, phase = _frame_delays(case, seed)
    fringe = torch.polar(torch.ones_like(phase), phase) if case["form"] == "chosen" else _polar32(phase)
    _, a1s, a1e, a2s = _band(case)
    ov, df = a1e - a1s, case["msps"] * 1e6 / n
    acf1 = torch.zeros(m + 1, dtype=torch.float64, device=DEV)
    acf2, power, xcf = acf1.clone(), acf1.clone(), torch.zeros(m + 1, dtype=torch.complex128, device=DEV)
    series = []
    block = max(1, min(nf, (1 << 24) // n))
    if case["form"] == "plain" and m > CHAIN_MIN:
        block = max(block, min(nf, (1 << 26) // n))    # the recurrence walks all of a block's frames at once
    for at in range(0, nf, block):
        e = min(nf, at + block)
        f = slice(at, e)
        s1 = _spectrum(codes[0][at * n:e * n], case["bits1"], False, shift[f], n)
        s2 = _spectrum(codes[1][at * n:e * n], case["bits2"], case["lsb2"], None, n)
        step = -2.0 * np.pi * df * frac[f]
        if case["kind"] != "phased":
            acf1 += (s1.abs() ** 2).sum(0)
            acf2[a1s:a1e] += (s2[:, a2s:a2s + ov].abs() ** 2).sum(0)
            rot = _phasors(case, step * a1s, step, ov) * fringe[f, None]
            xcf[a1s:a1e] += (s1[:, a1s:a1e] * s2[:, a2s:a2s + ov].conj() * rot).sum(0)
            continue
        s1 = s1 * _phasors(case, 0.0 * step, step, m + 1)
        s1[:, m] = s1[:, m].real.to(s1.dtype)
        s2[:, m] = s2[:, m].real.to(s2.dtype)
        cb = s1 * fringe[f, None]
        cb[:, a1s:a1e] += s2[:, a2s:a2s + ov]
        power += (cb.abs() ** 2).sum(0)
        if case["raw"]:
            t = torch.fft.irfft(torch.cat([cb[:, :1].real.to(cb.dtype), cb[:, 1:m], cb[:, m:].real.to(cb.dtype)], 1),
                                n=n).float().reshape(-1)
            lv = torch.from_numpy(_levels(case["bits1"])).to(DEV).float()
            mids = (lv[1:] + lv[:-1]) / 2     # a sample between two levels takes the lower one
            series.append(_pack(torch.bucketize(t, mids).to(torch.uint8), _bit_out(case), bit_map))
    if case["kind"] == "phased":
        return dict(power=power, series=torch.cat(series)) if case["raw"] else dict(power=power)
    if case["kind"] == "fringe":
        return dict(xcf=xcf / (float(n) * n))
    if case["kind"] == "host":
        return dict(acf1=acf1, acf2=acf2, xcf=xcf)
    return dict(acf1=acf1, acf2=acf2, xcf=torch.stack([xcf.real, xcf.imag]))
