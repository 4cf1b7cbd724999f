"""The wave kernel (N = 256..8192 off the producer/consumer kernels) against
the oracle: every size, both stage-1 forms, code widths, shuffles and LSB
input, shifts inside and past the staging padding and past the frame, band
offsets on both grids, product subsets, ragged last rounds, and the frame
counts on both sides of its line against the Stockham kernel."""
import ctypes
import functools

import numpy as np
import pytest

import fxcorr as F
import fxref as R
from _cases import gpu_run, make_case, oracle_run, spectra_err
from _synth import LEVELS_2BIT

pytestmark = pytest.mark.gpu
ACF, XCF, OV = F.PRODUCT_ACF, F.PRODUCT_XCF, F.PRODUCT_ACF_OVERLAP_ONLY
PERM = np.random.default_rng(4).permutation(32).astype(np.int32)
SWAP = np.arange(32, dtype=np.int32) ^ 1


@functools.lru_cache(None)
def line(n):
    """Longest ACF/XCF sector (frames) that stays on the Stockham kernel on this device."""
    p = F.Plan(n, levels=[LEVELS_2BIT, LEVELS_2BIT], df_hz=64e6 / n)
    lo, hi = 0, 1 << 16
    while hi - lo > 1:
        mid = (lo + hi) // 2
        lo, hi = (lo, mid) if F.lib().fxc_internal_wave_for(p.h, ctypes.c_int64(mid)) else (mid, hi)
    assert 0 < lo < 1 << 15
    return lo


def check(c, form):
    plain = form == "plain"
    g = gpu_run(c, F.PRECISION_PLAIN_FP32 if plain else F.PRECISION_CHOSEN)
    o = oracle_run(c, R.MODE_F32 if plain else R.MODE_F64)
    errs = spectra_err(g, o)   # bars of the two forms, as everywhere in the parity tests
    assert g["n_failed"] == 0 and all(e < (1e-5 if plain else 1e-4) for e in errs.values()), errs
    for k in ("acc11", "acc22", "acc12"):
        assert np.array_equal(g[k] == 0, o[k] == 0), k


@pytest.mark.parametrize("form", ["plain", "chosen"])
@pytest.mark.parametrize("n,extra", [(256, 0), (256, 1), (256, 70), (512, 13), (1024, 1), (1024, 260), (2048, 3),
                                     (4096, 1), (4096, 2), (8192, 1), (8192, 0), (8192, 515)])
def test_wave_sizes(n, extra, form):
    # band offset of one bin: also the chosen form leaves the producer/consumer kernels
    c = make_case(n=n, fs=64e6, nf=line(n) + extra, rho=0.2, seed=n + extra, band=(1, 0, n // 2 - 1, 1),
                  delay_user_samples=5.3, extra_delay_rate_sps=3e-8, lo1_hz=6.7e9, lo2_hz=6.7e9)
    check(c, form)


@pytest.mark.parametrize("form", ["plain", "chosen"])
@pytest.mark.parametrize("n", [256, 512, 1024, 2048, 4096, 8192])
@pytest.mark.parametrize("bits,shuffles,lsb,shift,grid,delay,products", [
    ((1, 8), (None, PERM), (False, True), 0, 0, -70.6, ACF | XCF),
    ((8, 2), (PERM, None), (True, False), 5, 1, 33.2, ACF | XCF),
    ((4, 1), (SWAP, PERM), (True, True), -7, 0, 64.9, ACF | XCF | OV),
    ((2, 4), (None, SWAP), (False, False), 32, 1, -31.7, XCF),
    ((2, 2), (None, None), (False, True), 0, 1, 129.4, ACF),
])
def test_wave_options(n, bits, shuffles, lsb, shift, grid, delay, products, form):
    m = n // 2
    a1s = max(0, -shift)
    band = (shift, a1s, min(m, m - shift), a1s + shift)
    c = make_case(n=n, fs=64e6, nf=line(n) + 9, bits=bits, shuffles=shuffles, lsb=lsb, band=band, grid=grid,
                  products=products, rho=0.3, seed=n, delay_samples=3.0, delay_user_samples=delay,
                  lo1_hz=1.2e9, lo2_hz=1.2e9)
    check(c, form)


@pytest.mark.parametrize("n", [256, 2048, 4096, 8192])
def test_wave_shift_past_the_frame(n):
    """Station 1 shifted out of most frames: the sweep crosses +-N."""
    fs = 64e6
    c = make_case(n=n, fs=fs, nf=line(n) + 5, rho=0.3, seed=3, delay_user_samples=-1.2 * n, lo1_hz=1e9, lo2_hz=1e9,
                  extra_delay_rate_sps=2.4 * n / fs / ((line(n) + 5) * n / fs))
    check(c, "plain")


@pytest.mark.parametrize("n,form", [(256, "plain"), (1024, "plain"), (2048, "plain"), (4096, "chosen"), (8192, "plain"),
                                    (8192, "chosen")])
def test_wave_grid_divisors(n, form):
    """The autotuner's configurations of this kernel (variant 0), and the
    Stockham kernel's radix-16 variant on the same sector."""
    plain = form == "plain"
    c = make_case(n=n, fs=64e6, nf=2 * line(n) + 77, rho=0.3, seed=n, delay_user_samples=2.3, lo1_hz=3e9)
    o = oracle_run(c, R.MODE_F32 if plain else R.MODE_F64)
    for variant, div in ((0, 1), (0, 2), (0, 4)) + (((1, 1),) if n >= 2048 else ()):
        p = F.Plan(n, bits=c["bits"], levels=c["levels"], band=c["band"], df_hz=c["fs"] / n, products=c["products"],
                   precision=F.PRECISION_PLAIN_FP32 if plain else F.PRECISION_CHOSEN)
        F.plan_set_tuning(p, variant=variant, grid_divisor=div)
        errs = spectra_err(gpu_run(c, plan=p), o)
        assert all(e < (1e-5 if plain else 1e-4) for e in errs.values()), (variant, div, errs)


@pytest.mark.parametrize("form", ["plain", "chosen"])
@pytest.mark.parametrize("n,nf,shift,grid", [(256, 3001, 3, 0), (512, 1300, -5, 1), (1024, 30_000, 0, 0),
                                             (2048, 1025, -1, 1), (4096, 6001, 0, 1), (8192, 1500, 7, 0)])
def test_wave_phased_both_stations_delayed(n, nf, shift, grid, form):
    """The analytic delay model gives both stations a delay (two rotation
    chains per frame in the plain form); the larger sectors take two chunks."""
    m, fs = n // 2, 64e6
    a1s = max(0, -shift)
    c = make_case(n=n, fs=fs, nf=nf, bits=(2, 4), shuffles=(None, PERM), lsb=(True, False),
                  band=(shift, a1s, min(m, m - shift), a1s + shift), grid=grid, rho=0.4, delay_samples=3.0,
                  products=F.PRODUCT_PHASED | F.PRODUCT_RAW_OUT, seed=n, no_table=True, net_d1_base=4.4 / fs,
                  total_rate1_base=1e-9, net_d2_base=-2.7 / fs, total_rate2_base=-2e-9, lo1_hz=1.5e9, lo2_hz=1.4e9)
    w, plain = (0.8, 1.1), form == "plain"
    p = F.Plan(n, bits=c["bits"], levels=c["levels"], shuffles=c["shuffles"], lsb=c["lsb"], band=c["band"],
               df_hz=fs / n, products=c["products"], out_grid=grid, w=w, bit_out=4,
               precision=F.PRECISION_PLAIN_FP32 if plain else F.PRECISION_CHOSEN)
    g = p.sector_run(c["raw1"], c["raw2"], 0, nf, F.make_delay_cfg(c["table"], **c["delay"]))
    desc = dict(fft_len=n, bits1=2, bits2=4, levels1=c["levels"][0], levels2=c["levels"][1],
                shuffle1=c["shuffles"][0], shuffle2=c["shuffles"][1], lsb1=1, lsb2=0, a1s=c["band"][1],
                a1e=c["band"][2], a2s=c["band"][3], out_grid=grid, df_hz=fs / n, need_acf=0, need_xcf=0,
                need_phased=1, write_raw=1, w1=w[0], w2=w[1], bit_out=4, output_lsb=0, cpu_threads=8)
    o = R.sector_run(desc, c["raw1"], c["raw2"], 0, nf, R.make_delay_cfg(c["table"], **c["delay"]),
                     mode=R.MODE_F32 if plain else R.MODE_F64, threads=8)
    # power: the forms' bars; codes: a byte holds two, each may flip at a decision boundary (1e-4 of codes)
    assert np.max(np.abs(g["acc_ph"] / o["acc_ph"] - 1)) < (1e-5 if plain else 1e-4)
    assert np.count_nonzero(g["raw_out"] != o["raw_out"]) <= 2e-4 * o["raw_out"].size + 2


@pytest.mark.parametrize("n,form,products,small,large", [
    (4096, "chosen", ACF | XCF, 0, 3000), (1024, "plain", ACF | XCF, 700, 5000), (4096, "plain", XCF, 3000, 1500),
    (2048, "chosen", F.PRODUCT_PHASED, 0, 3000), (1024, "plain", F.PRODUCT_PHASED | F.PRODUCT_RAW_OUT, 9000, 2500),
    (16384, "plain", ACF | XCF, 900, 600), (16384, "plain", ACF, 0, 600), (16384, "plain", F.PRODUCT_PHASED, 700, 600)])
def test_capture_without_room_to_grow(n, form, products, small, large):
    """A captured call runs where the plan's scratch may not grow: as the
    plan's first call (small = 0) or after an eager call of another length;
    also while the graph is alive.  Against an eager call on a fresh plan."""
    fs, m = 64e6, n // 2
    raw = bool(products & F.PRODUCT_RAW_OUT)
    c = make_case(n=n, fs=fs, nf=max(small, large), rho=0.3, seed=n, no_table=True, net_d1_base=4.4 / fs,
                  total_rate1_base=1e-9, band=(0, 0, m, 0) if n > 4096 else (1, 0, m - 1, 1))
    cfg, prec = F.make_delay_cfg(c["table"], **c["delay"]), (F.PRECISION_PLAIN_FP32 if form == "plain" else
                                                             F.PRECISION_CHOSEN)
    s = F.Stream()
    r1, r2 = F.DeviceBuffer(c["raw1"].size), F.DeviceBuffer(c["raw2"].size)
    r1.upload(c["raw1"])
    r2.upload(c["raw2"])

    def plan():
        return F.Plan(n, bits=c["bits"], levels=c["levels"], band=c["band"], df_hz=fs / n, products=products,
                      bit_out=2, precision=prec)

    keep = []   # buffers stay until the end

    def run(p, nf):
        acc, out = F.DeviceBuffer(F.N_PRODUCTS * p.half * 8), F.DeviceBuffer(max(8, nf * n // 4))
        keep.extend((acc, out))
        return acc, lambda: p.sector_run_device(r1.ptr, r2.ptr, 0, nf, cfg, acc.ptr,
                                                     **(dict(d_raw_out=out.ptr) if raw else {}), stream=s.ptr)

    p, q = plan(), plan()
    acc_q, call_q = run(q, large)
    call_q()
    if small:
        run(p, small)[1]()
    s.sync()
    want = acc_q.download(np.zeros(F.N_PRODUCTS * q.half))
    acc, call = run(p, large)
    g = F.Graph(s)
    call()
    g.end()
    acc2, eager = run(p, large)
    for _ in range(2):
        g.launch()
        eager()
        s.sync()
        for a in (acc, acc2):   # either path: the form's bar on the spectrum's scale
            got = a.download(np.zeros(F.N_PRODUCTS * p.half))
            assert np.max(np.abs(got - want)) < (1e-5 if form == "plain" else 1e-4) * np.max(np.abs(want))
    g.close()
