"""The plain form's ACF/XCF on the fused four-step (N = 16384 / 32768 / 65536,
band shift a multiple of 128) against the oracle's f32 branch and against the
general path (variant 0): every code width's decode, shuffles, LSB input, both
grids, product subsets, ragged iterations and last chunks, shifts past the frame, and
the frame counts on both sides of the line between the two."""
import numpy as np
import pytest

import fxcorr as F
import fxref as R
from _cases import make_case, oracle_run, spectra_err

pytestmark = pytest.mark.gpu
ACF, XCF, OV = F.PRODUCT_ACF, F.PRODUCT_XCF, F.PRODUCT_ACF_OVERLAP_ONLY
PERM = np.random.default_rng(4).permutation(32).astype(np.int32)
SWAP = np.arange(32, dtype=np.int32) ^ 1
LINE = 512   # frames


@pytest.mark.parametrize("n,extra,chunk,bits,shuffles,lsb,shift,grid,delay,products", [
    (16384, 1, 1024, (2, 2), (None, None), (False, False), 0, 0, 5.3, ACF | XCF),
    (16384, 45, 64, (1, 8), (None, PERM), (False, True), 128, 1, -70.6, ACF | XCF),
    (16384, 0, 33, (4, 2), (PERM, None), (True, False), -4096, 0, 33.2, ACF | XCF | OV),
    (16384, -1, 1024, (2, 4), (None, SWAP), (False, False), 0, 1, 16500.0, XCF),
    (16384, 9, 131, (8, 1), (SWAP, PERM), (True, True), -128, 1, 1.5, ACF),
    (16384, 2, 300, (3, 5), (PERM, None), (False, True), 0, 0, 12.2, ACF | XCF),
    (32768, 3, 512, (2, 2), (None, None), (False, False), 0, 0, -31.7, ACF | XCF),
    (32768, 41, 99, (4, 1), (SWAP, PERM), (True, True), -256, 1, 64.9, ACF | XCF),
    (32768, 0, 100, (8, 2), (None, PERM), (False, True), 15744, 0, 2.5, XCF),
    (65536, 23, 131, (1, 4), (PERM, None), (False, True), 2048, 0, -40.7, ACF | XCF | OV),
    (65536, 0, 100, (2, 8), (SWAP, None), (True, True), -128, 1, 129.4, ACF | XCF),
])
def test_plain_fused(n, extra, chunk, bits, shuffles, lsb, shift, grid, delay, products):
    m, nf = n // 2, LINE + extra
    a1s = max(0, -shift)
    c = make_case(n=n, fs=256e6, nf=nf, bits=bits, shuffles=shuffles, lsb=lsb,
                  band=(shift, a1s, min(m, m - shift), a1s + shift), grid=grid, products=products, rho=0.3,
                  seed=n + nf, delay_samples=3.0, delay_user_samples=delay, lo1_hz=1.2e9, lo2_hz=1.2e9)
    o = oracle_run(c, R.MODE_F32)
    for variant in (1, 0):
        p = F.Plan(n, bits=bits, levels=c["levels"], shuffles=shuffles, lsb=lsb, band=c["band"], df_hz=256e6 / n,
                   products=products, out_grid=grid)
        F.plan_set_tuning(p, variant=variant, split_m1=128, chunk_frames=chunk)
        g = p.sector_run(c["raw1"], c["raw2"], 0, nf, F.make_delay_cfg(c["table"], **c["delay"]))
        errs = spectra_err(g, o)   # the plain form's bar, as everywhere in the parity tests
        assert g["n_failed"] == 0 and all(e < 1e-5 for e in errs.values()), (variant, errs)
        for k in ("acc11", "acc22", "acc12"):
            assert np.array_equal(g[k] == 0, o[k] == 0), (variant, k)


@pytest.mark.parametrize("n,extra,chunk,shift,grid,raw,table", [
    (16384, 1, 1024, 0, 0, True, False), (16384, 45, 64, -128, 1, True, False), (16384, 0, 107, 4096, 0, False, True),
    (32768, 3, 512, 0, 1, True, True), (32768, 41, 99, 256, 0, True, False), (32768, -1, 101, -2048, 1, False, False),
    (65536, 19, 101, -128, 1, True, False), (65536, 0, 144, 15744, 0, False, True)])
def test_plain_phased_fused(n, extra, chunk, shift, grid, raw, table):
    """The phased sum likewise, with both stations delayed (two rotation
    chains per frame) and with the geometric table (station 2 has none)."""
    m, fs, nf = n // 2, 256e6, LINE + extra
    a1s = max(0, -shift)
    prods = F.PRODUCT_PHASED | (F.PRODUCT_RAW_OUT if raw else 0)
    model = (dict(delay_user_samples=4.4, extra_delay_rate_sps=1e-9) if table else
             dict(no_table=True, net_d1_base=4.4 / fs, total_rate1_base=1e-9, net_d2_base=-2.7 / fs,
                  total_rate2_base=-2e-9))
    c = make_case(n=n, fs=fs, nf=nf, bits=(2, 4), shuffles=(None, PERM), lsb=(True, False),
                  band=(shift, a1s, min(m, m - shift), a1s + shift), grid=grid, rho=0.4, delay_samples=3.0,
                  products=prods, seed=n + nf, lo1_hz=1.5e9, lo2_hz=1.4e9, **model)
    w = (0.8, 1.1)
    desc = dict(fft_len=n, bits1=2, bits2=4, levels1=c["levels"][0], levels2=c["levels"][1],
                shuffle1=c["shuffles"][0], shuffle2=c["shuffles"][1], lsb1=1, lsb2=0, a1s=c["band"][1],
                a1e=c["band"][2], a2s=c["band"][3], out_grid=grid, df_hz=fs / n, need_acf=0, need_xcf=0,
                need_phased=1, write_raw=1, w1=w[0], w2=w[1], bit_out=4, output_lsb=0, cpu_threads=8)
    o = R.sector_run(desc, c["raw1"], c["raw2"], 0, nf, R.make_delay_cfg(c["table"], **c["delay"]),
                     mode=R.MODE_F32, threads=8)
    for variant in (1, 0):
        p = F.Plan(n, bits=c["bits"], levels=c["levels"], shuffles=c["shuffles"], lsb=c["lsb"], band=c["band"],
                   df_hz=fs / n, products=prods, out_grid=grid, w=w, bit_out=4)
        F.plan_set_tuning(p, variant=variant, split_m1=128, chunk_frames=chunk)
        g = p.sector_run(c["raw1"], c["raw2"], 0, nf, F.make_delay_cfg(c["table"], **c["delay"]))
        assert g["n_failed"] == 0
        assert np.max(np.abs(g["acc_ph"] / o["acc_ph"] - 1)) < 1e-5, variant   # the plain form's bar
        if raw:   # a byte holds two codes, each may flip at a decision boundary (1e-4 of codes)
            assert np.count_nonzero(g["raw_out"] != o["raw_out"]) <= 2e-4 * o["raw_out"].size + 2
