"""The chosen form's phased sum on the fused four-step at N = 32768 / 65536
(band shift a multiple of 128) against the oracle, and against the four-step
through HBM (variant 0): both grids, one-row and many-row shifts, few frames,
a ragged last chunk, with and without the .raw output."""
import numpy as np
import pytest

import fxcorr as F
import fxref as R
from _cases import make_case

pytestmark = pytest.mark.gpu
PERM = np.random.default_rng(4).permutation(32).astype(np.int32)


@pytest.mark.parametrize("n,nf,chunk,shift,grid,raw", [(32768, 3, 512, 0, 0, True), (32768, 41, 16, -128, 1, True),
                                                       (32768, 30, 7, 4096, 0, False), (65536, 1, 256, 0, 1, True),
                                                       (65536, 19, 6, 128, 0, True), (65536, 26, 26, -2048, 1, False)])
def test_phased_fused_large(n, nf, chunk, shift, grid, raw):
    m, fs = n // 2, 256e6
    a1s = max(0, -shift)
    prods = F.PRODUCT_PHASED | (F.PRODUCT_RAW_OUT if raw else 0)
    c = make_case(n=n, fs=fs, nf=nf, bits=(2, 4), shuffles=(None, PERM), lsb=(True, False),
                  band=(shift, a1s, min(m, m - shift), a1s + shift), grid=grid, rho=0.4, delay_samples=3.0,
                  products=prods, seed=n + nf, no_table=True, net_d1_base=4.4 / fs, total_rate1_base=1e-9,
                  net_d2_base=-2.7 / fs, total_rate2_base=-2e-9, lo1_hz=1.5e9, lo2_hz=1.4e9)
    w, got = (0.8, 1.1), []
    for variant in (1, 0):
        p = F.Plan(n, bits=c["bits"], levels=c["levels"], shuffles=c["shuffles"], lsb=c["lsb"], band=c["band"],
                   df_hz=fs / n, products=prods, out_grid=grid, w=w, bit_out=4, precision=F.PRECISION_CHOSEN)
        F.plan_set_tuning(p, variant=variant, split_m1=128, chunk_frames=chunk)
        got.append(p.sector_run(c["raw1"], c["raw2"], 0, nf, F.make_delay_cfg(c["table"], **c["delay"])))
    desc = dict(fft_len=n, bits1=2, bits2=4, levels1=c["levels"][0], levels2=c["levels"][1],
                shuffle1=c["shuffles"][0], shuffle2=c["shuffles"][1], lsb1=1, lsb2=0, a1s=c["band"][1],
                a1e=c["band"][2], a2s=c["band"][3], out_grid=grid, df_hz=fs / n, need_acf=0, need_xcf=0,
                need_phased=1, write_raw=1, w1=w[0], w2=w[1], bit_out=4, output_lsb=0, cpu_threads=8)
    o = R.sector_run(desc, c["raw1"], c["raw2"], 0, nf, R.make_delay_cfg(c["table"], **c["delay"]),
                     mode=R.MODE_F64, threads=8)
    for g in got:
        assert g["n_failed"] == 0
        # the chosen form's bar, relative to the bin or (a bin where the stations cancel) to the mean bin
        assert np.max(np.abs(g["acc_ph"] - o["acc_ph"]) / (o["acc_ph"] + 0.1 * o["acc_ph"].mean())) < 1e-4
        if raw:   # a byte holds two codes, each may flip at a decision boundary (1e-4 of codes)
            assert np.count_nonzero(g["raw_out"] != o["raw_out"]) <= 2e-4 * o["raw_out"].size + 2
