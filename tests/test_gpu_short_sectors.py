"""Sectors around the launch grid's edges: one frame per workgroup up to the
workgroup cap, the first count past it (two frames per workgroup, a ragged
last one), and slot counts below, at and past the reduce's rows."""
import pytest

import fxcorr as F
import fxref as R
from _cases import gpu_run, make_case, oracle_run, spectra_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nf", [(64, 1), (256, 5), (512, 63), (1024, 65), (1024, 2049), (4096, 513), (16384, 3)])
@pytest.mark.parametrize("form", ["plain", "chosen"])
def test_short_sector_vs_oracle(n, nf, form):
    c = make_case(n=n, fs=64e6, nf=nf, rho=0.2, seed=nf, delay_user_samples=5.3, lo1_hz=6.7e9, lo2_hz=6.7e9)
    plain = form == "plain"
    g = gpu_run(c, F.PRECISION_PLAIN_FP32 if plain else F.PRECISION_CHOSEN)
    o = oracle_run(c, R.MODE_F32 if plain else R.MODE_F64)
    # the bars of the two forms (FP32 FFTs against the oracle of the same phases)
    tol = 1e-5 if plain else 1e-4
    errs = spectra_err(g, o)
    assert g["n_failed"] == 0 and all(e < tol for e in errs.values()), errs
    assert not g["acc_ph"].any()
