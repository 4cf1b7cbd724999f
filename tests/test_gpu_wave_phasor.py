"""The plain form's XCF phasors in the wave kernel, up to 512 overlap bins: the
FP64 powers of the reference's f32 start and step (main.rs:133-149), rounded
to f32 at the bin.  Both stations carry one impulse per frame (level 1 at
sample 0, level 0 elsewhere), so every spectrum is exactly 1 and the summed
cross spectrum is the frames' phasor times their number."""
import numpy as np
import pytest

import fxcorr as F

pytestmark = pytest.mark.gpu


def polar32(theta):
    t = np.float64(np.float32(theta))
    return complex(np.float32(np.cos(t)), np.float32(np.sin(t)))


@pytest.mark.parametrize("delay", [0.437, -0.3, 0.0213])
@pytest.mark.parametrize("n,shift", [(256, 0), (256, 37), (512, -5), (1024, 0), (1024, -2), (2048, 600), (4096, -1700),
                                     (8192, 3600)])
def test_plain_xcf_phasors(n, shift, delay):
    fs, nf, m = 64e6, 2048, n // 2
    a1s = max(0, -shift)
    band = (shift, a1s, min(m, m - shift), a1s + shift)
    codes = np.zeros((nf, n), dtype=np.uint8)
    codes[:, 0] = 1
    raw = np.packbits(codes.reshape(-1), bitorder="little")
    lv = np.array([0.0, 1.0])
    p = F.Plan(n, bits=(1, 1), levels=(lv, lv), band=band, df_hz=fs / n, products=F.PRODUCT_XCF)
    g = p.sector_run(raw, raw, 0, nf, F.make_delay_cfg(np.zeros(4), frame_dt=n / fs, fs=fs, delay_user_samples=delay))
    step = -2.0 * np.pi * (fs / n) * (delay / fs)
    k = np.arange(band[2] - a1s)
    q = polar32(step)   # its powers: modulus and angle in FP64
    want = polar32(step * a1s) * abs(q) ** k * np.exp(1j * np.angle(q) * k)
    got = g["acc12"][a1s:band[2]] / nf
    # one rounding to f32 of parts below 1 (2^-25), and 2% for the FP64 angle arithmetic
    tol = 1.02 * 2.0 ** -25
    assert np.max(np.abs(got.real - want.real)) < tol and np.max(np.abs(got.imag - want.imag)) < tol
