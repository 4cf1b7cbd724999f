"""The autotuner on samples shorter than the plan's kernel for long sectors
takes: the default stays, so that later long sectors run on that kernel."""
import numpy as np
import pytest

import fxcorr as F
from _synth import LEVELS_2BIT

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,form,shift,nf,variant", [
    (4096, "chosen", 0, 300, 0), (8192, "plain", 0, 500, 0), (1024, "plain", 0, 200, 0), (2048, "chosen", 3, 400, 0),
    (16384, "plain", 0, 300, 1), (65536, "plain", 128, 64, 1)])
def test_short_sample_leaves_the_default(n, form, shift, nf, variant):
    fs, m = 256e6, n // 2
    s = F.Stream()
    r = [F.DeviceBuffer(nf * n // 4) for _ in range(2)]
    for st in range(2):
        F.synth_station_device(r[st].ptr, nf * n, 2, None, False, 9, st, 0.2, 3, s.ptr)
    s.sync()
    p = F.Plan(n, levels=[LEVELS_2BIT, LEVELS_2BIT], df_hz=fs / n, band=(shift, 0, m - shift, shift),
               precision=F.PRECISION_PLAIN_FP32 if form == "plain" else F.PRECISION_CHOSEN)
    default = (p.info.variant, p.info.grid_divisor)
    cfg = F.make_delay_cfg(np.zeros(4), frame_dt=n / fs, fs=fs, delay_user_samples=3.3, lo1_hz=3e9)
    rep = F.plan_autotune(p, r[0].ptr, r[1].ptr, nf, cfg, s.ptr)
    assert default == (variant, 1) and (rep["variant"], rep["grid_divisor"]) == default
    assert (p.info.variant, p.info.grid_divisor) == default
    assert rep["candidates"] == 1 and 0 < rep["best_ms"] == rep["default_ms"]
