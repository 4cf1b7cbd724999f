"""The wave kernel over several parameter slabs: the allocation-free entry
against the plan's own, bit for bit where its static scratch holds as many
partial slots (N <= 4096), and both against the Stockham kernel."""
import numpy as np
import pytest

import fxcorr as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,form,nf", [(256, "plain", 600_000), (1024, "plain", 600_001), (4096, "chosen", 480_000),
                                       (8192, "chosen", 140_001)])
def test_noalloc_and_plan_over_slabs(n, form, nf):
    fs = 1024e6
    s = F.Stream()
    r = [F.DeviceBuffer(nf * n // 8) for _ in range(2)]
    for st in range(2):
        F.synth_station_device(r[st].ptr, nf * n, 1, None, False, 9, st, 0.2, 3, s.ptr)
    cfg = F.make_delay_cfg(np.zeros(8), frame_dt=n / fs, fs=fs, delay_user_samples=3.3, extra_delay_rate_sps=2e-9,
                           lo1_hz=6.7e9, lo2_hz=6.7e9)
    lv = np.array([-1.0, 1.0])
    kw = dict(bits=(1, 1), levels=[lv, lv], df_hz=fs / n,
              precision=F.PRECISION_PLAIN_FP32 if form == "plain" else F.PRECISION_CHOSEN)
    p = F.Plan(n, **kw)
    acc = [F.DeviceBuffer(F.N_PRODUCTS * p.half * 8) for _ in range(2)]
    p.sector_run_device(r[0].ptr, r[1].ptr, 0, nf, cfg, acc[0].ptr, stream=s.ptr)
    p.sector_run_device_noalloc(r[0].ptr, r[1].ptr, 0, nf, cfg, acc[1].ptr, stream=s.ptr)
    s.sync()
    own, na = (a.download(np.zeros(F.N_PRODUCTS * p.half)).reshape(F.N_PRODUCTS, p.half) for a in acc)
    if n <= 4096:
        assert np.array_equal(own, na), np.max(np.abs(own - na))
    scale = np.abs(own).max(axis=1, keepdims=True) + 1e-300
    assert np.all(np.abs(own - na) <= 1e-11 * scale)   # another order of up to 512 FP64 partial sums
    if n >= 2048:
        q = F.Plan(n, **kw)
        F.plan_set_tuning(q, variant=1)
        q.sector_run_device(r[0].ptr, r[1].ptr, 0, nf, cfg, acc[1].ptr, stream=s.ptr)
        s.sync()
        st = acc[1].download(np.zeros(F.N_PRODUCTS * p.half)).reshape(F.N_PRODUCTS, p.half)
        assert np.all(np.abs(own - st) <= 1e-6 * scale)   # FP32 transforms, each within 5e-7
