"""Device memory of the plain form at N = 16384: the chain table's bound, the
general kernels where the fused four-step's scratch may not be taken, and the
job server's budget counting that scratch before a job's first long sector."""
import numpy as np
import pytest

import fxcorr as F
from _synth import LEVELS_2BIT

pytestmark = pytest.mark.gpu
N, FS = 16384, 256e6
HALF = N // 2 + 1
KW = dict(bits=(2, 2), levels=[LEVELS_2BIT, LEVELS_2BIT], df_hz=FS / N, precision=F.PRECISION_PLAIN_FP32)


def setup(nf):
    s = F.Stream()
    r = [F.DeviceBuffer(nf * N // 4) for _ in range(2)]
    for st in range(2):
        F.synth_station_device(r[st].ptr, nf * N, 2, None, False, 5, st, 0.2, 3, s.ptr)
    cfg = F.make_delay_cfg(np.zeros(8), frame_dt=N / FS, fs=FS, delay_user_samples=3.3, lo1_hz=1e9, lo2_hz=1e9)
    return s, r, cfg


def spectra(p, s, r, cfg, nf):
    acc = F.DeviceBuffer(F.N_PRODUCTS * HALF * 8)
    p.sector_run_device(r[0].ptr, r[1].ptr, 0, nf, cfg, acc.ptr, stream=s.ptr)
    s.sync()
    return acc.download(np.zeros(F.N_PRODUCTS * HALF))


def test_chain_table_bound():
    nf = 12_000
    s, r, cfg = setup(nf)
    p = F.Plan(N, **KW)
    base = F.plan_device_bytes(p)
    spectra(p, s, r, cfg, nf)
    # two Y buffers of 1024 frames, 512 MiB of chains (a link's row: 9 to 24 frames of padding), parameters
    y, chains = 2 * 1024 * (N // 2) * 8, (8192 + 24) * (N // 2) * 8
    assert y + chains // 2 < F.plan_device_bytes(p) - base < y + chains + (16 << 20)


def test_lean_plan_runs_the_general_kernels():
    nf = 700
    s, r, cfg = setup(nf)
    p, q = F.Plan(N, **KW), F.Plan(N, **KW)
    F.plan_set_tuning(q, variant=0)
    F.lib().fxc_internal_plan_lean(p.h, 1)
    a, b = spectra(p, s, r, cfg, nf), spectra(q, s, r, cfg, nf)
    assert np.array_equal(a, b)
    # rows of the general path alone
    assert F.plan_device_bytes(p) == F.plan_device_bytes(q)
    F.lib().fxc_internal_plan_lean(p.h, 0)
    c = spectra(p, s, r, cfg, nf)
    assert not np.array_equal(a, c) and np.max(np.abs(a - c)) < 1e-5 * np.max(np.abs(a))
    assert F.plan_device_bytes(p) > F.plan_device_bytes(q)


@pytest.mark.parametrize("jobs_fit", [1, 0])
def test_server_budget_counts_the_scratch(jobs_fit):
    """jobs_fit = 1: the budget holds one job's plan with its scratch, not
    two.  0: it holds no such plan; the jobs run on the general kernels."""
    nf = 1200
    s, r, cfg = setup(nf)
    probe = F.Plan(N, **KW)
    held = F.plan_device_bytes(probe)
    want = spectra(probe, s, r, cfg, nf)
    grown = F.plan_device_bytes(probe)
    probe.close()
    # a job's most: Y, parameters and the whole chain table
    full = grown + (512 << 20) - 1200 * (N // 2) * 8
    spectra_bytes = 2 * F.N_PRODUCTS * HALF * 8
    budget = int(1.5 * full) if jobs_fit else 2 * (held + spectra_bytes) + (8 << 20)
    sv = F.Server(hbm_budget_bytes=budget, max_active_jobs=4, n_streams=2)
    jobs = []
    for _ in range(3):
        j = sv.submit(dict(KW, fft_len=N), cfg)
        sv.push(j, r[0].ptr, r[1].ptr, nf)
        jobs.append(j)
    for j in jobs:
        sv.close_job(j)
    for j in jobs:
        assert sv.wait(j, 120.0)
    st = sv.stats()
    got = [sv.result(j, HALF)[0] for j in jobs]
    sv.close()
    assert st.jobs_done == 3 and st.jobs_failed == 0
    if jobs_fit:
        assert st.max_concurrent_jobs == 1 and st.peak_hbm_bytes <= budget
    for g in got:
        assert np.array_equal(g, got[0]) and np.max(np.abs(g - want)) < 1e-5 * np.max(np.abs(want))
