"""Phase cal of few bins with the blocks of a group enough for a wavefront each
and with fewer (then the workgroup shares a block), samples from the fast and
the frame-by-frame path, against the FP64 oracle; and a few blocks of long
transforms in a lossy stream no slower than a thread per bin took.

Tolerance: a tone adds blocks x L terms in partial sums whose every addition
rounds by half an ulp; relative to the root sum of squares of uncorrelated
samples that is at most the square root of the terms, in ulps, with the table's
and the product's two more."""
import ctypes as C

import numpy as np
import pytest

from fxcorr import JobSpec, check
from fxsynth import make_subint
from fxtestlib import GpuJob, oracle_results, rel_err

pytestmark = pytest.mark.gpu

# 32, 64 and 128 bins, with and without the mixer, real and complex
COMBS = [dict(bw_mhz=16.0, pcal_interval_mhz=1.0), dict(bw_mhz=32.0, pcal_interval_mhz=1.0),
         dict(bw_mhz=64.0, pcal_interval_mhz=1.0), dict(bw_mhz=16.0, pcal_interval_mhz=3.0, base_freq_mhz=8401.0),
         dict(bw_mhz=16.0, pcal_interval_mhz=3.0, base_freq_mhz=8401.0, sampling="complex"),
         dict(bw_mhz=32.0, pcal_interval_mhz=5.0, base_freq_mhz=8401.0, nbits=8)]


@pytest.mark.parametrize("blocks", [3, 64, 65, 192, 193, 256, 330])      # 64 groups of a job of 16 bands
@pytest.mark.parametrize("kw", COMBS, ids=lambda kw: f"{kw['bw_mhz']:.0f}MHz_{kw['pcal_interval_mhz']:.0f}_{kw.get('sampling', 'real')}_{kw.get('nbits', 2)}bit")
def test_groups(gpu, oracle, kw, blocks):
    lib, ctx = gpu
    spec = JobSpec(nstations=2, nsubbands=4, npol=2, nchan=128, blockspersend=blocks, crosspol=False, **kw)
    job, keep = spec.build()
    sd = make_subint(spec, seed=blocks, delays_us=[0.0, 2.5], rates_us_per_s=[0.2, -0.4],
                     invalid_frames={1: [1, 2]} if spec.nbits == 2 else None, invalid_blocks={0: [1]})
    g = GpuJob(lib, ctx, job)
    got = g.process(sd)
    ref = oracle_results(oracle, job, sd, fp64=True, nthreads=8)
    p0 = C.c_int64()
    check(lib, lib.fxg_plan_pcal_offset(C.byref(job), 0, C.byref(p0)), "pcal offset")
    tol = (np.sqrt(blocks * spec.fftchannels) + 2) * 2.0 ** -24
    assert rel_err(got[p0.value:], ref[p0.value:]) < tol, (rel_err(got[p0.value:], ref[p0.value:]), tol)
    g.close()


def test_time_of_few_lossy_blocks(gpu):
    lib, ctx = gpu
    spec = JobSpec(nstations=5, nsubbands=1, npol=1, bw_mhz=8.0, nchan=4096, nbits=8, blockspersend=25,
                   pcal_interval_mhz=5.0, base_freq_mhz=8400.25)
    job, keep = spec.build()
    frames = 25 * spec.fftchannels // spec.framesamples
    sd = make_subint(spec, seed=1, delays_us=[float(s) for s in range(5)],
                     invalid_frames={s: list(range(s % 3, frames, 3)) for s in range(5)})
    g = GpuJob(lib, ctx, job)
    check(lib, lib.fxg_job_set_profiling(g.h, 1), "profiling")
    ms, n = (C.c_double * 10)(), (C.c_int64 * 10)()
    best = 1e9
    for _ in range(10):
        g.process(sd)
        check(lib, lib.fxg_job_stage_times(g.h, ms, n, 1), "stage_times")
        best = min(best, 1e3 * ms[8])
    g.close()
    print(f"25 blocks: {best:.1f} us", flush=True)
    # a wavefront to a block, one block to a group, took 98 us; a thread per bin 80
    assert best < 70.0
