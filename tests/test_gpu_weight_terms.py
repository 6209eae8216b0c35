"""Weight sums whose terms are mostly neither 0 nor 1: streams of short frames
with many of them lost or, INTERLACEDVDIF, blanked band by band.  The weights
are the oracle's bit for bit (the same FP32 terms in block order), and the sums
take no longer than one addition at a time did."""
import ctypes as C
import random

import numpy as np
import pytest

from fxcorr import FXG_FORMAT_INTERLACEDVDIF, FXG_FORMAT_VDIF, JobSpec, check
from fxsynth import make_subint, set_edv4
from fxtestlib import GpuJob, oracle_results, plan_info, region_slices

pytestmark = pytest.mark.gpu


def job_of(fmt, blocks, lost):
    spec = JobSpec(nstations=2, nsubbands=1, npol=2, bw_mhz=16.0, nchan=64, blockspersend=blocks, framebytes=352, fmt=fmt)
    rng = random.Random(blocks)
    frames = blocks * spec.fftchannels // spec.framesamples
    sd = make_subint(spec, seed=3, delays_us=[0.0, 1.3],
                     invalid_frames={s: [f for f in range(frames) if rng.random() < lost] for s in range(2)})
    if fmt == FXG_FORMAT_INTERLACEDVDIF:
        for st in sd.stations:
            n = st.raw.size // spec.framebytes
            set_edv4(st.raw, spec.framebytes, 2, {f: rng.getrandbits(2) for f in range(0, n, 3)})
    return spec, sd


@pytest.mark.parametrize("blocks", [1, 63, 64, 65, 300, 4095, 4097, 8200])
@pytest.mark.parametrize("fmt,lost", [(FXG_FORMAT_VDIF, 0.2), (FXG_FORMAT_VDIF, 0.01), (FXG_FORMAT_INTERLACEDVDIF, 0.0),
                                      (FXG_FORMAT_INTERLACEDVDIF, 0.1)])
def test_weights(gpu, oracle, fmt, lost, blocks):
    lib, ctx = gpu
    spec, sd = job_of(fmt, blocks, lost)
    job, keep = spec.build()
    g = GpuJob(lib, ctx, job)
    got, ref = g.process(sd), oracle_results(oracle, job, sd)
    xend, a0, a1 = region_slices(oracle, job, plan_info(oracle, "orc_", job))
    for r in (slice(xend, a0), slice(a1, None)):
        assert np.array_equal(got[r].view(np.uint32), ref[r].view(np.uint32))
    g.close()


@pytest.mark.parametrize("fmt,lost", [(FXG_FORMAT_VDIF, 0.2), (FXG_FORMAT_INTERLACEDVDIF, 0.0)])
def test_time(gpu, fmt, lost):
    lib, ctx = gpu
    spec, sd = job_of(fmt, 20000, lost)
    job, keep = spec.build()
    g = GpuJob(lib, ctx, job)
    check(lib, lib.fxg_job_set_profiling(g.h, 1), "profiling")
    ms, n = (C.c_double * 10)(), (C.c_int64 * 10)()
    best = 1e9
    for _ in range(10):
        g.process(sd)
        check(lib, lib.fxg_job_stage_times(g.h, ms, n, 1), "stage_times")
        best = min(best, 1e3 * ms[4])
    g.close()
    print(f"20000 blocks: {best:.1f} us", flush=True)
    # one addition at a time took 140 and 150 us, by the place of each odd term 260 and 295
    assert best < 150.0
