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


def job_of(fmt, blocks, lost, nstations=2, nsubbands=1, framebytes=352):
    spec = JobSpec(nstations=nstations, nsubbands=nsubbands, npol=2, bw_mhz=16.0, nchan=64, blockspersend=blocks,
                   framebytes=framebytes, fmt=fmt)
    rng = random.Random(blocks)
    frames = blocks * spec.fftchannels // spec.framesamples
    sd = make_subint(spec, seed=3, delays_us=[1.3 * s for s in range(nstations)],
                     invalid_frames={s: [f for f in range(frames) if rng.random() < lost] for s in range(nstations)})
    if fmt == FXG_FORMAT_INTERLACEDVDIF:
        for st in sd.stations:
            n = st.raw.size // spec.framebytes
            nb = spec.nrecbands
            set_edv4(st.raw, spec.framebytes, nb, {f: rng.getrandbits(nb) for f in range(0, n, 3)})
    return spec, sd


def compare(gpu, oracle, spec, sd):
    lib, ctx = gpu
    job, keep = spec.build()
    g = GpuJob(lib, ctx, job)
    got, ref = g.process(sd), oracle_results(oracle, job, sd, nthreads=8)
    xend, a0, a1 = region_slices(oracle, job, plan_info(oracle, "orc_", job))
    for r in (slice(xend, a0), slice(a1, None)):
        assert np.array_equal(got[r].view(np.uint32), ref[r].view(np.uint32))
    g.close()


@pytest.mark.parametrize("blocks", [1, 63, 64, 65, 300, 511, 513, 1024, 1025, 4095, 4097, 8200])
@pytest.mark.parametrize("fmt,lost", [(FXG_FORMAT_VDIF, 0.2), (FXG_FORMAT_VDIF, 0.01), (FXG_FORMAT_INTERLACEDVDIF, 0.0),
                                      (FXG_FORMAT_INTERLACEDVDIF, 0.1)])
def test_weights(gpu, oracle, fmt, lost, blocks):
    compare(gpu, oracle, *job_of(fmt, blocks, lost))


# 24 stations of two bands: 1452 entries
@pytest.mark.parametrize("nstations,blocks", [(9, 1), (9, 513), (24, 5), (24, 1030)])
def test_many_entries(gpu, oracle, nstations, blocks):
    compare(gpu, oracle, *job_of(FXG_FORMAT_INTERLACEDVDIF, blocks, 0.0, nstations))


def weights_us(gpu, spec, sd):
    lib, ctx = gpu
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
    print(f"{spec.blockspersend} blocks: {best:.1f} us", flush=True)
    return best


@pytest.mark.parametrize("fmt,lost", [(FXG_FORMAT_VDIF, 0.2), (FXG_FORMAT_INTERLACEDVDIF, 0.0)])
def test_time_of_long_sums(gpu, fmt, lost):
    # one addition at a time took 140 and 150 us, by the place of each odd term 260 and 295
    assert weights_us(gpu, *job_of(fmt, 20000, lost)) < 150.0


def test_time_of_many_entries(gpu):
    # 6500 entries of 4 blocks: a workgroup an entry with one adding thread took 13 us, with 4096 terms' masks 35
    assert weights_us(gpu, *job_of(FXG_FORMAT_INTERLACEDVDIF, 4, 0.0, 20, 8, 8032)) < 13.0
