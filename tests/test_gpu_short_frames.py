"""Streams of short frames, whose every group of the corner turn lies in
another frame: the spectra against the FP64 oracle, and a small job's corner
turn no slower than a few times that of the same samples in long frames."""
import ctypes as C

import numpy as np
import pytest

from fxcorr import JobSpec, check
from fxsynth import make_subint
from fxtestlib import GpuJob, oracle_spectra, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsb,npol,nbits,sampling,payload", [
    (1, 1, 2, "real", 8), (1, 1, 2, "real", 24), (1, 2, 2, "real", 16), (2, 2, 2, "real", 40), (4, 2, 2, "real", 8),
    (4, 2, 2, "real", 136), (1, 1, 8, "real", 8), (1, 2, 8, "real", 24), (4, 2, 8, "real", 16), (16, 2, 8, "real", 32),
    (1, 2, 2, "complex", 8), (1, 1, 8, "complex", 8), (4, 2, 8, "complex", 16)])
def test_spectra(gpu, oracle, nsb, npol, nbits, sampling, payload):
    lib, ctx = gpu
    spec = JobSpec(nstations=2, nsubbands=nsb, npol=npol, bw_mhz=16.0, nchan=128, nbits=nbits, blockspersend=9,
                   crosspol=npol == 2, sampling=sampling, framebytes=32 + payload)
    job, keep = spec.build()
    sd = make_subint(spec, seed=payload + nbits, delays_us=[0.0, 3.3], rates_us_per_s=[0.1, -0.2])
    g = GpuJob(lib, ctx, job)
    g.process(sd, keep_taps=True)
    # a wrong sample moves a spectrum by far more than the F stage's rounding
    # (3 log2 L + 8 half ulps)
    tol = (3 * np.log2(spec.fftchannels) + 8) * 2.0 ** -25
    for ds in range(2):
        for blk in (0, 4, 8):
            ref = oracle_spectra(oracle, job, sd, ds, blk, spec.nrecbands, spec.nchan, fp64=True)
            for band in range(spec.nrecbands):
                assert rel_err(g.spectrum(ds, band, blk, spec.nchan), ref[band]) < 4 * tol, (ds, blk, band)
    g.close()


def frames_us(gpu, payload):
    """The frame table and corner turn of a small job, the quickest of ten."""
    lib, ctx = gpu
    spec = JobSpec(nstations=4, nsubbands=1, npol=2, bw_mhz=16.0, nchan=256, nbits=8, blockspersend=8,
                   framebytes=32 + payload)
    job, keep = spec.build()
    sd = make_subint(spec, seed=3)
    g = GpuJob(lib, ctx, job)
    check(lib, lib.fxg_job_set_profiling(g.h, 1), "profiling")
    ms, n = (C.c_double * 10)(), (C.c_int64 * 10)()
    best = 1e9
    for _ in range(10):
        g.process(sd)
        check(lib, lib.fxg_job_stage_times(g.h, ms, n, 1), "stage_times")
        best = min(best, 1e3 * ms[0])
    g.close()
    return best


def test_small_job_time(gpu):
    # one word of a band in four a frame: finding a group's frame by steps of a
    # frame took 288 us against 13; the entries of the frame table alone, one
    # thread each, differ by a factor that a wavefront hides
    short, long = frames_us(gpu, 8), frames_us(gpu, 8000)
    print(f"payload 8: {short:.1f} us, 8000: {long:.1f} us", flush=True)
    assert short < 4 * long
