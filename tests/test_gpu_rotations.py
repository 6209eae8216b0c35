"""The rotations of a datastream's frequencies, which the block prologue forms
a thread a block (one or two) or over the whole workgroup (more): spectra of
jobs of 1 to 16 subbands against the FP64 oracle at block counts around a
workgroup's 128, and the prologue of 16 subbands in little more time than one's.

Tolerance: a transform of log2(L) butterfly stages of three FP32 roundings
each, with the table, rotation and store roundings (eight more), every one
half an ulp (2^-25 relative to the value's binade top), added as they stand."""
import ctypes as C

import numpy as np
import pytest

from fxcorr import JobSpec, check
from fxsynth import make_subint
from fxtestlib import GpuJob, oracle_spectra, rel_err

pytestmark = pytest.mark.gpu


def make(nsb, blocks, nstations=2):
    spec = JobSpec(nstations=nstations, nsubbands=nsb, npol=1, bw_mhz=16.0, nchan=64, blockspersend=blocks, crosspol=False,
                   lsb=[sb % 3 == 1 for sb in range(nsb)], looffset_hz=[0.0, 37.5], clockoffset_us=[0.0, 0.013],
                   base_freq_mhz=8400.25)
    sd = make_subint(spec, seed=nsb + blocks, delays_us=[2.3 * s for s in range(nstations)],
                     rates_us_per_s=[0.4 - 0.9 * s for s in range(nstations)],
                     invalid_blocks={0: [blocks // 2]} if blocks > 1 else None)
    return spec, sd


@pytest.mark.parametrize("blocks", [1, 5, 127, 128, 129, 257])
@pytest.mark.parametrize("nsb", [1, 2, 4, 16])
def test_spectra(gpu, oracle, nsb, blocks):
    lib, ctx = gpu
    spec, sd = make(nsb, blocks)
    job, keep = spec.build()
    g = GpuJob(lib, ctx, job)
    g.process(sd, keep_taps=True)
    tol = (3 * np.log2(spec.fftchannels) + 8) * 2.0 ** -25
    for ds in range(2):
        for blk in sorted({0, min(126, blocks - 1), blocks // 2, blocks - 1}):
            ref = oracle_spectra(oracle, job, sd, ds, blk, nsb, spec.nchan, fp64=True)
            for band in range(nsb):
                got = g.spectrum(ds, band, blk, spec.nchan)
                assert (rel_err(got, ref[band]) < tol) if np.any(ref[band]) else not np.any(got), (ds, blk, band)
    g.close()


def prologue_us(gpu, nsb):
    lib, ctx = gpu
    spec, sd = make(nsb, 1)
    job, keep = spec.build()
    g = GpuJob(lib, ctx, job)
    check(lib, lib.fxg_job_set_profiling(g.h, 1), "profiling")
    ms, n = (C.c_double * 10)(), (C.c_int64 * 10)()
    best = 1e9
    for _ in range(20):
        g.process(sd)
        check(lib, lib.fxg_job_stage_times(g.h, ms, n, 1), "stage_times")
        best = min(best, 1e3 * ms[1])
    g.close()
    return best


def test_time(gpu):
    one, many = prologue_us(gpu, 1), prologue_us(gpu, 16)
    print(f"1 subband {one:.1f}, 16 subbands {many:.1f} us", flush=True)
    assert many < 1.5 * one      # 1.9 with a thread a block
