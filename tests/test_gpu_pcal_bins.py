"""Phase-cal accumulation of combs with few bins (k_pcal_few: a wavefront or
a workgroup per block, slices over the bins), against the FP64 oracle: 32 to
256 bins, numbers that do and do not divide a wavefront, real and complex
samples, the mixer, a bad frame and a flagged block.

Tolerance: a tone adds blocks x L terms of which each of the up to 1024
threads' partial sums and their tree rounds every addition by half an ulp;
relative to the root sum of squares of uncorrelated samples that is at most
sqrt(terms per thread) ulps with the table's and the product's two more."""
import ctypes as C

import numpy as np
import pytest

from fxcorr import JobSpec, check
from fxsynth import make_subint
from fxtestlib import GpuJob, oracle_results, rel_err

pytestmark = pytest.mark.gpu

CASES = [dict(bw_mhz=16.0, pcal_interval_mhz=1.0), dict(bw_mhz=32.0, pcal_interval_mhz=1.0),
         dict(bw_mhz=64.0, pcal_interval_mhz=1.0), dict(bw_mhz=128.0, pcal_interval_mhz=1.0),
         dict(bw_mhz=16.0, pcal_interval_mhz=3.0, base_freq_mhz=8401.0),
         dict(bw_mhz=32.0, pcal_interval_mhz=5.0, base_freq_mhz=8401.0, nbits=8),
         dict(bw_mhz=64.0, pcal_interval_mhz=1.0, sampling="complex", nbits=8),
         dict(bw_mhz=32.0, pcal_interval_mhz=3.0, sampling="complex", base_freq_mhz=8401.0)]


@pytest.mark.parametrize("kw", CASES, ids=lambda kw: f"{kw['bw_mhz']:.0f}MHz_{kw['pcal_interval_mhz']:.0f}_{kw.get('sampling', 'real')}_{kw.get('nbits', 2)}bit")
def test_few_bins(gpu, oracle, kw):
    lib, ctx = gpu
    spec = JobSpec(nstations=2, nsubbands=1, npol=2, nchan=256, blockspersend=37, **kw)
    job, keep = spec.build()
    sd = make_subint(spec, seed=5, delays_us=[0.0, 2.5], rates_us_per_s=[0.2, -0.4],
                     invalid_frames={1: [1]} if spec.nbits == 2 else None, invalid_blocks={0: [3]})
    g = GpuJob(lib, ctx, job)
    got = g.process(sd)
    ref = oracle_results(oracle, job, sd, fp64=True, nthreads=4)
    p0 = C.c_int64()
    check(lib, lib.fxg_plan_pcal_offset(C.byref(job), 0, C.byref(p0)), "pcal offset")
    terms = spec.blockspersend * spec.fftchannels
    tol = (np.sqrt(terms) + 2) * 2.0 ** -24
    assert rel_err(got[p0.value:], ref[p0.value:]) < tol, (rel_err(got[p0.value:], ref[p0.value:]), tol)
    g.close()
