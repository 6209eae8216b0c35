"""V of the reduced-precision streamed cross-multiply stored eight rows at a
time, rows past the last input left out: input counts either side of every
eighth row of one to three tiles of 32 and of a second chunk, against the FP64
oracle product by product.

Tolerance: twice the spectra's bound ((3 log2 L + 8) half ulps of FP32 and half
an ulp of fp16) for the two factors of a product, and half an ulp for each of
the blocks added up."""
import numpy as np
import pytest

from fxcorr import JobSpec
from fxsynth import make_subint
from fxtestlib import GpuJob, oracle_results, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nin", [2, 7, 8, 9, 16, 17, 24, 25, 32, 33, 41, 49, 57, 64, 65, 72, 73, 81, 88, 89, 97, 129])
def test_rows(gpu, oracle, nin):
    lib, ctx = gpu
    nchan, blocks = 64, 9
    spec = JobSpec(nstations=nin, nsubbands=1, npol=1, bw_mhz=16.0, nchan=nchan, blockspersend=blocks, crosspol=False,
                   xmac="fp16")
    job, keep = spec.build()
    rng = np.random.default_rng(nin)
    sd = make_subint(spec, seed=nin, rho=0.3, delays_us=rng.uniform(-5, 5, nin), rates_us_per_s=rng.uniform(-1, 1, nin))
    g = GpuJob(lib, ctx, job)
    got = g.process(sd)
    ref = oracle_results(oracle, job, sd, fp64=True, nthreads=8)
    tol = (2 * (3 * np.log2(spec.fftchannels) + 8) + blocks) * 2.0 ** -25 + 2.0 ** -10
    assert rel_err(got, ref) < tol, (rel_err(got, ref), tol)
    for k in range(nin * (nin - 1) // 2):
        a, b = got[k * nchan:(k + 1) * nchan], ref[k * nchan:(k + 1) * nchan]
        assert np.linalg.norm(a - b) < tol * np.sqrt(nchan) * blocks * spec.fftchannels * 4.4 * 2, k
    g.close()
