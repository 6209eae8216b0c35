"""The FP32 cross-multiply of up to 8 inputs (real and imaginary parts in one
tile), against the FP64 oracle: 1 to 9 inputs, block counts around its stages
of 16 blocks, with the blocks split over workgroups and over passes.

Tolerance: twice the spectra's bound ((3 log2 L + 8) half ulps) for the two
factors of a product, and half an ulp for each of the blocks added up."""
import numpy as np
import pytest

from fxcorr import JobSpec
from fxsynth import make_subint
from fxtestlib import GpuJob, oracle_results, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nstations,npol,blocks,chunk", [(2, 1, 1, 0), (3, 1, 16, 0), (2, 2, 15, 0), (5, 1, 17, 0),
                                                         (3, 2, 33, 7), (7, 1, 200, 0), (4, 2, 300, 100), (9, 1, 50, 0)])
def test_few_inputs(gpu, oracle, nstations, npol, blocks, chunk):
    lib, ctx = gpu
    spec = JobSpec(nstations=nstations, nsubbands=1, npol=npol, bw_mhz=16.0, nchan=64, blockspersend=blocks,
                   crosspol=npol == 2, max_chunk_blocks=chunk)
    job, keep = spec.build()
    rng = np.random.default_rng(nstations)
    sd = make_subint(spec, seed=nstations + blocks, rho=0.3, delays_us=rng.uniform(-5, 5, nstations),
                     rates_us_per_s=rng.uniform(-1, 1, nstations))
    g = GpuJob(lib, ctx, job)
    got = g.process(sd)
    ref = oracle_results(oracle, job, sd, fp64=True, nthreads=8)
    tol = 2 * (3 * np.log2(spec.fftchannels) + 8) * 2.0 ** -25 + blocks * 2.0 ** -25
    assert rel_err(got, ref) < tol, (rel_err(got, ref), tol)
    nprod = nstations * (nstations - 1) // 2 * npol * npol
    for k in range(nprod):
        a, b = got[k * 64:(k + 1) * 64], ref[k * 64:(k + 1) * 64]
        assert np.linalg.norm(a - b) < tol * np.sqrt(64.0) * blocks * spec.fftchannels * 4.4 * 2, k
    g.close()
