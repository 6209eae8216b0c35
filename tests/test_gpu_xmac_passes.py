"""Visibilities added up over several passes of blocks in the streamed
cross-multiplies of more than 8 inputs, whose tiles leave through LDS and are
added to what V holds: input counts of one to four tiles and of two chunks,
FP32 and reduced precision, whole passes in one row of workgroups and passes
split over several, against the FP64 oracle product by product.

Tolerance: twice the spectra's bound ((3 log2 L + 8) half ulps of FP32, in
reduced precision half an ulp of the stored type more) for the two factors of
a product, and half an ulp for each of the blocks and passes added up."""
import numpy as np
import pytest

from fxcorr import JobSpec
from fxsynth import make_subint
from fxtestlib import GpuJob, oracle_results, rel_err

pytestmark = pytest.mark.gpu

HALF_ULP = {"fp32": 0.0, "fp16": 2.0 ** -11, "bf16": 2.0 ** -8}
CASES = ([("fp32", nst, npol, 17, 5) for nst, npol in ((9, 1), (8, 2), (16, 2), (33, 1), (24, 2), (32, 2), (33, 2))] +
         [("fp32", 32, 2, 100, 40), ("fp32", 40, 2, 17, 5)] +
         [(x, nst, npol, 17, 5) for x in ("fp16", "bf16") for nst, npol in ((3, 1), (4, 2), (9, 1), (16, 2), (17, 2), (32, 2),
                                                                             (40, 2))] +
         [("fp16", 12, 2, 100, 40)])


@pytest.mark.parametrize("xmac,nstations,npol,blocks,chunk", CASES)
def test_passes(gpu, oracle, xmac, nstations, npol, blocks, chunk):
    lib, ctx = gpu
    nchan = 64
    spec = JobSpec(nstations=nstations, nsubbands=1, npol=npol, bw_mhz=16.0, nchan=nchan, blockspersend=blocks,
                   crosspol=npol == 2, xmac=xmac, max_chunk_blocks=chunk)
    job, keep = spec.build()
    rng = np.random.default_rng(nstations)
    sd = make_subint(spec, seed=nstations + blocks, rho=0.3, delays_us=rng.uniform(-5, 5, nstations),
                     rates_us_per_s=rng.uniform(-1, 1, nstations))
    g = GpuJob(lib, ctx, job)
    assert g.info.chunk_blocks == chunk
    got = g.process(sd)
    ref = oracle_results(oracle, job, sd, fp64=True, nthreads=8)
    passes = (blocks + chunk - 1) // chunk
    tol = (2 * (3 * np.log2(spec.fftchannels) + 8) + blocks + passes) * 2.0 ** -25 + 2 * HALF_ULP[xmac]
    assert rel_err(got, ref) < tol, (rel_err(got, ref), tol)
    # every product by itself: none hides behind the autocorrelations; 4.4 is
    # above the levels' mean square, its double the spread of the powers
    nprod = nstations * (nstations - 1) // 2 * npol * npol
    for k in range(nprod):
        a, b = got[k * nchan:(k + 1) * nchan], ref[k * nchan:(k + 1) * nchan]
        assert np.linalg.norm(a - b) < tol * np.sqrt(nchan) * blocks * spec.fftchannels * 4.4 * 2, k
    # a second subintegration starts from nothing
    assert np.array_equal(g.process(sd).view(np.uint32), got.view(np.uint32))
    g.close()
