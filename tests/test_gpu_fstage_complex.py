"""The shifted-grid F stage of complex samples at every transform length,
against the FP64 oracle: block counts around the blocks a workgroup holds, both
sample sizes, the four sideband layouts, blanked frames (the staged validity
path), flagged blocks and an LO offset.

Tolerance: a transform of log2(L) butterfly stages of three FP32 roundings
each, with the table, rotation and store roundings (eight more), every one
half an ulp (2^-25 relative to the value's binade top), added as they stand."""
import numpy as np
import pytest

from fxcorr import JobSpec
from fxsynth import make_subint
from fxtestlib import GpuJob, oracle_spectra, rel_err

pytestmark = pytest.mark.gpu

# (channels, blocks): one workgroup holds 32, 16, 8, 4, 2 or 1 blocks
SHAPES = [(128, 1), (128, 33), (256, 17), (512, 9), (1024, 5), (2048, 3), (4096, 2), (8192, 2)]


@pytest.mark.parametrize("sampling", ["complex", "complex_dsb"])
@pytest.mark.parametrize("nbits", [2, 8])
@pytest.mark.parametrize("nchan,blocks", SHAPES)
def test_spectra_of_every_length(gpu, oracle, nchan, blocks, nbits, sampling):
    lib, ctx = gpu
    spec = JobSpec(nstations=2, nsubbands=2, npol=2, bw_mhz=16.0, nchan=nchan, nbits=nbits, blockspersend=blocks,
                   lsb=[0, 1], sampling=sampling, looffset_hz=[0.0, 37.5], clockoffset_us=[0.0, 0.013],
                   phaseoffset_deg=[0.0, 40.0], base_freq_mhz=8400.25)
    job, keep = spec.build()
    sd = make_subint(spec, seed=nchan + blocks, delays_us=[0.0, 4.7], rates_us_per_s=[0.4, -0.9],
                     invalid_frames={1: [1, 2]}, invalid_blocks={0: [blocks // 2]} if blocks > 1 else None)
    g = GpuJob(lib, ctx, job)
    g.process(sd, keep_taps=True)
    tol = (3 * np.log2(spec.fftchannels) + 8) * 2.0 ** -25
    for ds in range(2):
        for blk in sorted({0, blocks // 2, blocks - 1}):
            ref = oracle_spectra(oracle, job, sd, ds, blk, spec.nrecbands, spec.nchan, fp64=True)
            for band in range(spec.nrecbands):
                got = g.spectrum(ds, band, blk, spec.nchan)
                if not np.any(ref[band]):
                    assert not np.any(got)
                else:
                    assert rel_err(got, ref[band]) < tol, (ds, blk, band, rel_err(got, ref[band]), tol)
    g.close()
