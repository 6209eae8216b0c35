"""The register corner turn for every unit size and band count: the bit
permutation on the host against its definition, and the kernel through whole
jobs against the oracle at frame sizes whose groups straddle frames."""
import os
import subprocess

import numpy as np
import pytest

from fxcorr import FXG_FORMAT_MARK5B, JobSpec
from fxsynth import make_subint

HERE = os.path.dirname(os.path.abspath(__file__))
BUILD = os.path.join(os.path.dirname(HERE), "difx-svn2git-try3_amd", "_build")


def test_turn_units_bits():
    exe = os.path.join(BUILD, "test_turn")
    assert os.path.exists(exe), "build first (__graft_entry__.build())"
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


# (subbands, pols, bits, sampling, payload): payloads in 8-byte steps that do
# and do not hold whole groups of 32 bits per band; 16-byte steps load wider
SHAPES = [(1, 1, 2, "real", 1000), (1, 2, 2, "real", 1000), (2, 2, 2, "real", 1000), (4, 2, 2, "real", 1000),
          (4, 2, 2, "real", 8000), (8, 2, 2, "real", 1008), (16, 2, 2, "real", 1056), (1, 1, 8, "real", 1000),
          (1, 2, 8, "real", 1000), (4, 2, 8, "real", 1000), (8, 2, 8, "real", 4000), (16, 2, 8, "real", 8000),
          (1, 2, 2, "complex", 1000), (4, 2, 2, "complex", 1000), (1, 2, 8, "complex", 1000), (4, 2, 8, "complex", 4000),
          (16, 2, 8, "complex", 8000)]


@pytest.mark.gpu
@pytest.mark.parametrize("nsb,npol,nbits,sampling,payload", SHAPES)
def test_streams_through_jobs(gpu, oracle, nsb, npol, nbits, sampling, payload):
    from fxtestlib import GpuJob, oracle_spectra, rel_err
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


@pytest.mark.gpu
@pytest.mark.parametrize("nsb", [1, 2, 4, 8])
def test_mark5b_streams(gpu, oracle, nsb):
    from fxtestlib import GpuJob, oracle_spectra, rel_err
    lib, ctx = gpu
    spec = JobSpec(nstations=2, nsubbands=nsb, npol=2, bw_mhz=16.0, nchan=256, blockspersend=21, framebytes=10016,
                   headerbytes=16, fmt=FXG_FORMAT_MARK5B)
    job, keep = spec.build()
    sd = make_subint(spec, seed=nsb, delays_us=[0.0, 2.1], invalid_frames={1: [1]})
    g = GpuJob(lib, ctx, job)
    g.process(sd, keep_taps=True)
    tol = (3 * np.log2(spec.fftchannels) + 8) * 2.0 ** -25
    for ds in range(2):
        for blk in (0, 10, 20):
            ref = oracle_spectra(oracle, job, sd, ds, blk, spec.nrecbands, spec.nchan, fp64=True)
            for band in range(spec.nrecbands):
                got = g.spectrum(ds, band, blk, spec.nchan)
                assert (rel_err(got, ref[band]) < 4 * tol) if np.any(ref[band]) else not np.any(got), (ds, blk, band)
    g.close()
