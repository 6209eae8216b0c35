"""Two bands of one rotation to a workgroup (the shifted-grid F stage of 2048
to 8192 points takes them in launches of 4096 workgroups and more), against the
FP64 oracle and against the same blocks one band at a time (a pass of few
blocks): both sample sizes and sidebands, a polarisation phase, a frequency
whose bands have no common rotation, blanked frames and a flagged block.

Tolerance: a transform of log2(L) butterfly stages of three FP32 roundings
each, with the table, rotation and store roundings (eight more), every one
half an ulp (2^-25 relative to the value's binade top), added as they stand;
the two forms do the same operations in the same order, so they agree in every
bit."""
import ctypes as C

import numpy as np
import pytest

from fxcorr import JobSpec, Schedule, check
from fxsynth import StationData, SubintData, vdif_headers
from fxtestlib import GpuJob, oracle_spectra, rel_err

pytestmark = pytest.mark.gpu

STATIONS, SUBBANDS, PASS = 2, 4, 16
BANDPAIRS = STATIONS * (SUBBANDS - 1)          # the last subband's bands turn differently


def noise_subint(spec, seed, bad, flagged):
    """Frames of uniform random samples (levels and bytes alike); station 1
    has the invalid frames `bad`, station 0 the flagged block."""
    rng = np.random.default_rng(seed)
    fs, ts = spec.framesamples, spec.sampletime_us
    guard = 2
    while abs(guard * fs * ts * 1000.0 - round(guard * fs * ts * 1000.0)) > 1e-6:
        guard += 1                              # the data start on a whole nanosecond
    nframes = (spec.blockspersend * spec.fftchannels + fs - 1) // fs + 2 * guard + 1
    sec, ns = divmod(10 * 10 ** 9 - int(round(guard * fs * ts * 1000.0)), 10 ** 9)
    fps = int(round(1e6 / ts)) // fs
    stations = []
    for s in range(spec.nstations):
        fr = np.frombuffer(rng.bytes(nframes * spec.framebytes), np.uint8).reshape(nframes, -1).copy()
        fr[:, :32] = vdif_headers(sec, int(round(ns / 1000.0 / ts)) // fs, nframes, fps, spec.framebytes,
                                  spec.nrecbands, spec.nbits, s)
        if s == 1:
            for f in bad:
                fr[guard + f, 3] |= 0x80
        flags = np.zeros((spec.blockspersend + 29) // 30, np.int64)
        for b in range(spec.blockspersend):
            if s != 0 or b != flagged:
                flags[b // 30] |= 1 << (b % 30)
        block_s = spec.fftchannels * ts * 1e-6
        stations.append(StationData(raw=fr.reshape(-1), datasec=sec, datans=ns, validflags=flags.astype(np.int32),
                                    interpolator=np.array([0.0, (0.7 - s) * block_s, 0.37 * s]), delay_samples=0))
    return SubintData(spec=spec, sub_sec=10, sub_ns=0, scan_start_sec=0, stations=stations)


# twice the workgroups from which bands go in pairs; at 8192 points, whose grid the 32-station tests reach too, a
# quarter more
@pytest.mark.parametrize("nbits", [2, 8])
@pytest.mark.parametrize("nchan,blocks", [(1024, 1365), (2048, 1365), (4096, 853)])
def test_pairs_of_bands(gpu, oracle, nchan, blocks, nbits):
    lib, ctx = gpu
    spec = JobSpec(nstations=STATIONS, nsubbands=SUBBANDS, npol=2, bw_mhz=16.0, nchan=nchan, nbits=nbits,
                   blockspersend=blocks, lsb=[0, 1, 0, 1], looffset_hz=[0.0, 37.5], clockoffset_us=[0.0, 0.013],
                   phaseoffset_deg=[0.0, 40.0], base_freq_mhz=8400.25)
    assert (blocks + 7) // 8 * 8 * BANDPAIRS >= 4096 * 5 // 4
    job, keep = spec.build()
    for s in range(STATIONS):
        job.datastreams[s].recfreq_clockoffsetdelta_us[SUBBANDS - 1] = 0.021
    last = blocks - 1 - (blocks - 1) % PASS     # the last pass of few blocks
    per = spec.fftchannels / spec.framesamples  # frames of a block
    sd = noise_subint(spec, nchan + nbits, bad=[int(1.5 * per), int((last + 1) * per), int((last + 2.5) * per)],
                      flagged=last + 3)
    g = GpuJob(lib, ctx, job)
    g.process(sd, keep_taps=True)
    tol = (3 * np.log2(spec.fftchannels) + 8) * 2.0 ** -25
    paired = {}
    for ds in range(STATIONS):
        for blk in [0, 1, 2, blocks // 2] + list(range(last, blocks)):
            ref = oracle_spectra(oracle, job, sd, ds, blk, spec.nrecbands, nchan, fp64=True) if blk < last + 4 else None
            for band in range(spec.nrecbands):
                got = paired[ds, blk, band] = g.spectrum(ds, band, blk, nchan)
                if ref is None:
                    continue
                if not np.any(ref[band]):
                    assert not np.any(got), (ds, blk, band)
                else:
                    assert rel_err(got, ref[band]) < tol, (ds, blk, band, rel_err(got, ref[band]), tol)
    assert not np.any(paired[0, last + 3, 0]) and np.any(paired[1, last + 3, 0])
    s = Schedule()
    check(lib, lib.fxg_job_get_schedule(g.h, C.byref(s)), "get_schedule")
    s.chunk_blocks = PASS
    check(lib, lib.fxg_job_set_schedule(g.h, C.byref(s)), "set_schedule")
    g.process(sd, keep_taps=True)
    for ds in range(STATIONS):
        for blk in range(last, blocks):
            for band in range(spec.nrecbands):
                got = g.spectrum(ds, band, blk, nchan)
                assert np.array_equal(got.view(np.uint32), paired[ds, blk, band].view(np.uint32)), (ds, blk, band)
    g.close()
