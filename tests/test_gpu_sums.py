"""The sums behind the spectra: weights over thousands of blocks (k_weights
adds runs of ones at once), results that land in a caller's device buffer with
nothing left of what it held.  The weights are the oracle's bit for bit (the
same FP32 terms in block order)."""
import ctypes as C

import numpy as np
import pytest

from fxcorr import JobSpec, check
from fxsynth import make_subint
from fxtestlib import GpuJob, oracle_results, plan_info, region_slices

pytestmark = pytest.mark.gpu


def data(spec, **kw):
    n = spec.nstations
    return make_subint(spec, seed=7, delays_us=[0.7 * i for i in range(n)],
                       rates_us_per_s=[0.2 - 0.3 * i for i in range(n)], **kw)


@pytest.mark.parametrize("nblocks,payload,every", [(63, 1000, 2), (64, 1000, 0), (65, 104, 3), (4095, 1000, 40),
                                                   (4097, 104, 11), (9000, 104, 2), (9000, 1000, 97)])
def test_long_weight_sums(gpu, oracle, nblocks, payload, every):
    """Every nth frame of two stations lost; a frame holds 15.6 or 1.6 blocks,
    so that the blocks at its ends have fractions of a sample count."""
    lib, ctx = gpu
    spec = JobSpec(nstations=3, nsubbands=1, npol=2, bw_mhz=16.0, nchan=64, blockspersend=nblocks,
                   framebytes=32 + payload)
    job, keep = spec.build()
    frames = nblocks * 128 // (2 * payload)
    lost = {s: list(range(s, frames, every)) for s in (0, 2)} if every else None
    sd = data(spec, invalid_frames=lost, invalid_blocks={1: [b for b in (3, 5, 64, 4096) if b < nblocks]})
    g = GpuJob(lib, ctx, job)
    got, ref = g.process(sd), oracle_results(oracle, job, sd)
    xend, a0, a1 = region_slices(oracle, job, plan_info(oracle, "orc_", job))
    for r in (slice(xend, a0), slice(a1, None)):
        assert np.array_equal(got[r].view(np.uint32), ref[r].view(np.uint32))
    g.close()


@pytest.mark.parametrize("kw", [dict(), dict(crosspol=False), dict(zoom=[(1, 64, 32)]), dict(pcal_interval_mhz=1.0)],
                         ids=["full", "parallel", "zoom", "pcal"])
def test_results_replace_what_the_buffer_held(gpu, oracle, kw):
    lib, ctx = gpu
    spec = JobSpec(nstations=3, nsubbands=2, npol=2, bw_mhz=16.0, nchan=128, blockspersend=20, **kw)
    job, keep = spec.build()
    sd = data(spec)
    ref = oracle_results(oracle, job, sd).view(np.float32)
    g = GpuJob(lib, ctx, job)
    held = np.full(ref.size, np.nan, dtype=np.float32)
    p = C.c_void_p()
    check(lib, lib.fxg_device_alloc(ctx, held.nbytes, C.byref(p)), "alloc")
    check(lib, lib.fxg_memcpy_h2d(ctx, p, held.ctypes.data, held.nbytes), "h2d")
    sub = sd.subint_desc()
    st, keep2 = sd.station_inputs()
    check(lib, lib.fxg_subint_process(g.h, C.byref(sub), st, 0, p, 1), "process")
    check(lib, lib.fxg_memcpy_d2h(ctx, held.ctypes.data, p, held.nbytes), "d2h")
    lib.fxg_device_free(ctx, p)
    assert np.all(np.isfinite(held))
    assert not np.any(held[ref == 0.0])
    assert np.array_equal(held, g.process(sd).view(np.float32))
    g.close()
