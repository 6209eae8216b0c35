"""The multiplexer's corner turn over unit sizes and thread counts (each
power of two up to 32 and counts that need padding), threads missing, payloads
that leave part of a workgroup, output frames that wide stores cannot reach:
the oracle's bytes."""
import ctypes as C

import numpy as np
import pytest

import fxcorr
from fxcorr import check
from muxlib import mux_desc, orc_mux, thread_stream

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (1, 1, 8), (2, 1, 2), (2, 1, 3), (2, 1, 8), (2, 1, 16), (2, 1, 17), (1, 1, 31), (2, 2, 5), (2, 4, 4), (2, 8, 2),
          (4, 1, 16), (4, 4, 8), (8, 1, 1), (8, 1, 4), (8, 2, 16), (8, 4, 2), (16, 2, 8)]


@pytest.mark.parametrize("offset", [0, 4])
@pytest.mark.parametrize("bits,chans,threads", SHAPES, ids=lambda v: str(v))
def test_units(gpu, oracle, bits, chans, threads, offset):
    lib, ctx = gpu
    ids = list(range(threads))
    for framebytes, flags in ((40, 0), (1056, 0), (4136, fxcorr.FXG_MUX_PROPAGATEVALIDITY)):
        kw = dict(framebytes=framebytes, nbits=bits, nchan=chans, nsort=threads, ngap=threads, flags=flags)
        src, _ = thread_stream(ids, framebytes=framebytes, nframes=7, nbits=bits, nchan=chans, seed=threads,
                               drop={(3, threads // 2)})
        r0, d0, s0 = orc_mux(oracle, src, ids, 9, **kw)
        d = mux_desc(ids, **kw)
        p = C.c_void_p()
        check(lib, lib.fxg_device_alloc(ctx, d0.size + 16, C.byref(p)), "alloc")
        st = fxcorr.VdifMuxStats()
        src = np.ascontiguousarray(src)
        r1 = lib.fxg_vdifmux(ctx, C.byref(d), src.ctypes.data, None, src.size, C.c_void_p(p.value + offset), d0.size,
                             -1, C.byref(st))
        out = np.zeros(d0.size, np.uint8)
        check(lib, lib.fxg_memcpy_d2h(ctx, out.ctypes.data, C.c_void_p(p.value + offset), d0.size), "d2h")
        lib.fxg_device_free(ctx, p)
        assert (r1, st.as_list()) == (r0, s0)
        used = s0[12]
        assert used > 0 and np.array_equal(out[:used], d0[:used]), (framebytes, flags)
