"""The work that users of this correlator have it do, as cases that can be timed.

A case is one subintegration of one job (`fxg_subint_process`: raw VDIF or
Mark5B frames in device memory in, the slot's result buffer out), or one call
of the VDIF thread multiplexer (`fxg_vdifmux`: host bytes in, frames in device
memory out).  `listed()` names the cases, `draw()` gives others of the same
ranges, `prepare()` makes what a correlator process holds before the call (the
job handle, the frames, the result buffer), `run()` is one call, `work()` the
bytes and operations it cannot do without, and `exact()` the result in 64 bits
by torch alone.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "difx-svn2git-try3_amd"))
import fxcorr  # noqa: E402
import fxsynth  # noqa: E402
from fxcorr import JobSpec, PlanInfo, check  # noqa: E402

DEV = "cuda:0"
FORMATS = {"vdif": fxcorr.FXG_FORMAT_VDIF, "mark5b": fxcorr.FXG_FORMAT_MARK5B}


def _subint(name, stations, subbands, mhz, chans, blocks, xmac, bits=2, graph=False, sampling="real", order=1,
            fmt="vdif", bad=0.0, pcal=0.0, zoom=False, avg=1, framebytes=8032):
    case = dict(kind="subint", stations=stations, subbands=subbands, mhz=float(mhz), chans=chans, blocks=blocks,
                xmac=xmac, bits=bits, graph=graph, sampling=sampling, order=order, fmt=fmt, bad=bad, pcal=float(pcal),
                zoom=zoom, avg=avg, framebytes=10016 if fmt == "mark5b" else framebytes)
    if name:
        case["name"] = name
    return case


def _mux(name, threads, frames, bits, framebytes):
    case = dict(kind="mux", threads=threads, frames=frames, bits=bits, framebytes=framebytes)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # the smallest call: a few blocks of a three-station test job (the size
        # of smoke()), where launches, table copies and the wait are the time
        _subint("small_3st_256ch_fp32", 3, 2, 16, 256, 8, "fp32"),
        # a four-station spectral-line-free experiment at the CPU correlator's
        # traditional 256 channels, one-second subintegration
        _subint("vlbi_4st_256ch_fp32", 4, 1, 16, 256, 62500, "fp32"),
        # a ten-station network, 8 x 32 MHz, drop-in FP32 arithmetic
        _subint("vlbi_10st_1024ch_fp32", 10, 8, 32, 1024, 4096, "fp32"),
        # the serving mix's 20- and 32-station jobs, 8 x 64 MHz, 125 ms
        # subintegrations replayed as graphs
        _subint("serve_20st_4096ch_fp16", 20, 8, 64, 4096, 1953, "fp16", graph=True),
        _subint("serve_32st_8192ch_fp16", 32, 8, 64, 8192, 976, "fp16", graph=True),
        # the benchmark's default workload, mixed precision (128 ms)
        _subint("head_32st_4096ch_fp16", 32, 16, 64, 4096, 2000, "fp16", graph=True),
        # and its plain FP32 form on a quarter of the subintegration
        _subint("head_32st_4096ch_fp32", 32, 16, 64, 4096, 500, "fp32", graph=True),
        # from the mix of uneven jobs: 8-bit samples at few channels with zoom
        # bands, and the longest transforms (65536 points)
        _subint("mix_7st_256ch_8bit_zoom", 7, 8, 32, 256, 16000, "fp16", bits=8, zoom=True),
        _subint("mix_30st_32768ch_fp16_zoom", 30, 4, 128, 32768, 500, "fp16", zoom=True, graph=True),
        # double-sideband complex samples from a digital back end
        _subint("dsb_8st_1024ch_fp32", 8, 4, 32, 1024, 4001, "fp32", sampling="complex_dsb"),
        # Mark5B recordings with one bad frame in a hundred and 1 MHz phase cal
        _subint("mark5b_6st_512ch_lossy_pcal", 6, 4, 16, 512, 8001, "fp32", fmt="mark5b", bad=0.01, pcal=1.0),
        # eight single-channel VDIF threads of a second's recording to one
        # eight-channel stream
        _mux("mux_8_threads_2bit", 8, 4000, 2, 8032),
    ]


def draw(rng):
    if rng.random() < 0.08:
        threads = rng.choice([2, 3, 4, 5, 8, 11, 16])
        frames = int(2.0 ** rng.uniform(3.0, 12.0)) | 1
        return _mux(None, threads, frames, rng.choice([2, 2, 8]), rng.choice([1032, 5032, 8032]))
    sampling = rng.choice(["real"] * 6 + ["complex", "complex_dsb"])
    chans = 2 ** (rng.randint(7, 14) if sampling != "real" else rng.randint(6, 15))
    stations = int(round(2.0 ** rng.uniform(1.0, 5.0)))
    subbands = rng.choice([1, 2, 4, 8, 16])
    bits = rng.choice([2, 2, 2, 8])
    fmt = "vdif"
    if sampling != "real":
        subbands = min(subbands, 8)
    elif bits == 2 and subbands <= 8 and rng.random() < 0.15:
        fmt = "mark5b"
    xmac = rng.choice(["fp32", "fp16", "fp16", "bf16"])
    order = rng.choice([1, 1, 1, 1, 1, 0, 2]) if sampling == "real" else rng.choice([1, 1, 1, 2])
    length = chans if sampling != "real" else 2 * chans
    per_block = stations * 2 * subbands * length
    blocks = int(2.0 ** rng.uniform(20.0, 31.5) / per_block)
    # reduced precision is for long integrations, and no subintegration is
    # longer than a second or so
    blocks = max(64 if xmac != "fp32" else 3, min(blocks, 40000))
    bad = 0.01 if bits == 2 and rng.random() < 0.12 else 0.0
    pcal = 1.0 if sampling == "real" and length <= 8192 and rng.random() < 0.12 else 0.0
    zoom = sampling == "real" and chans >= 256 and rng.random() < 0.2
    avg = rng.choice([1, 1, 1, 2, 4]) if not zoom else 1
    return _subint(None, stations, subbands, rng.choice([16, 32, 64, 128]), chans, blocks, xmac, bits=bits,
                   graph=rng.random() < 0.4, sampling=sampling, order=order, fmt=fmt, bad=bad, pcal=pcal, zoom=zoom,
                   avg=avg)


# ---------------------------------------------------------------------------
# the job and its data
# ---------------------------------------------------------------------------
def _spec(case):
    nchan = case["chans"]
    zoom = ()
    if case["zoom"]:                       # two windows of a sixteenth of a subband, as in the mix of uneven jobs
        w = nchan // 16
        zoom = [(0, nchan // 4, w), (case["subbands"] - 1, nchan // 2 + w // 2, w)]
    fmt = FORMATS[case["fmt"]]
    return JobSpec(nstations=case["stations"], nsubbands=case["subbands"], npol=2, bw_mhz=case["mhz"], nchan=nchan,
                   nbits=case["bits"], blockspersend=case["blocks"], crosspol=True, xmac=case["xmac"],
                   framebytes=case["framebytes"], headerbytes=16 if case["fmt"] == "mark5b" else 32, fmt=fmt,
                   base_freq_mhz=8200.0, fringe_order=case["order"], chans_to_avg=case["avg"], zoom=zoom,
                   pcal_interval_mhz=case["pcal"], sampling=case["sampling"],
                   # a subintegration's spectra stay resident as a whole where a
                   # user with this card's memory would keep them
                   max_chunk_blocks=case["blocks"] if case["graph"] and nchan <= 8192 else 0)


def _geometry(case, spec, seed):
    """Delays, rates and times of the stations, from the seed alone."""
    rng = np.random.default_rng(seed)
    ts = spec.sampletime_us
    L, fs, nst = spec.fftchannels, spec.framesamples, spec.nstations
    delays = [int(v) & ~3 for v in rng.integers(-2000, 2000, nst)]
    nsamp = spec.blockspersend * L
    block_s = L * ts * 1e-6
    rates = rng.uniform(-1.0, 1.0, nst)                               # us of delay per second
    drift = np.abs(rates).max() * nsamp * ts * 1e-6 / ts              # samples over the subintegration
    guard = (2000 + int(drift) + 2 * L + fs - 1) // fs + 1
    while abs(guard * fs * ts * 1000.0 - round(guard * fs * ts * 1000.0)) > 1e-6:
        guard += 1                                                    # the data start on a whole nanosecond
    nframes = (nsamp + fs - 1) // fs + 2 * guard + 1
    start_ns = int(round(10 * 1_000_000_000 - guard * fs * ts * 1000.0))
    sec, ns = divmod(start_ns, 1_000_000_000)
    interp = []
    for s in range(nst):
        # a fraction of a sample off the data, and a slow curvature
        frac = rng.uniform(-0.5, 0.5) * ts
        interp.append([rng.uniform(-1e-3, 1e-3) * block_s * block_s, rates[s] * block_s, delays[s] * ts + frac])
    bad = []
    for s in range(nst):
        bad.append(np.nonzero(rng.random(nframes) < case["bad"])[0] if case["bad"] else np.empty(0, np.int64))
    return dict(delays=delays, nframes=nframes, sec=int(sec), ns=int(ns), interp=interp, bad=bad)


def _random_bytes(n, gen):
    words = (n + 7) // 8
    v = torch.randint(-2 ** 63, 2 ** 63 - 1, (words,), dtype=torch.int64, generator=gen, device=DEV)
    return v.view(torch.uint8)[:n]


def _noise(nbytes, bits, gen):
    """Bytes of quantised unit-variance Gaussian samples."""
    if bits == 8:
        x = torch.randn(nbytes, generator=gen, device=DEV)
        return x.mul_(8.0).round_().add_(128.0).clamp_(0, 255).to(torch.uint8)
    out = torch.zeros(nbytes, dtype=torch.uint8, device=DEV)
    u = _random_bytes(4 * nbytes, gen).view(4, nbytes)
    for k in range(4):                     # thresholds at +-0.98 sigma: 16.4 % of the samples in each outer level
        c = (u[k] >= 42).to(torch.uint8) + (u[k] >= 128).to(torch.uint8) + (u[k] >= 214).to(torch.uint8)
        out |= c << (2 * k)
    return out


def _frames(case, spec, geo, seed):
    """Raw frames of every station: one sample in twenty comes from a common
    signal at the station's delay, the rest from the station's own noise."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed) * 7919 + 17)
    db = spec.framebytes - spec.headerbytes
    nb = geo["nframes"] * db
    bytes4 = 4 * spec.nrecbands * spec.unitbits // 8                  # bytes of four sample-times
    lo, hi = min(geo["delays"]), max(geo["delays"])
    common = _noise(nb + (hi - lo) // 4 * bytes4, case["bits"], gen)
    fps = int(round(1e6 / spec.sampletime_us)) // spec.framesamples
    first = int(round(geo["ns"] / 1000.0 / spec.sampletime_us)) // spec.framesamples
    raws = []
    for s in range(spec.nstations):
        own = _noise(nb, case["bits"], gen)
        at = (geo["delays"][s] - lo) // 4 * bytes4
        pick = _random_bytes(nb, gen) < 13
        payload = torch.where(pick, common[at:at + nb], own)
        del own, pick
        out = torch.empty((geo["nframes"], spec.framebytes), dtype=torch.uint8, device=DEV)
        out[:, spec.headerbytes:] = payload.view(geo["nframes"], db)
        del payload
        n = geo["nframes"]
        if case["fmt"] == "mark5b":
            w = np.zeros((n, 4), np.uint32)
            w[:, 0] = 0xABADDEED
            w[:, 1] = (first + np.arange(n)) % fps & 0x7FFF
            w[geo["bad"][s], 1] |= np.uint32(1 << 15)
            hdr = w.view(np.uint8).reshape(n, 16)
        else:
            hdr = fxsynth.vdif_headers(geo["sec"], first, n, fps, spec.framebytes, spec.nrecbands, spec.nbits, s)
            w = hdr.view(np.uint32)
            if spec.is_complex:
                w[:, 3] |= np.uint32(1 << 31)
            w[geo["bad"][s], 0] |= np.uint32(1 << 31)
        out[:, :spec.headerbytes] = torch.from_numpy(np.ascontiguousarray(hdr)).to(DEV)
        raws.append(out.view(-1))
    return raws


_ctx = None


def _context():
    """One library context for the process, as a correlator keeps it."""
    global _ctx
    lib = fxcorr.load_gpu_lib()
    if _ctx is None:
        c = C.c_void_p()
        check(lib, lib.fxg_ctx_create(0, C.byref(c)), "fxg_ctx_create")
        _ctx = c
    return lib, _ctx


class _Job:
    """A job handle that ends with its last reference."""

    def __init__(self, spec):
        self.lib, ctx = _context()
        self.desc, self.keep = spec.build()
        self.h = C.c_void_p()
        check(self.lib, self.lib.fxg_job_create(ctx, C.byref(self.desc), C.byref(self.h)), "fxg_job_create")
        info = PlanInfo()
        check(self.lib, self.lib.fxg_job_plan_info(self.h, C.byref(info)), "fxg_job_plan_info")
        self.length = info.result_length

    def __del__(self):
        if getattr(self, "h", None):
            self.lib.fxg_job_destroy(self.h)


def _inputs(spec, geo, raws):
    nb = spec.blockspersend
    per = fxcorr.FXG_FLAGS_PER_INT
    flags = np.full((nb + per - 1) // per, (1 << per) - 1, dtype=np.int32)
    if nb % per:
        flags[-1] = (1 << (nb % per)) - 1
    arr = (fxcorr.StationInput * spec.nstations)()
    for s in range(spec.nstations):
        a = arr[s]
        a.data, a.nbytes = raws[s].data_ptr(), raws[s].numel()
        a.scan, a.sec, a.ns = 0, geo["sec"], geo["ns"]
        a.nvalidflags = flags.size
        a.validflags = flags.ctypes.data_as(C.POINTER(C.c_int32))
        for k in range(3):
            a.interpolator[k] = geo["interp"][s][k]
    sub = fxcorr.SubintDesc()
    sub.sec, sub.model_ok = 10, 1
    return arr, sub, flags


def _mux_stream(case, seed):
    """Frames of every thread in turn, as a recorder interleaves them."""
    n, nt, fb = case["frames"], case["threads"], case["framebytes"]
    rng = np.random.default_rng(seed)
    fr = rng.integers(0, 2 ** 63, (n, nt, fb // 8), dtype=np.int64).view(np.uint8).reshape(n, nt, fb)
    w = fr[:, :, :32].copy().view(np.uint32).reshape(n, nt, 8)
    f = np.arange(n)[:, None]
    w[:] = 0
    w[:, :, 0] = 100 + f // 4000
    w[:, :, 1] = (f % 4000) | (20 << 24)
    w[:, :, 2] = fb // 8
    w[:, :, 3] = 7 | (np.arange(nt)[None, :] << 16) | ((case["bits"] - 1) << 26)
    fr[:, :, :32] = w.view(np.uint8).reshape(n, nt, 32)
    return np.ascontiguousarray(fr.reshape(-1))


def prepare(case, seed):
    if case["kind"] == "mux":
        lib, ctx = _context()
        d = fxcorr.VdifMuxDesc()
        d.input_frame_bytes, d.frames_per_second, d.bits_per_sample = case["framebytes"], 4000, case["bits"]
        d.nthreads, d.channels_per_thread = case["threads"], 1
        for t in range(case["threads"]):
            d.thread_ids[t] = t
        d.nsort = d.ngap = 2 * case["threads"]
        fb, nch = C.c_int32(), C.c_int32()
        check(lib, lib.fxg_vdifmux_output_shape(C.byref(d), C.byref(fb), C.byref(nch)), "fxg_vdifmux_output_shape")
        dest = torch.zeros(fb.value * case["frames"], dtype=torch.uint8, device=DEV)
        return dict(kind="mux", lib=lib, ctx=ctx, desc=d, src=_mux_stream(case, seed), dest=dest,
                    stats=fxcorr.VdifMuxStats())
    spec = _spec(case)
    geo = _geometry(case, spec, seed)
    raws = _frames(case, spec, geo, seed)
    job = _Job(spec)
    if case["graph"]:
        check(job.lib, job.lib.fxg_job_set_graph(job.h, 1), "fxg_job_set_graph")
    arr, sub, flags = _inputs(spec, geo, raws)
    result = torch.empty(2 * job.length, dtype=torch.float32, device=DEV)
    return dict(kind="subint", job=job, arr=arr, sub=sub, raws=raws, flags=flags, result=result,
                split=_layout(case, spec)["pcal"])


def run(state):
    if state["kind"] == "mux":
        src, dest = state["src"], state["dest"]
        used = state["lib"].fxg_vdifmux(state["ctx"], C.byref(state["desc"]), src.ctypes.data, None, src.size,
                                        C.c_void_p(dest.data_ptr()), dest.numel(), -1, C.byref(state["stats"]))
        if used < 0:
            raise RuntimeError("fxg_vdifmux: %d" % used)
        return {"frames": dest, "used": int(used)}
    job, r = state["job"], state["result"]
    check(job.lib, job.lib.fxg_subint_process(job.h, C.byref(state["sub"]), state["arr"], 1,
                                              C.c_void_p(r.data_ptr()), 1), "fxg_subint_process")
    out = {"result": r[:state["split"]]}
    if state["split"] < r.numel():
        out["tones"] = r[state["split"]:]
    return out


# ---------------------------------------------------------------------------
# the result buffer (Configuration::populateResultLengths) and the exact result
# ---------------------------------------------------------------------------
def _freqs(case, spec):
    """(parent subband, channel offset, channels) of every frequency."""
    return [(sb, 0, spec.nchan) for sb in range(spec.nsubbands)] + [tuple(z) for z in spec.zoom]


def _tones(case, spec, sb):
    """Phase-cal tone frequencies of a subband in Hz from its lower edge."""
    lo, bw, step = int(round(spec.base_freq_mhz + sb * spec.bw_mhz)), int(spec.bw_mhz), int(case["pcal"])
    return [1e6 * (f - lo) for f in range(lo // step * step, lo + bw + 1, step) if f > lo]


def _layout(case, spec):
    """Float offsets of the regions of the result buffer."""
    nst, fr = spec.nstations, _freqs(case, spec)
    nbl = nst * (nst - 1) // 2
    nout = [n // case["avg"] for _, _, n in fr]
    at = 0
    vis = []
    for n in nout:
        vis.append(at)
        at += nbl * 4 * n * 2
    bw = at
    at += len(fr) * nbl * 4                                           # four weights: two complex elements
    ac = at
    at += nst * 2 * 2 * sum(nout) * 2                                 # two passes of two polarisations
    acw = at
    at += nst * 4 * len(fr)
    return dict(vis=vis, bweights=bw, autos=ac, aweights=acw, pcal=at, nout=nout)


def _decode(case, spec, raw, geo, s):
    """(sample-times, bands) of codes and the validity of each sample-time."""
    n = geo["nframes"]
    fr = raw.view(n, spec.framebytes)[:, spec.headerbytes:].reshape(-1)
    ub = spec.unitbits
    if case["bits"] == 8:
        codes = fr.view(torch.int16) if ub == 16 else fr
    elif ub == 4:
        codes = torch.stack([fr & 15, fr >> 4], 1).reshape(-1)
    else:
        codes = torch.stack([(fr >> (2 * k)) & 3 for k in range(4)], 1).reshape(-1)
    valid = torch.ones(n, dtype=torch.bool, device=raw.device)
    valid[torch.from_numpy(geo["bad"][s]).to(raw.device)] = False
    return codes.view(-1, spec.nrecbands), valid.repeat_interleave(spec.framesamples)


def _levels(case):
    if case["bits"] == 8:
        return (torch.arange(256, dtype=torch.float64, device=DEV) - 128.0) / 3.3
    hi = float(np.float32(3.3359))
    v = [-hi, 1.0, -1.0, hi] if case["fmt"] == "mark5b" else [-hi, -1.0, 1.0, hi]
    return torch.tensor(v, dtype=torch.float64, device=DEV)


def exact(case, seed):
    if case["kind"] == "mux":
        return None
    spec = _spec(case)
    nst, L, nchan, T = spec.nstations, spec.fftchannels, spec.nchan, spec.blockspersend
    if nst * spec.nrecbands * T * L > 2e10:
        return None
    geo = _geometry(case, spec, seed)
    raws = _frames(case, spec, geo, seed)
    lay, fr, avg = _layout(case, spec), _freqs(case, spec), case["avg"]
    cplx, dsb = spec.is_complex, spec.sampling == "complex_dsb"
    levels = _levels(case)
    ts, bw = spec.sampletime_us, spec.bw_mhz
    idx = torch.arange(T, dtype=torch.float64, device=DEV)
    nL = torch.arange(L, dtype=torch.float64, device=DEV) / L
    freq = torch.arange(nchan, dtype=torch.float64, device=DEV) * bw / nchan - (bw / 2 if dsb else 0.0)
    geom, weight, codes = [], torch.zeros(nst, T, dtype=torch.float64, device=DEV), []
    samples = torch.arange(L, device=DEV)
    for s in range(nst):
        q2, q1, q0 = geo["interp"][s]
        mid = q2 * (idx + 0.5) ** 2 + q1 * (idx + 0.5) + q0
        start = (10 - geo["sec"]) * 1e6 + (0 - geo["ns"]) / 1000.0 + idx * L * ts - mid
        near = torch.floor(start / ts + 0.5)
        d0 = q2 * idx ** 2 + q1 * idx + q0
        d2 = q2 * (idx + 1) ** 2 + q1 * (idx + 1) + q0
        a = d2 - d0
        geom.append((near.long(), start - near * ts, a, d0 + (mid - (a * 0.5 + d0)) / 3.0, mid))
        c, v = _decode(case, spec, raws[s], geo, s)
        codes.append((c, v))
        good = torch.cat([torch.zeros(1, dtype=torch.int64, device=DEV), torch.cumsum(v, 0)])
        weight[s] = (good[geom[s][0] + L] - good[geom[s][0]]).double() / L
    res = torch.zeros(lay["pcal"], dtype=torch.float64, device=DEV)
    pcal = []
    pairs = [(i, j) for i in range(nst) for j in range(i + 1, nst)]
    pi = torch.tensor([2 * i + p for i, j in pairs for p in (0, 0, 1, 1)], device=DEV)
    pj = torch.tensor([2 * j + p for i, j in pairs for p in (0, 1, 0, 1)], device=DEV)
    ai = torch.tensor([2 * s + p for s in range(nst) for p in (0, 1)], device=DEV)
    nac = 2 * sum(lay["nout"])                                        # values of one pass of one station
    mean = lambda x: x.view(x.shape[0], -1, avg).mean(2)  # noqa: E731
    tones = {}
    step = max(1, int(2 ** 26 // max(L, 1)))
    for sb in range(spec.nsubbands):
        X = torch.zeros(2 * nst, T, nchan, dtype=torch.complex128, device=DEV)
        lo = spec.base_freq_mhz + sb * bw + (bw / 2 if dsb else 0.0)
        for s in range(nst):
            near, fse, a, b, mid = geom[s]
            c, v = codes[s]
            ip = geo["interp"][s]
            for t0 in range(0, T, step):
                t1 = min(T, t0 + step)
                at = near[t0:t1, None] + samples[None]
                if case["order"] == 1:
                    ph = lo * (a[t0:t1, None] * nL[None] + b[t0:t1, None])
                elif case["order"] == 2:
                    i = idx[t0:t1, None]
                    ph = lo * (ip[0] * (i + nL[None]) ** 2 + ip[1] * (i + nL[None]) + ip[2])
                else:
                    ph = lo * mid[t0:t1, None]
                rot = torch.polar(torch.ones_like(ph), -2 * math.pi * (ph - torch.floor(ph)))
                frac = 2 * math.pi * freq[None] * fse[t0:t1, None]
                frac = torch.polar(torch.ones_like(frac), frac)
                for p in range(2):
                    code = c[:, 2 * sb + p][at].long()
                    if cplx:
                        nb = case["bits"]
                        x = torch.complex(levels[code & ((1 << nb) - 1)], levels[(code >> nb) & ((1 << nb) - 1)])
                    else:
                        x = levels[code]
                    x = x * v[at]
                    if case["pcal"]:
                        fs = int(round(1e6 / ts))
                        so = at + int(geo["ns"] / (ts * 1e3) + 0.5)
                        xr = torch.where(weight[s, t0:t1, None] > 0, x, torch.zeros_like(x)).reshape(-1)
                        bins = torch.zeros(int(2 * bw), dtype=torch.float64, device=DEV)
                        bins.index_add_(0, (so % bins.numel()).reshape(-1), xr)
                        key = (s, sb, p)
                        tones[key] = tones.get(key, 0) + bins
                    y = torch.fft.fft(x * rot)
                    if dsb:
                        y = torch.roll(y, -(nchan // 2), 1)
                    X[2 * s + p, t0:t1] = y[:, :nchan] * frac
        for f, (parent, off, n) in enumerate(fr):
            if parent != sb:
                continue
            V = torch.empty(2 * nst, 2 * nst, n, dtype=torch.complex128, device=DEV)
            for c0 in range(0, n, 256):
                c1 = min(n, c0 + 256)
                M = X[:, :, off + c0:off + c1].permute(2, 0, 1).contiguous()
                V[:, :, c0:c1] = torch.matmul(M, M.conj().transpose(1, 2).resolve_conj().contiguous()).permute(1, 2, 0)
                del M
            no = lay["nout"][f]
            if pairs:
                res[lay["vis"][f]:lay["vis"][f] + len(pairs) * 8 * no] = torch.view_as_real(mean(V[pi, pj])).reshape(-1)
            before = 2 * sum(lay["nout"][:f])
            for k, other in ((0, ai), (1, ai ^ 1)):
                A = torch.view_as_real(mean(V[ai, other])).reshape(nst, -1)
                for s in range(nst):
                    o = lay["autos"] + 2 * (s * 2 * nac + k * nac + before)
                    res[o:o + A.shape[1]] = A[s]
            del V
        del X
    nf = len(fr)
    if pairs:
        wb = torch.stack([(weight[i] * weight[j]).sum() for i, j in pairs])
        res[lay["bweights"]:lay["bweights"] + nf * len(pairs) * 4] = wb[:, None].expand(-1, 4).reshape(-1).repeat(nf)
    res[lay["aweights"]:lay["pcal"]] = weight.sum(1)[:, None].expand(-1, 4 * nf).reshape(-1)
    out = {"result": res}
    if case["pcal"]:
        fs = 2 * bw                                                   # whole MHz: the tones repeat every fs samples
        for s in range(nst):
            for sb in range(spec.nsubbands):
                fk = torch.tensor(_tones(case, spec, sb), dtype=torch.float64, device=DEV) / 1e6
                m = torch.arange(int(fs), dtype=torch.float64, device=DEV)
                ph = fk[:, None] * m[None] % fs / fs
                w = torch.polar(torch.ones_like(ph), -2 * math.pi * ph)
                for p in range(2):
                    pcal.append(torch.view_as_real(w @ tones[(s, sb, p)].to(torch.complex128)).reshape(-1))
        out["tones"] = torch.cat(pcal)
    return out


def work(case):
    if case["kind"] == "mux":
        units = 1
        while units < case["threads"]:
            units *= 2
        n, db = case["frames"], case["framebytes"] - 32
        return {"bytes": float(n * (case["threads"] * case["framebytes"] + units * db + 32)), "flops": 0.0}
    spec = _spec(case)
    L, nin, T = spec.fftchannels, 2 * spec.nstations, spec.blockspersend
    transforms = spec.nstations * spec.nrecbands * T
    raw = transforms * L * spec.unitbits / 8.0
    chans = sum(n for _, _, n in _freqs(case, spec))
    result = 4.0 * _layout(case, spec)["pcal"]
    # an L-point transform of real samples (half a complex one), a rotation of
    # every sample and of every channel, and each product of a pair once
    per = (5.0 if spec.is_complex else 2.5) * L * math.log2(L) + 6.0 * L + 6.0 * spec.nchan
    return {"bytes": raw + result, "flops": transforms * per + 8.0 * chans * T * nin * (nin + 1) / 2}
