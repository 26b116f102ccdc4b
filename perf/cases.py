"""The work that programs have this framework do, as timed cases.

Every case is a pass over the public entry points of gcorr_amd with inputs
made from a seed on the GPU (or, for the streamed case, in pinned host
memory).  `listed()` names the fixed cases, `draw(rng)` gives one more of the
same ranges, `prepare` builds what a program holds before the call, `run` is
one pass, `work` the bytes and operations the path cannot do without, and
`exact` the same outputs in 64 bits from plain torch and numpy.

One pass of a correlation case is one subintegration as a correlator runs
it: the input buffers and the delay model of that subintegration are handed
over, it is processed, and the visibilities (and the per-row FFT counts) are
read.  Small cases read them into host memory, as fxkernel's callers do;
large ones keep them on the GPU, as an imaging or averaging stage behind the
correlator does.
"""
import math

import numpy as np
import torch

import gcorr_amd

HIMAG = float(np.float32(3.3359))
THRESH = 0.98  # 2-bit decision level in sigma
DEV = "cuda"

# Bandwidth (Hz) and channels of the eight uneven subbands of the batched workload.
SUBBANDS = [(16e6, 256), (16e6, 512), (32e6, 512), (32e6, 1024), (64e6, 1024), (64e6, 2048),
            (128e6, 2048), (128e6, 4096)]


def _fx(name, nant, nchan, numffts, bw, **kw):
    c = dict(name=name, kind="fx", nant=nant, nchan=nchan, numffts=numffts, bw=bw, lo=1.65e9,
             precision="fp32", autos=True, exact_phase=False, is_complex=False, fblock=0, xtile=0,
             xsplits=0, host=False)
    c.update(kw)
    return c


def listed():
    return [
        # A look at a few milliseconds of three stations while an array is set
        # up: the call itself is what costs.
        _fx("quicklook_3st_256ch", 3, 256, 64, 16e6, host=True),
        # A small array at 32 MS/s, one tenth of a second, fxkernel's own call
        # sequence with the result in host memory.
        _fx("small_4st_128ch", 4, 128, 12500, 16e6, host=True),
        # Six stations x 64 MHz x 1024 channels, one second, a handle with
        # default launch shapes (what FxKernel and the command line make).
        _fx("mid_6st_1024ch", 6, 1024, 62500, 64e6),
        # Sixteen stations x 128 MHz x 4096 channels, half a second, with the
        # launch shapes an earlier tuning run wrote down.
        _fx("large_16st_4096ch_tuned", 16, 4096, 15625, 128e6, fblock=256, xtile=16, xsplits=8),
        # The same in FP16 with the matrix-core F-stage.
        _fx("large_16st_4096ch_fp16_tuned", 16, 4096, 15625, 128e6, precision="fp16", fblock=-1, xtile=32,
            xsplits=8),
        # An odd array size and FFT count, BF16 spectra, the exact phase law, a
        # local oscillator off the whole hertz, result in host memory.
        _fx("odd_10st_2048ch_bf16", 10, 2048, 5001, 64e6, precision="bf16", exact_phase=True,
            lo=1.4204057517e9, host=True),
        # Spectral-line channels on a complex 8-bit sampler: the longest FFT.
        _fx("line_8st_32768ch_cplx_fp16", 8, 32768, 1000, 512e6, precision="fp16", is_complex=True),
        # Many stations with few channels on complex 8-bit data.
        _fx("many_32st_1024ch_cplx", 32, 1024, 6000, 64e6, is_complex=True, exact_phase=True),
        # Eight uneven subbands of one observation, 0.25 s, in one batch.
        dict(name="batch_8sub_8st", kind="batch", nant=8, seconds=0.25, nsub=8, precision="fp32", autos=True,
             fstage_mfma=0),
        # Recorded VDIF frames with a few lost ones, circular feeds made from
        # linear ones, and the fringe check an observer looks at.
        dict(name="vdif_fringe_5st_512ch", kind="vdif", nant=5, nchan=512, numffts=20000, bw=32e6, lo=1.65e9,
             payload=8000, lost=0.0005),
        # Subintegrations arriving in pinned host memory, summed on the GPU.
        dict(name="stream_4st_1024ch", kind="stream", nant=4, nchan=1024, numffts=8000, bw=64e6, lo=1.65e9,
             subints=3),
        # Filterbank voltages packed to 2 bits for the correlator.
        dict(name="requantise_2bit", kind="requant2", nsamples=100_000_002, threshold=0.98),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["small", "mid", "mid", "tuned", "reduced", "cplx", "many", "batch", "vdif", "stream", "requant2"])
    lo = rng.choice([1.65e9, 1.4204057517e9, 8.4e9 + 0.25])
    if kind == "requant2":
        return dict(kind="requant2", nsamples=2 * _log_int(rng, 500_000, 60_000_000), threshold=rng.uniform(0.8, 1.1))
    if kind == "batch":
        return dict(kind="batch", nant=rng.randint(3, 12), seconds=rng.uniform(0.02, 0.15), nsub=rng.randint(2, 8),
                    precision=rng.choice(["fp32", "fp32", "fp16"]), autos=True, fstage_mfma=rng.choice([0, 2]))
    if kind == "vdif":
        nchan = 2 ** rng.randint(7, 11)
        nant = rng.randint(2, 8)
        return dict(kind="vdif", nant=nant, nchan=nchan, numffts=_numffts(rng, nant, 2 * nchan, 2e7, 4e8), bw=32e6,
                    lo=lo, payload=8 * rng.randint(250, 1000), lost=10 ** rng.uniform(-4, -2.5))
    if kind == "stream":
        nchan = 2 ** rng.randint(7, 12)
        nant = rng.randint(2, 8)
        return dict(kind="stream", nant=nant, nchan=nchan, numffts=_numffts(rng, nant, 2 * nchan, 2e7, 2e8), bw=64e6,
                    lo=lo, subints=rng.randint(2, 5))
    bw = rng.choice([16e6, 32e6, 64e6, 128e6])
    c = _fx("", 0, 0, 0, bw, lo=lo, exact_phase=rng.random() < 0.3)
    del c["name"]
    if kind == "small":
        c.update(nant=rng.randint(2, 6), nchan=2 ** rng.randint(5, 11), autos=rng.random() < 0.5, host=True)
        c["numffts"] = _numffts(rng, c["nant"], 2 * c["nchan"], 2e5, 1e7)
    elif kind == "mid":
        c.update(nant=rng.randint(2, 20), nchan=2 ** rng.randint(7, 14), host=rng.random() < 0.5)
        c["numffts"] = _numffts(rng, c["nant"], 2 * c["nchan"], 3e7, 1.5e9)
    elif kind == "tuned":
        c.update(nant=rng.randint(4, 16), nchan=2 ** rng.randint(10, 12), xsplits=rng.choice([4, 8, 16]))
        c["fblock"] = c["nchan"] // 16
        c["xtile"] = 16
        c["numffts"] = _numffts(rng, c["nant"], 2 * c["nchan"], 1e8, 2e9)
    elif kind == "reduced":
        c.update(nant=rng.randint(2, 16), nchan=2 ** rng.randint(8, 12), precision=rng.choice(["fp16", "bf16"]))
        if c["nchan"] >= 1024 and rng.random() < 0.4:
            c.update(fblock=-1)
        c["numffts"] = max(601, _numffts(rng, c["nant"], 2 * c["nchan"], 5e7, 1e9))
    elif kind == "cplx":
        c.update(nant=rng.randint(2, 12), nchan=2 ** rng.randint(8, 15), is_complex=True, bw=4 * bw,
                 precision=rng.choice(["fp32", "fp16"]))
        c["numffts"] = max(601, _numffts(rng, c["nant"], c["nchan"], 3e7, 4e8))
    else:
        c.update(nant=rng.randint(17, 32), nchan=2 ** rng.randint(8, 11), precision=rng.choice(["fp32", "fp16"]))
        c["numffts"] = max(601, _numffts(rng, c["nant"], 2 * c["nchan"], 1e8, 6e8))
    return c


def _numffts(rng, nant, L, lo, hi):
    return max(17, min(60000, _log_int(rng, lo, hi) // (2 * nant * L)))


# ---- inputs -----------------------------------------------------------------

def _geom(nchan, numffts, bw, cplx):
    L = nchan if cplx else 2 * nchan
    Ts = 1.0 / bw if cplx else 0.5 / bw
    return L, Ts, (numffts + 1) * L


def _delays(nant, L, Ts, numffts, rng):
    """Quadratic delays of a few milliseconds, t in FFTs, and file offsets that
    leave a net delay of a few samples in mid-subintegration."""
    T = numffts * L * Ts
    Tf = L * Ts
    c0 = rng.uniform(-5e-3, 5e-3, nant)
    c1 = rng.uniform(-5e-7, 5e-7, nant)
    c2 = rng.uniform(-2.5e-7, 2.5e-7, nant) / T
    poly = np.stack([c2 * Tf * Tf, c1 * Tf, c0], axis=1)
    mid = T / 2
    offs = c2 * mid * mid + c1 * mid + c0 + rng.uniform(-3.0, 3.0, nant) * Ts
    return poly, offs


def _stations(nant, nchan, numffts, bw, lo, cplx, seed, rho=0.02):
    """Packed voltages of one subintegration: a common signal at the
    integer delay and fringe phase of each station, plus station noise."""
    L, Ts, n = _geom(nchan, numffts, bw, cplx)
    poly, offs = _delays(nant, L, Ts, numffts, np.random.default_rng(seed))
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    margin = 4096
    common = [torch.view_as_complex(torch.randn(n + 2 * margin, 2, generator=g, device=DEV)) for _ in range(2)]
    amp, noise = math.sqrt(rho), math.sqrt(1.0 - rho)
    out = []
    piece = 1 << 25
    for a in range(nant):
        buf = torch.empty(4 * n if cplx else n // 2, dtype=torch.uint8, device=DEV)
        p0, p1, p2 = (float(v) for v in poly[a])
        for s in range(0, n, piece):
            e = min(n, s + piece)
            k = torch.arange(s, e, device=DEV, dtype=torch.float64)
            u = k / L
            tau = (p0 * u + p1) * u + p2
            d = torch.round((tau - float(offs[a])) / Ts).clamp_(-margin, margin)
            idx = (k + d).long() + margin
            ph = (2 * math.pi * torch.remainder(lo * tau, 1.0)).float()
            fringe = torch.polar(torch.full_like(ph, amp), ph)
            pols = []
            for c in common:
                z = c[idx] * fringe
                if cplx:
                    w = torch.randn(e - s, 2, generator=g, device=DEV)
                    x = torch.view_as_real(z) * math.sqrt(0.5) + w * (noise * math.sqrt(0.5))
                    pols.append(torch.clamp(torch.round(x * 20.0), -127, 127).to(torch.int8))
                else:
                    x = z.real + torch.randn(e - s, generator=g, device=DEV) * noise
                    code = (x >= 0).to(torch.uint8) + 1
                    code += (x >= THRESH).to(torch.uint8)
                    code -= (x < -THRESH).to(torch.uint8)
                    pols.append(code)
            if cplx:
                buf[4 * s:4 * e] = torch.stack(pols, 1).reshape(-1).view(torch.uint8)
            else:
                A, B = pols
                buf[s // 2:e // 2] = A[0::2] | (B[0::2] << 2) | (A[1::2] << 4) | (B[1::2] << 6)
        out.append(buf)
    del common
    return out, poly, offs


def _batch_subbands(case):
    subs = []
    for bw, nchan in SUBBANDS[8 - case["nsub"]:]:
        subs.append((nchan, max(17, int(round(case["seconds"] * bw / nchan))), 1.65e9, bw))
    return subs


def _vdif_frames(buf, payload, fps, lost, seed):
    """32-byte headers before every payload, lost frames left out; the frames
    and the flag per slot."""
    n = -(-buf.numel() // payload)
    body = torch.zeros(n * payload, dtype=torch.uint8, device=DEV)
    body[:buf.numel()] = buf
    k = torch.arange(n, device=DEV, dtype=torch.int64)
    w = torch.zeros(n, 8, device=DEV, dtype=torch.int64)
    w[:, 0] = 100 + k // fps                     # seconds
    w[:, 1] = k % fps                            # frame within the second
    w[:, 2] = (1 << 24) | ((payload + 32) // 8)  # two channels, frame length
    w[:, 3] = 1 << 26                            # 2 bits, thread 0
    frames = torch.cat([w.to(torch.int32).view(torch.uint8).reshape(n, 32), body.reshape(n, payload)], 1)
    rng = np.random.default_rng(seed)
    ok = rng.random(n) >= lost
    return frames[torch.from_numpy(ok).to(DEV)].contiguous(), ok


def _gains(nant, nchan, seed):
    """Linear to circular with a few per cent of station and channel ripple."""
    rng = np.random.default_rng(seed + 3)
    g = np.empty((nant, 2, nchan), np.complex64)
    ripple = 1 + 0.03 * (rng.standard_normal((2, nant, nchan)) + 1j * rng.standard_normal((2, nant, nchan)))
    g[:, 0] = math.sqrt(0.5) * ripple[0]
    g[:, 1] = 1j * math.sqrt(0.5) * ripple[1]
    return g


class _DeviceArray:
    """The handle's visibilities in GPU memory, for torch.as_tensor; the
    tensor holds this object and so keeps the handle alive."""

    def __init__(self, k):
        self.owner = k
        ptr, shape = gcorr_amd.load().gxc_visibilities_device(k._h), (k.nrows, 4, k.nchan)
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<c8", "data": (ptr, False), "version": 3,
                                         "strides": None}


def _handle(c):
    return gcorr_amd.FxKernel(c["nant"], c["nchan"], c["numffts"], 8 if c["is_complex"] else 2, c["lo"], c["bw"],
                              c["is_complex"], precision=c["precision"], autos=c["autos"],
                              exact_phase=c["exact_phase"], fblock=c["fblock"], xtile=c["xtile"],
                              xsplits=c["xsplits"])


def _payload_fps(case):
    # frames per second of a stream whose seconds hold whole frames need not
    # follow the sample rate here: the time stamps only place the frames
    return 4000


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "fx":
        bufs, poly, offs = _stations(case["nant"], case["nchan"], case["numffts"], case["bw"], case["lo"],
                                     case["is_complex"], seed)
        st.update(bufs=bufs, ptrs=[b.data_ptr() for b in bufs], poly=poly, offs=offs, k=_handle(case))
        if not case["host"]:
            st["vis"] = torch.as_tensor(_DeviceArray(st["k"]), device=DEV)
    elif kind == "batch":
        subs = _batch_subbands(case)
        st["subs"] = []
        for i, (nchan, nfft, lo, bw) in enumerate(subs):
            bufs, poly, offs = _stations(case["nant"], nchan, nfft, bw, lo, False, seed * 16 + i)
            st["subs"].append((bufs, [b.data_ptr() for b in bufs], poly, offs))
        st["b"] = gcorr_amd.Batch(case["nant"], subs, precision=case["precision"], autos=case["autos"],
                                  fstage_mfma=case["fstage_mfma"])
    elif kind == "vdif":
        bufs, poly, offs = _stations(case["nant"], case["nchan"], case["numffts"], case["bw"], case["lo"], False, seed)
        fps = _payload_fps(case)
        st["frames"] = [_vdif_frames(b, case["payload"], fps, case["lost"], seed * 64 + a)[0]
                        for a, b in enumerate(bufs)]
        st.update(poly=poly, offs=offs, fps=fps)
        k = gcorr_amd.FxKernel(case["nant"], case["nchan"], case["numffts"], 2, case["lo"], case["bw"], autos=True)
        k.set_pol_conversion(_gains(case["nant"], case["nchan"], seed))
        st["k"] = k
    elif kind == "stream":
        st["sub"] = []
        for i in range(case["subints"]):
            bufs, poly, offs = _stations(case["nant"], case["nchan"], case["numffts"], case["bw"], case["lo"], False,
                                         seed * 8 + i)
            pins = [gcorr_amd.PinnedBuffer(b.numel()) for b in bufs]
            for p, b in zip(pins, bufs):
                p.array[:] = b.cpu().numpy()
            st["sub"].append((pins, [p.array for p in pins], poly, offs))
        st["k"] = gcorr_amd.FxKernel(case["nant"], case["nchan"], case["numffts"], 2, case["lo"], case["bw"],
                                     autos=True)
    else:
        g = torch.Generator(device=DEV)
        g.manual_seed(seed)
        n = case["nsamples"]
        st["pols"] = [torch.randn(n, generator=g, device=DEV) for _ in range(2)]
        st["out"] = torch.empty(n // 2, dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "fx":
        k = state["k"]
        k.setInputDevice(state["ptrs"], keepalive=state["bufs"])
        k.setDelays(state["poly"], state["offs"])
        k.process()
        return (k.visibilities() if case["host"] else state["vis"]), k.row_counts()
    if kind == "batch":
        b = state["b"]
        for i, (bufs, ptrs, poly, offs) in enumerate(state["subs"]):
            b.set_input_device(i, ptrs, keepalive=bufs)
            b.set_delays(i, poly, offs)
        b.process()
        return [(b.visibilities(i), b.row_counts(i)) for i in range(len(state["subs"]))]
    if kind == "vdif":
        k = state["k"]
        for a, f in enumerate(state["frames"]):
            k.setInputVDIF(a, f.data_ptr(), f.numel(), frames_per_second=state["fps"], ref_second=100,
                           frame_bytes=case["payload"] + 32, header_bytes=32, keepalive=f, stats=False)
        k.setDelays(state["poly"], state["offs"])
        k.process()
        snr, peak = k.lag_snr()
        return k.visibilities(), k.row_counts(), snr, peak
    if kind == "stream":
        k = state["k"]
        k.integrate_begin()
        for _, arrays, poly, offs in state["sub"]:
            k.submit(arrays, poly, offs)
        return k.integrate_end()[0]
    a, b = state["pols"]
    gcorr_amd.requantise_2bit(a.data_ptr(), b.data_ptr(), case["nsamples"], case["threshold"],
                              state["out"].data_ptr(), stream=torch.cuda.current_stream().cuda_stream)
    return state["out"]


# ---- work -------------------------------------------------------------------

def _fx_work(nant, nchan, numffts, cplx, autos, precision):
    """Packed samples in, visibilities out; 5 N log2 N for the FFTs, the two
    rotations, and the multiply-accumulate of every product (8 per term)."""
    L = nchan if cplx else 2 * nchan
    rows = nant * (nant - 1) // 2 + (nant if autos else 0)
    samples = 2.0 * nant * numffts * L
    read = samples * (2 if cplx else 0.25)
    flops = samples * (5 * math.log2(L) + 6) + 6.0 * 2 * nant * numffts * nchan + 8.0 * 4 * rows * nchan * numffts
    return read + rows * 4.0 * nchan * 8, flops


def work(case):
    kind = case["kind"]
    if kind == "fx":
        b, f = _fx_work(case["nant"], case["nchan"], case["numffts"], case["is_complex"], case["autos"],
                        case["precision"])
    elif kind == "batch":
        b = f = 0.0
        for nchan, nfft, _, _ in _batch_subbands(case):
            x = _fx_work(case["nant"], nchan, nfft, False, case["autos"], case["precision"])
            b, f = b + x[0], f + x[1]
    elif kind == "vdif":
        b, f = _fx_work(case["nant"], case["nchan"], case["numffts"], False, True, "fp32")
    elif kind == "stream":
        b, f = _fx_work(case["nant"], case["nchan"], case["numffts"], False, True, "fp32")
        b, f = b * case["subints"], f * case["subints"]
    else:
        b, f = case["nsamples"] * 8.5, case["nsamples"] * 6.0
    return {"bytes": b, "flops": f}


# ---- the same outputs in 64 bits ----------------------------------------------

def _fx64(bufs, poly, offs, nchan, numffts, bw, lo, cplx, exact_phase, autos, frame_ok=None, payload=0, gains=None):
    nant = len(bufs)
    L, Ts, _ = _geom(nchan, numffts, bw, cplx)
    s = 1 << (int(math.log2(nchan)) // 2)
    S2 = s if cplx else 2 * s
    stepmul = S2 if exact_phase else s
    maxoff = (numffts - 1) * L
    t = np.arange(numffts, dtype=np.float64)
    A, B, F, O, V = [], [], [], [], []
    for a in range(nant):
        c0, c1, c2 = (np.float64(v) for v in poly[a])
        d0 = c0 * t * t + c1 * t + c2
        th, t1 = t + 0.5, t + 1.0
        d1 = c0 * th * th + c1 * th + c2
        d2 = c0 * t1 * t1 + c1 * t1 + c2
        da = d2 - d0
        db = d0 + (d1 - (da * 0.5 + d0)) / 3.0
        ndf = (da * 0.5 + db - offs[a]) / Ts
        nd = np.trunc(ndf + 0.5)
        frac = -(ndf - nd) * Ts
        off = t.astype(np.int64) * L - nd.astype(np.int64)
        lo1, hi1 = off == -1, off == maxoff + 1
        off = off + lo1 - hi1
        frac = frac + lo1 * Ts - hi1 * Ts
        ok = (off >= 0) & (off <= maxoff)
        if frame_ok is not None:
            spf = payload * 2
            bad = np.concatenate([[0], np.cumsum(~frame_ok[a])])
            o = np.clip(off, 0, maxoff)
            ok &= bad[(o + L - 1) // spf + 1] == bad[o // spf]
        A.append(da), B.append(db), F.append(frac), O.append(np.clip(off, 0, maxoff)), V.append(ok)
    dev = lambda x: torch.from_numpy(np.stack(x)).to(DEV)
    A, B, F, O, valid = dev(A), dev(B), dev(F), dev(O), np.stack(V)
    okd = torch.from_numpy(valid).to(DEV)
    n = torch.arange(L, device=DEV)
    e = (n % S2).double() / L
    i = (n // S2 * stepmul).double() / L
    c = torch.arange(nchan, device=DEV, dtype=torch.float64) * (2 * math.pi * bw / nchan)
    lofrac = lo - math.trunc(lo)
    lv = torch.tensor([-HIMAG, -1.0, 1.0, HIMAG], dtype=torch.float64, device=DEV)
    M = 2 * nant
    R = torch.zeros(nchan, 2 * M, 2 * M, dtype=torch.float64, device=DEV)
    piece = max(1, int(6e8 // (M * L * 16)))
    for f0 in range(0, numffts, piece):
        f1 = min(numffts, f0 + piece)
        spec = torch.empty(f1 - f0, M, nchan, dtype=torch.complex128, device=DEV)
        for a in range(nant):
            ax, bx = A[a, f0:f1, None], B[a, f0:f1, None]
            whole = torch.trunc(bx)
            ph = (e[None] * ax + (bx - whole)) * lo
            if lofrac > 1e-11:
                ph = ph + lofrac * whole
            ph = torch.frac(ph) + torch.frac(i[None] * ax * lo)
            rot = torch.polar(torch.ones_like(ph), -2 * math.pi * ph)
            pos = O[a, f0:f1, None] + n[None]
            corr = torch.polar(torch.ones(f1 - f0, nchan, dtype=torch.float64, device=DEV), c[None] * F[a, f0:f1, None])
            corr = corr * okd[a, f0:f1, None]
            if cplx:
                w = bufs[a].view(torch.int8).view(-1, 4)[pos].double()
            else:
                w = bufs[a][pos // 2] >> (4 * (pos % 2)).to(torch.uint8)
            for p in range(2):
                if cplx:
                    x = torch.view_as_complex(w[..., 2 * p:2 * p + 2].contiguous())
                else:
                    x = lv[((w >> (2 * p)) & 3).long()]
                spec[:, 2 * a + p] = torch.fft.fft(x * rot, dim=1)[:, :nchan] * corr
        ri = torch.cat([spec.real, spec.imag], 1)
        R += torch.bmm(ri.permute(2, 1, 0).contiguous(), ri.permute(2, 0, 1).contiguous())
    rr, ii, ir = R[:, :M, :M], R[:, M:, M:], R[:, M:, :M]
    full = torch.complex(rr + ii, ir - ir.transpose(1, 2))
    rows = [(j, k) for j in range(nant) for k in range(j + 1, nant)] + ([(j, j) for j in range(nant)] if autos else [])
    counts = np.array([int((valid[j] & valid[k]).sum()) for j, k in rows], np.int32)
    vis = torch.empty(len(rows), 4, nchan, dtype=torch.complex128, device=DEV)
    for r, (j, k) in enumerate(rows):
        for p in range(4):
            vis[r, p] = full[:, 2 * j + p // 2, 2 * k + p % 2] / max(1, int(counts[r]))
    if gains is not None:
        G = torch.from_numpy(gains.astype(np.complex128)).to(DEV)
        J = torch.stack([torch.stack([G[:, 0], -G[:, 1]], 1), torch.stack([G[:, 0], G[:, 1]], 1)], 1)  # [ant][2][2][c]
        v = vis.view(len(rows), 2, 2, nchan).clone()
        for r, (j, k) in enumerate(rows):
            for l in range(2):
                for m in range(2):
                    vis[r, 2 * l + m] = sum(J[j, l, x] * v[r, x, y] * J[k, m, y].conj() for x in range(2) for y in range(2))
    return vis, counts


def exact(case, seed):
    kind = case["kind"]
    if kind == "fx":
        bufs, poly, offs = _stations(case["nant"], case["nchan"], case["numffts"], case["bw"], case["lo"],
                                     case["is_complex"], seed)
        vis, _ = _fx64(bufs, poly, offs, case["nchan"], case["numffts"], case["bw"], case["lo"], case["is_complex"],
                       case["exact_phase"], case["autos"])
        return (vis.cpu().numpy() if case["host"] else vis), None
    if kind == "batch":
        out = []
        for i, (nchan, nfft, lo, bw) in enumerate(_batch_subbands(case)):
            bufs, poly, offs = _stations(case["nant"], nchan, nfft, bw, lo, False, seed * 16 + i)
            vis, _ = _fx64(bufs, poly, offs, nchan, nfft, bw, lo, False, False, case["autos"])
            out.append((vis.cpu().numpy(), None))
        return out
    if kind == "vdif":
        bufs, poly, offs = _stations(case["nant"], case["nchan"], case["numffts"], case["bw"], case["lo"], False, seed)
        ok = [_vdif_frames(b, case["payload"], _payload_fps(case), case["lost"], seed * 64 + a)[1]
              for a, b in enumerate(bufs)]
        vis, _ = _fx64(bufs, poly, offs, case["nchan"], case["numffts"], case["bw"], case["lo"], False, False, True,
                       frame_ok=ok, payload=case["payload"], gains=_gains(case["nant"], case["nchan"], seed))
        lag = torch.fft.ifft(vis, dim=2).abs()
        snr = lag.amax(2) / lag.std(2, unbiased=False)
        return vis.cpu().numpy(), None, snr.cpu().numpy(), None
    if kind == "stream":
        total = None
        for i in range(case["subints"]):
            bufs, poly, offs = _stations(case["nant"], case["nchan"], case["numffts"], case["bw"], case["lo"], False,
                                         seed * 8 + i)
            vis, _ = _fx64(bufs, poly, offs, case["nchan"], case["numffts"], case["bw"], case["lo"], False, False, True)
            total = vis if total is None else total + vis
        return total.cpu().numpy()
    return None
