"""The work that users of sdbe_amd have it do, as cases to be measured.

A case is a dict of plain values; ``prepare`` makes what a program holds before
the call (device inputs, a handle or plan, output buffers), ``run`` makes one
call through the Python entry points of ``sdbe_amd``.  Kinds:

spectra   SdbeStage.process_spectra: n_bp block-pols of int8 spectra -> VDIF frames
batch     process_blocks: a ragged batch of streams (beams x sidebands), every
          second one a lower sideband -> VDIF frames
group     SdbeStage.process_group: a group's shuffled packets with drops -> VDIF
          frames of both polarisations (what the hashpipe thread does per slot)
resample  SdbeStage.resample_f32: the resampled series as floats, with its
          mean and sigma (the verification code's entry)
unpack    SdbeStage.unpack_int8: a group's packets -> reordered int8 spectra
pfb       Pfb.forward / Pfb.inverse: 16384-channel polyphase filterbank
xcorr     XCorr.search: the FX fringe search of the verification scripts
reorder   reorder_2015: the 2015-format B-engine reorder

Rates: 0 is the 39 -> 64 resampler, 6 / 8 / 10 / 11 the band-trimmed presets.
Spectra are 2-bit quantised circular Gaussian noise with a tone at channel 5000
at -20 dB, as SWARM delivers them.
"""
import math

import numpy as np
import torch

from sdbe_amd import _lib as L
from sdbe_amd.formats import reorder_2015
from sdbe_amd.pfb import Pfb
from sdbe_amd.qa import XCorr
from sdbe_amd.stage import BatchStream, SdbeStage, process_blocks

NCH = 16384
LB = 32768
DEV = "cuda:0"
QUANT = 0.9816                       # 2-bit thresholds in units of sigma
POLICY = {"reference": L.THRESH_REFERENCE, "per_block": L.THRESH_PER_BLOCK, "fixed": L.THRESH_FIXED}
# MHz trimmed from DC where the preset's band allows
SKIP = {0: 0, 6: 150, 8: 150, 10: 16, 11: 150}
# samples out per snapshot block / 2 bits each: frames per block-pol
SAMPLES = {0: 2097152, 6: 1048576, 8: 262144, 10: 2097152, 11: 4194304}


def _snaps(rate):
    return 39 if rate == 0 else L.TRIM_PRESETS[rate][0]


def listed():
    return [
        # one block of one polarisation: the smallest unit of work, handed in as
        # it arrives (what a program pays in latency per block)
        dict(name="spectra_1", kind="spectra", rate=0, n_bp=1, policy="reference"),
        # a live site: 3 beams x 2 sidebands, one block of each per call, the
        # launches captured in a graph
        dict(name="batch_6x1", kind="batch", blocks="1,1,1,1,1,1", policy="per_block", graph=True),
        # one slot of the stage at the full rate: 39 B-frames, 256 block-pols
        dict(name="group_64_39", kind="group", rate=0, geometry=0, drop=0.001, policy="per_block"),
        # the same slot in the band-trimmed thread, lowest and highest SWARM rate
        dict(name="group_6_11", kind="group", rate=6, geometry=0, drop=0.001, policy="reference"),
        dict(name="group_11_11", kind="group", rate=11, geometry=0, drop=0.001, policy="reference"),
        # recorded scans of uneven length, processed together
        dict(name="batch_ragged", kind="batch", blocks="17,64,128,5,200,33", policy="per_block", graph=False),
        # verification: float samples of an odd number of block-pols
        dict(name="resample_33", kind="resample", rate=0, n_bp=33),
        # the unpack alone: one slot's packets to int8 spectra
        dict(name="unpack_group", kind="unpack", rate=0, geometry=0, drop=0.001),
        # recovering the R2DBE-like time series from channelised data: a scan of
        # 4096 spectra each way
        dict(name="pfb_forward_4096", kind="pfb", direction="forward", n=4096, window="hann_sinc"),
        dict(name="pfb_inverse_4096", kind="pfb", direction="inverse", n=4096, window="hann_sinc"),
        # fringe search over +-128 windows, 256 averaged (the checker's default capacity)
        dict(name="xcorr_257x256", kind="xcorr", offsets=257, avg=256),
        # a group of 39 B-frames in the 2015 format
        dict(name="reorder_2015_39", kind="reorder", frames=39),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["spectra", "batch", "group", "resample", "unpack", "pfb", "pfb", "xcorr", "reorder"])
    rate = rng.choice([0, 0, 0, 6, 8, 10, 11])
    if kind == "spectra":
        return dict(kind=kind, rate=rate, n_bp=_log_int(rng, 1, 256), policy=rng.choice(sorted(POLICY)))
    if kind == "batch":
        blocks = [_log_int(rng, 1, 74) for _ in range(rng.randint(1, 6))]
        return dict(kind=kind, blocks=",".join(str(b) for b in blocks), policy=rng.choice(sorted(POLICY)),
                    graph=rng.random() < 0.5)
    if kind == "group":
        return dict(kind=kind, rate=rate, geometry=rng.randint(0, 1), drop=round(rng.uniform(0.0, 0.02), 5),
                    policy=rng.choice(["reference", "per_block"]))
    if kind == "resample":
        return dict(kind=kind, rate=rate, n_bp=_log_int(rng, 1, 33))
    if kind == "unpack":
        return dict(kind=kind, rate=rate, geometry=rng.randint(0, 1), drop=round(rng.uniform(0.0, 0.02), 5))
    if kind == "pfb":
        return dict(kind=kind, direction=rng.choice(["forward", "inverse"]), n=_log_int(rng, 16, 4096),
                    window=rng.choice(["hann_sinc", "hamming"]))
    if kind == "xcorr":
        return dict(kind=kind, offsets=2 * _log_int(rng, 1, 128) + 1, avg=_log_int(rng, 4, 256))
    return dict(kind="reorder", frames=_log_int(rng, 2, 39))


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _codes(g, n_snap, n_comp):
    """2-bit codes [n_snap][16384][n_comp] (uint8) of unit-variance noise, every
    pair of components a complex value, with the tone at channel 5000."""
    p0 = 0.5 * (1.0 + math.erf(-QUANT / math.sqrt(2.0)))
    u = torch.rand((n_snap, NCH, n_comp), generator=g, device=DEV)
    c = (u >= p0).to(torch.uint8)
    c += u >= 0.5
    c += u >= 1.0 - p0
    z = torch.randn((n_snap, n_comp), generator=g, device=DEV) * math.sqrt(0.5)
    ph = 2.0 * math.pi * (0.0371 * torch.arange(n_snap, device=DEV))
    for i in range(n_comp):
        z[:, i] += 0.1 * (torch.cos(ph) if i % 2 == 0 else torch.sin(ph))
    t = QUANT * math.sqrt(0.5)
    c[:, 5000, :] = (z >= -t).to(torch.uint8) + (z >= 0) + (z >= t)
    return c


def _spectra(g, n_snap):
    """int8 [n_snap][16384][2 = (im, re)] of values code - 2."""
    out = torch.empty((n_snap, NCH, 2), dtype=torch.int8, device=DEV)
    for s in range(0, n_snap, 1024):
        out[s:s + 1024] = _codes(g, min(1024, n_snap - s), 2).to(torch.int8) - 2
    return out


def _packets(g, frames, geometry, drop, b_first):
    """A group's packets (uint8 [n][packet bytes]), shuffled, a fraction dropped."""
    per = 256 if geometry else 2048
    size = 32 + 8192 if geometry else 1056
    pk = torch.zeros((frames, per, size), dtype=torch.uint8, device=DEV)
    order = torch.tensor([3, 2, 1, 0, 7, 6, 5, 4], device=DEV)
    for f in range(frames):
        c = _codes(g, 128, 4)           # pol0 re, im, pol1 re, im
        byte = c[..., 3] | (c[..., 2] << 2) | (c[..., 1] << 4) | (c[..., 0] << 6)
        if geometry:
            pay = byte.reshape(16, 8, 16, 256, 4).flip(-1).permute(2, 0, 1, 3, 4)
        else:
            pay = byte.reshape(128, 128, 8, 2, 8)[..., order].permute(1, 3, 2, 0, 4)
        pk[f, :, 32:] = pay.reshape(per, size - 32)
    n = torch.arange(frames * per, device=DEV)
    fids = 16 if geometry else 8
    cid, fid, b = n % per // fids, n % fids, b_first + n // per
    w = torch.zeros((frames * per, 8), dtype=torch.int64, device=DEV)
    w[:, 0] = 1000 + n // 125000
    w[:, 1] = (n % 125000) | (30 << 24)
    w[:, 2] = size // 8
    w[:, 3] = 0x536D | (1 << 26)
    w[:, 4] = b >> 8
    w[:, 5] = cid | (fid << 16) | ((b & 0xFF) << 24)
    w[:, 6] = n
    w = torch.where(w >= 1 << 31, w - (1 << 32), w).to(torch.int32)
    pk = pk.reshape(frames * per, size)
    pk[:, :32] = w.view(torch.uint8)
    keep = torch.randperm(frames * per, generator=g, device=DEV)[int(round(drop * frames * per)):]
    return pk[keep]


def _window(kind):
    m = np.arange(4 * LB, dtype=np.float64)
    c = np.cos(2.0 * np.pi * m / (4 * LB - 1))
    if kind == "hamming":
        return (0.54 - 0.46 * c).astype(np.float32)
    return ((0.5 - 0.5 * c) * np.sinc((m - (4 * LB - 1) / 2.0) / LB)).astype(np.float32)


def _levels(g, shape):
    """2-bit quantised unit noise as values -3, -1, 1, 3."""
    u = torch.randn(shape, generator=g, device=DEV)
    return 2.0 * ((u >= -QUANT).float() + (u >= 0).float() + (u >= QUANT).float()) - 3.0


def _pfb_input(case, g):
    n = case["n"]
    if case["direction"] == "forward":
        return torch.randn(((n + 3) * LB,), generator=g, device=DEV)
    spec = torch.complex(_levels(g, (n, NCH + 1)), _levels(g, (n, NCH + 1)))
    spec.imag[:, 0] = 0.0
    spec.imag[:, NCH] = 0.0
    return spec


def _xcorr_input(case, g):
    """Two recordings of one signal, 37 samples and 2 windows apart, 2-bit."""
    n = case["offsets"] + case["avg"] + 1
    common = torch.randn((n + 4) * LB, generator=g, device=DEV)
    x0 = common[4 * LB:] + 0.5 * torch.randn(n * LB, generator=g, device=DEV)
    x1 = common[2 * LB - 37:2 * LB - 37 + n * LB] + 0.5 * torch.randn(n * LB, generator=g, device=DEV)
    t = QUANT * math.sqrt(1.25)
    q = [2.0 * ((x >= -t).float() + (x >= 0).float() + (x >= t).float()) - 3.0 for x in (x0, x1)]
    return q[0].contiguous(), q[1].contiguous()


def _stage(case, **kw):
    rate = case.get("rate", 0)
    st = SdbeStage(policy=POLICY[case.get("policy", "per_block")], out_mode=L.OUT_FRAMES, station="Sm", fixed=(0.6, 0.0),
                   rate_frac=rate, skip_mhz=SKIP[rate], packet_geometry=case.get("geometry", 0), **kw)
    st.set_state(secs=1000, df=0, ref_epoch=30, psn=1)
    return st


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    s = {"kind": kind}
    if kind in ("spectra", "resample"):
        n = case["n_bp"]
        st = _stage(case, chunk=min(256, n + (n & 1)), max_spectra=n)
        s["stage"] = st
        s["x"] = _spectra(g, n * st.snaps).reshape(n, st.snaps, NCH, 2)
        if kind == "spectra":
            s["out"] = torch.empty((n, st.frames, st.frame_bytes), dtype=torch.uint8, device=DEV)
    elif kind in ("group", "unpack"):
        st = _stage(case, max_spectra=1)
        s["stage"], s["b0"] = st, 1000
        s["pk"] = _packets(g, st.group_frames, case["geometry"], case["drop"], 1000)
        if kind == "group":
            s["out"] = st.group_out()
            s["bitmap"] = torch.zeros((st.group_frames, 16 if case["geometry"] else 256),
                                      dtype=torch.int16 if case["geometry"] else torch.uint8, device=DEV)
    elif kind == "batch":
        blocks = [int(b) for b in case["blocks"].split(",")]
        total = 2 * sum(blocks)
        st = _stage(case, chunk=min(256, total), max_spectra=1, max_batch=total, use_graph=case["graph"])
        s["stage"], s["streams"] = st, []
        for i, nb in enumerate(blocks):
            out = torch.empty((2, 64 * nb, st.frame_bytes), dtype=torch.uint8, device=DEV)
            s["streams"].append(BatchStream(_spectra(g, 39 * nb), _spectra(g, 39 * nb), out, flip=bool(i & 1),
                                            policy=POLICY[case["policy"]], fixed=(0.6, 0.0), latch_slot=i,
                                            station="Sm", rx=i & 1, secs=1000, ref_epoch=30))
    elif kind == "pfb":
        s["pfb"] = Pfb(_window(case["window"]), max_spectra=case["n"])
        s["call"] = s["pfb"].forward if case["direction"] == "forward" else s["pfb"].inverse
        s["x"] = _pfb_input(case, g)
    elif kind == "xcorr":
        s["xc"] = XCorr(max_windows=case["offsets"] + case["avg"] - 1, max_offsets=case["offsets"])
        s["x"] = _xcorr_input(case, g)
        s["args"] = (-(case["offsets"] // 2), case["offsets"], case["avg"])
    else:
        x = torch.randn((NCH, case["frames"], 128, 2), generator=g, device=DEV)
        s["x"] = torch.view_as_complex(x)
        s["out"] = torch.empty((case["frames"] - 1, 128, NCH + 1), dtype=torch.complex64, device=DEV)
    return s


def run(s):
    kind = s["kind"]
    if kind == "spectra":
        return s["stage"].process_spectra(s["x"], out=s["out"])
    if kind == "resample":
        return s["stage"].resample_f32(s["x"])
    if kind == "group":
        out = s["stage"].process_group(s["pk"].view(-1), s["pk"].shape[0], s["b0"], out=s["out"], bitmap=s["bitmap"])
        return [out, s["bitmap"]]
    if kind == "unpack":
        return s["stage"].unpack_int8(s["pk"].view(-1), s["pk"].shape[0], s["b0"])
    if kind == "batch":
        process_blocks(s["stage"], s["streams"])
        return [b.out for b in s["streams"]]
    if kind == "pfb":
        return s["call"](s["x"])
    if kind == "xcorr":
        return s["xc"].search(s["x"][0], s["x"][1], *s["args"])
    return reorder_2015(s["x"], out=s["out"])


# ---------------------------------------------------------- work of a pass
def _fft_flops(n):
    """Of a real transform of n points."""
    return 2.5 * n * math.log2(n)


def _bp_flops(rate):
    """Of the transforms of one block-pol."""
    d = _snaps(rate)
    if rate == 0:
        return d * _fft_flops(2 * NCH) + _fft_flops(d * 2 * NCH) + _fft_flops(SAMPLES[0])
    e = L.TRIM_PRESETS[rate][1]
    return d * _fft_flops(2 * NCH) + 128 * (_fft_flops(256 * d) + _fft_flops(256 * e))


def work(case):
    kind, rate = case["kind"], case.get("rate", 0)
    snap_bytes = 2 * NCH                                     # int8 spectrum of one polarisation
    frame_out = SAMPLES[rate] // 4 * 8224 // 8192            # 2-bit frames of a block-pol
    if kind == "spectra":
        n = case["n_bp"]
        return dict(bytes=n * (_snaps(rate) * snap_bytes + frame_out), flops=n * _bp_flops(rate))
    if kind == "resample":
        n = case["n_bp"]
        return dict(bytes=n * (_snaps(rate) * snap_bytes + 4 * SAMPLES[rate]), flops=n * _bp_flops(rate))
    if kind == "batch":
        n = 2 * sum(int(b) for b in case["blocks"].split(","))
        return dict(bytes=n * (39 * snap_bytes + frame_out), flops=n * _bp_flops(0))
    if kind in ("group", "unpack"):
        d = _snaps(rate)
        pk = d * (256 * 8224 if case["geometry"] else 2048 * 1056) * (1.0 - case["drop"])
        if kind == "unpack":
            return dict(bytes=pk + 2 * d * 128 * snap_bytes, flops=0)
        return dict(bytes=pk + 256 * frame_out, flops=256 * _bp_flops(rate))
    if kind == "pfb":
        n = case["n"]
        flops = n * (_fft_flops(LB) + (8 if case["direction"] == "forward" else 22) * LB)
        return dict(bytes=4 * (n + 3) * LB + 8 * n * (NCH + 1) + 16 * LB, flops=flops)
    if kind == "xcorr":
        o, a = case["offsets"], case["avg"]
        return dict(bytes=4 * LB * (o + 2 * a - 1 + o),
                    flops=(o + 2 * a - 1 + o) * _fft_flops(LB) + 8.0 * o * a * NCH)
    f = case["frames"]
    return dict(bytes=8 * 128 * (NCH * f + (NCH + 1) * (f - 1)), flops=0)


# ------------------------------------------------------------ 64-bit values
def _exact_resample(case, seed):
    rate, n = case["rate"], case["n_bp"]
    d = _snaps(rate)
    x = _spectra(_gen(seed), n * d).reshape(n, d, NCH, 2).double()
    series, stats = [], []
    for b in range(n):
        spec = torch.zeros((d, NCH + 1), dtype=torch.complex128, device=DEV)
        spec[:, :NCH] = torch.complex(x[b, ..., 1], x[b, ..., 0])
        spec[:, 0] = spec[:, 0].real.to(torch.complex128)
        t = torch.fft.irfft(spec, n=2 * NCH, dim=1).reshape(-1)
        if rate == 0:
            pad = torch.zeros(SAMPLES[0] // 2 + 1, dtype=torch.complex128, device=DEV)
            pad[:d * NCH + 1] = torch.fft.rfft(t)
            y = torch.fft.irfft(pad, n=SAMPLES[0])
        else:
            e = L.TRIM_PRESETS[rate][1]
            skip = int(SKIP[rate] * 1e6 / (4576e6 * rate / 11 / (256 * d)))
            part = torch.fft.rfft(t.reshape(128, 256 * d), dim=1)[:, skip:skip + 128 * e + 1].clone()
            part[:, 0] = part[:, 0].real.to(torch.complex128)
            part[:, -1] = part[:, -1].real.to(torch.complex128)
            y = torch.fft.irfft(part, n=256 * e, dim=1).reshape(-1)
        series.append(y)
        stats.append(torch.stack([y.mean(), y.std()]))
    return torch.stack(series), torch.stack(stats)


def _exact_forward(case, seed):
    n = case["n"]
    x = _pfb_input(case, _gen(seed)).double().reshape(n + 3, LB)
    w = torch.from_numpy(_window(case["window"])).to(DEV).double().reshape(4, LB)
    y = torch.zeros((n, LB), dtype=torch.float64, device=DEV)
    for p in range(4):
        y += w[p] * x[p:p + n]
    return torch.fft.rfft(y, dim=1)


def _exact_inverse(case, seed):
    """Minimum-norm x with P x = irfft(spec) per branch: x = P^T (P P^T)^-1 yh,
    the banded Cholesky of P P^T run over all branches at once."""
    n = case["n"]
    yh = torch.fft.irfft(_pfb_input(case, _gen(seed)).to(torch.complex128), n=LB, dim=1)
    w = torch.from_numpy(_window(case["window"])).to(DEV).double().reshape(4, LB)
    a = [(w[d:] * w[:4 - d]).sum(0) for d in range(4)]
    zero = torch.zeros(LB, dtype=torch.float64, device=DEV)
    rows = torch.empty((n, 4, LB), dtype=torch.float64, device=DEV)      # 1 / L(i, i), L(i, i - 1..3)
    u = torch.empty((n, LB), dtype=torch.float64, device=DEV)
    r1 = r2 = r3 = torch.stack([zero + 1.0, zero, zero, zero])
    u1 = u2 = u3 = zero
    for i in range(n):
        d3 = a[3] * r3[0] if i >= 3 else zero
        d2 = ((a[2] if i >= 2 else zero) - d3 * r2[1]) * r2[0]
        d1 = ((a[1] if i >= 1 else zero) - d3 * r1[2] - d2 * r1[1]) * r1[0]
        inv = torch.rsqrt(a[0] - d1 * d1 - d2 * d2 - d3 * d3)
        rows[i, 0], rows[i, 1], rows[i, 2], rows[i, 3] = inv, d1, d2, d3
        u[i] = (yh[i] - d1 * u1 - d2 * u2 - d3 * u3) * inv
        r3, r2, r1 = r2, r1, rows[i]
        u3, u2, u1 = u2, u1, u[i]
    z = torch.zeros((n + 6, LB), dtype=torch.float64, device=DEV)        # z[i] at row i + 3
    for i in range(n - 1, -1, -1):
        t = u[i].clone()
        for d in range(1, min(4, n - i)):
            t -= rows[i + d, d] * z[i + d + 3]
        z[i + 3] = t * rows[i, 0]
    x = torch.zeros((n + 3, LB), dtype=torch.float64, device=DEV)
    for p in range(4):
        x += w[p] * z[3 - p:3 - p + n + 3]
    return x.reshape(-1)


def _exact_xcorr(case, seed):
    o, avg = case["offsets"], case["avg"]
    x0, x1 = (x.double().reshape(-1, LB) for x in _xcorr_input(case, _gen(seed)))
    c = x0.shape[0] // 2 - avg // 2
    X0 = torch.fft.rfft(x0[c:c + avg], dim=1)[:, :NCH]
    lo = c - o // 2
    X1 = torch.fft.rfft(x1[lo:lo + o + avg - 1], dim=1)[:, :NCH]
    wt = torch.full((NCH,), 2.0, dtype=torch.float64, device=DEV)
    wt[0] = 1.0
    p0 = (X0.abs().square().mean(0) * wt).sum() / LB
    p1 = (X1.abs().square() * wt).sum(1)
    s = []
    for k in range(o):
        S = torch.zeros(NCH + 1, dtype=torch.complex128, device=DEV)
        S[:NCH] = (X0 * X1[k:k + avg].conj()).mean(0)
        S[0] = S[0].real.to(torch.complex128)
        s.append(torch.fft.irfft(S, n=LB) / torch.sqrt(p0 * p1[k:k + avg].mean() / LB))
    s = torch.stack(s)
    return s, s.abs().amax(1), s.std(1, unbiased=False)


def _exact_reorder(case, seed):
    """Channels 0-3 of every 8 lag two snapshots, snapshots 69.. come from the
    next B-frame, and a zero channel 16384 follows."""
    f = case["frames"]
    x = torch.randn((NCH, f, 128, 2), generator=_gen(seed), device=DEV)
    r = torch.view_as_complex(x).clone().reshape(NCH // 8, 8, f, 128)
    r[:, :4] = torch.roll(r[:, :4], -2, -1)
    r[..., 69:] = torch.roll(r[..., 69:], -1, -2)
    out = torch.zeros((f - 1, 128, NCH + 1), dtype=torch.complex128, device=DEV)
    out[..., :NCH] = r.reshape(NCH, f, 128)[:, :-1].permute(1, 2, 0)
    return out


def exact(case, seed):
    """What run() returns in 64 bits; None where outputs are whole numbers."""
    if case["kind"] == "reorder":
        return _exact_reorder(case, seed)
    if case["kind"] == "resample":
        return _exact_resample(case, seed)
    if case["kind"] == "xcorr":
        return _exact_xcorr(case, seed)
    if case["kind"] == "pfb":
        return (_exact_forward if case["direction"] == "forward" else _exact_inverse)(case, seed)
    return None
