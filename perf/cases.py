"""Workloads that stand for what programs do with this framework, each through
its public entry points (FusedOctCQT, TrainableCQT, SlicedCQT, Graphed).

A case is a dict of plain values:
  kind    fwd     FusedOctCQT analysis of a batch of slices
          bwd     FusedOctCQT synthesis from coefficient planes
          rt      analysis, then synthesis of its coefficients
          graph   the same round trip recorded once with Graphed
          train   TrainableCQT: fwd -> bwd -> MSE -> gradient of the signal
          eq      TrainableCQT: per-band gains between fwd and bwd -> MSE -> gradients of the gains
          sliced  SlicedCQT: whole signals, forward and inverse
          stream  SlicedCQT: stream_fwd -> stream_bwd, one hop at a time
  layout  index into LAYOUTS
  batch   slices (fwd .. eq) or signals (sliced, stream)
  length  samples per signal (sliced)
  hops    hops per pass (stream)
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flash-cqt_amd"))
from flash_cqt import Graphed, OctCQT, SlicedCQT  # noqa: E402
from flash_cqt.fused import FusedOctCQT  # noqa: E402
from flash_cqt.trainable import TrainableCQT  # noqa: E402

N = 65536
H = N // 4

# (octaves per group, bins per octave, sample rate): the headline layout, the
# layout with the most overflow bins, one at 48 kHz with wide windows, and a
# coarse-to-fine one from the layout sweep
LAYOUTS = (((3, 4, 2), (8, 16, 32), 44100), ((2, 5, 2), (4, 8, 64), 44100), ((4, 3), (12, 48), 48000),
           ((5, 5), (4, 64), 44100))


def listed():
    def case(name, kind, batch, layout=0, length=0, hops=0):
        return dict(name=name, kind=kind, batch=batch, layout=layout, length=length, hops=hops)
    return [
        case("round_trip_1", "rt", 1),                     # interactive use, one slice: launches and latency
        case("graph_round_trip_1", "graph", 1),            # the same slice served by a recorded graph
        case("round_trip_16", "rt", 16),                   # a small batch
        case("analysis_64", "fwd", 64),                    # feature extraction, planes kept
        case("synthesis_64", "bwd", 64),                   # rendering from stored coefficients
        case("round_trip_127", "rt", 127, layout=2),       # odd batch, another layout
        case("round_trip_512", "rt", 512),                 # offline corpus processing, past every cache
        case("train_16", "train", 16),                     # training step through both adjoints
        case("eq_gains_6", "eq", 6, layout=1),             # learnt per-band gains, edited blocks
        case("sliced_8x441000", "sliced", 8, length=441000),     # eight clips of 10 s
        case("sliced_1x7300001", "sliced", 1, length=7300001),   # one long recording, odd length
        case("stream_8x4", "stream", 8, hops=4),           # bounded-state streaming of eight signals
    ]


def draw(rng):
    kind = rng.choice(("rt", "rt", "fwd", "bwd", "graph", "train", "eq", "sliced", "sliced", "stream"))
    layout = rng.choice((0, 0, 0, 1, 2, 3))
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    c = dict(kind=kind, layout=layout, batch=1, length=0, hops=0)
    if kind in ("rt", "fwd", "bwd"):
        c["batch"] = log(1, 512)
    elif kind == "graph":
        c["batch"] = log(1, 32)
    elif kind in ("train", "eq"):
        c["batch"] = log(1, 64)
    elif kind == "sliced":
        c["batch"] = log(1, 16)
        c["length"] = log(20000, 7500000 // c["batch"])
    else:
        c["batch"] = log(1, 32)
        c["hops"] = rng.randint(1, 4)
    return c


# ------------------------------------------------------------ what a program keeps

def _device():
    return torch.device("cuda", torch.cuda.current_device())


@functools.lru_cache(maxsize=None)
def _engine(kind, layout):
    """The engine object of a program, built once and given every input."""
    octs, bins, fs = LAYOUTS[layout]
    dev = _device()
    if kind in ("sliced", "stream"):
        return SlicedCQT(octs, bins, fs=fs, sl_len=N, device=dev)
    cqt = OctCQT(list(octs), list(bins), fs=fs, audio_len=N, device=dev)
    return TrainableCQT(cqt, dev) if kind in ("train", "eq") else FusedOctCQT(cqt, dev)


@functools.lru_cache(maxsize=8)
def _recorded(layout, batch):
    """The round trip of one batch size as a recorded graph."""
    f = _engine("graph", layout)

    def round_trip(x):
        kr, ki = f.fwd(x)
        return kr, ki, f.bwd(kr, ki)
    return Graphed(round_trip, torch.zeros(batch, N, device=_device()))


def _audio(rows, length, fs, seed, device):
    """Tones of log-uniform frequency (43 Hz to 20 kHz) in noise, [rows, length] fp32."""
    gen = torch.Generator(device=device).manual_seed(seed)
    tones = 43.0 * (20000.0 / 43.0) ** torch.rand(rows, 4, 1, generator=gen, device=device)
    x = 0.3 * torch.randn(rows, length, generator=gen, device=device)
    t = torch.arange(length, device=device, dtype=torch.float32) / fs
    for i in range(4):
        # the phase is kept below one turn, so that fp32 holds it
        x += torch.sin(2 * math.pi * torch.remainder(tones[:, i].round() * t, 1.0))
    return x


def _inputs(case, seed, device):
    """The tensors of a case from its seed alone, on `device` (fp32 / complex64)."""
    kind, b = case["kind"], case["batch"]
    fs = LAYOUTS[case["layout"]][2]
    if kind in ("sliced", "stream"):
        length = case["length"] if kind == "sliced" else case["hops"] * (N // 2)
        return dict(x=_audio(b, length, fs, seed, device).view(b, 1, length))
    x = _audio(b, N, fs, seed, device)
    if kind == "bwd":
        k = _Exact(case["layout"], device).analysis(x.double())
        return dict(kr=k.real.float().contiguous(), ki=k.imag.float().contiguous())
    d = dict(x=x)
    if kind in ("train", "eq"):
        d["target"] = _audio(b, N, fs, seed + 7919, device)
    if kind == "eq":
        gen = torch.Generator(device=device).manual_seed(seed + 104729)
        d["gains"] = [0.5 + torch.rand(n, 1, generator=gen, device=device) for n, _, _ in _bank(case["layout"])[1][:-2]]
    return d


def prepare(case, seed):
    kind = case["kind"]
    s = dict(_inputs(case, seed, _device()), kind=kind)
    s["engine"] = _recorded(case["layout"], case["batch"]) if kind == "graph" else _engine(kind, case["layout"])
    if kind == "train":
        s["x"].requires_grad_(True)
    if kind == "eq":
        for g in s["gains"]:
            g.requires_grad_(True)
    if kind == "stream":
        s["chunks"] = [c.contiguous() for c in s["x"].split(N // 2, dim=-1)]
    return s


# ------------------------------------------------------------ one pass

def run(s):
    kind, e = s["kind"], s["engine"]
    if kind == "fwd":
        return e.fwd(s["x"])
    if kind == "bwd":
        return e.bwd(s["kr"], s["ki"])
    if kind == "rt":
        kr, ki = e.fwd(s["x"])
        return kr, ki, e.bwd(kr, ki)
    if kind == "graph":
        return e(s["x"])
    if kind == "train":
        blocks, side = e.fwd(s["x"])
        y = e.bwd(blocks, side)
        loss = torch.nn.functional.mse_loss(y, s["target"])
        return loss.detach(), torch.autograd.grad(loss, s["x"])[0]
    if kind == "eq":
        blocks, side = e.fwd(s["x"])
        y = e.bwd([c * g for c, g in zip(blocks, s["gains"])], side)
        loss = torch.nn.functional.mse_loss(y, s["target"])
        return loss.detach(), y.detach(), list(torch.autograd.grad(loss, s["gains"]))
    if kind == "sliced":
        x = s["x"]
        with torch.no_grad():
            blocks, side = e.fwd(x)
            y = e.bwd(blocks, side, length=x.shape[-1])
        return list(blocks), list(side), y
    coefs, pieces = [], []

    def keep(it):
        for blocks, side in it:
            coefs.append(list(blocks) + list(side))
            yield blocks, side
    with torch.no_grad():
        for piece in e.stream_bwd(keep(e.stream_fwd(iter(s["chunks"])))):
            pieces.append(piece)
    return coefs, pieces


# ------------------------------------------------------------ cost and tolerance

def _slices(case):
    if case["kind"] == "sliced":
        return case["batch"] * _num_slices(case["length"])
    if case["kind"] == "stream":
        return case["batch"] * (case["hops"] + 1)
    return case["batch"]


def work(case):
    kind, n = case["kind"], _slices(case)
    bands, groups = _bank(case["layout"])
    ncoef = sum(b * m for b, m, _ in groups)
    lens = [m for b, m, _ in groups for _ in range(b)]
    one = 2.5 * N * math.log2(N) + sum(5 * m * math.log2(m) for m in lens) + 2 * sum(len_ for _, len_, _ in bands)
    coef = 8 * ncoef * n
    if kind in ("fwd", "bwd"):
        return dict(bytes=4 * N * n + coef, flops=one * n)
    if kind in ("rt", "graph"):
        return dict(bytes=8 * N * n + coef, flops=2 * one * n)
    if kind == "train":
        return dict(bytes=12 * N * n, flops=4 * one * n)
    if kind == "eq":
        return dict(bytes=12 * N * n, flops=3 * one * n + 20 * ncoef * n)
    samples = case["batch"] * (case["length"] if kind == "sliced" else case["hops"] * (N // 2))
    return dict(bytes=8 * samples + coef, flops=2 * one * n)


def tolerance(case):
    # fp32 transforms of 2^16 samples: whole outputs are 1e-7 to 7e-7 (2-norm)
    # off their float64 values, a band that holds little of its slice's energy
    # (the rounding of the slice's spectrum reaches every band) up to 1.5e-6
    return {"rel": 6e-6, "max": 5e-5}


# ------------------------------------------------------------ the transform in float64

@functools.lru_cache(maxsize=None)
def _bank(layout):
    """Bands of a layout in coefficient order, [(centre bin, window length,
    block length)], and its groups [(bands, block length, offset)]; the last
    two groups are the DC and the Nyquist band."""
    octs, bins, fs = LAYOUTS[layout]
    centres, lens = [], []
    for j, (n, b) in enumerate(zip(octs, bins)):
        top = fs * 2.0 ** (-1 - sum(octs[j + 1:]))
        below = top < fs / 2.0                       # such a group is laid out over one octave more, dropped again
        top, n_lay = (2.0 * top if below else top) - 1e-6, n + below
        bottom = top / 2.0 ** n_lay
        step = 2.0 ** ((math.log2(top) - math.log2(bottom)) / (n_lay * b - 1))
        f = bottom * step ** np.arange(n_lay * b + 1)
        f[-1] = min(f[-1], fs / 2.0)
        f *= N / fs
        keep = n * b
        centres += list(f[:keep])
        lens += [np.round(f[0] * 2.0 * (step - 1.0) / math.sqrt(step))]
        lens += [np.round(f[k + 1] - f[k - 1]) for k in range(1, keep)]
    count = len(centres)
    half = np.array([0.0] + centres + [N / 2.0])
    pos = np.concatenate((half, N - half[-2:0:-1]))
    pos[count] = (pos[count - 1] + pos[count + 1]) / 2.0          # the last band moves halfway to Nyquist
    pos[count + 2] = N - pos[count]
    pos = np.round(pos).astype(int)
    raw = np.array([np.round(2.0 * centres[0])] + lens + [np.round(N / 2.0 - centres[-2])] + lens[::-1])
    raw = np.maximum(raw, 4).astype(int)
    block = raw.copy()
    groups, start, off = [], 1, 0
    for n, b in zip(octs, bins):
        for _ in range(n):
            m = 1 << int(raw[start:start + b].max() - 1).bit_length()
            block[start:start + b] = m
            block[len(raw) - start - b:len(raw) - start] = m      # the mirrored half, one place low
            groups.append((b, m, off))
            start, off = start + b, off + b * m
    for i in (0, count + 1):
        groups.append((1, int(block[i]), off))
        off += int(block[i])
    diag = np.zeros(N)
    for p, w, m in zip(pos, raw, block):
        j = np.arange(-(w // 2), w - w // 2)
        diag[(p + j) % N] += m * (0.5 + 0.5 * np.cos(2 * np.pi * j / w)) ** 2
    order = list(range(1, count + 1)) + [0, count + 1]
    bands = [(int(pos[i]), int(raw[i]), int(block[i])) for i in order]
    _DIAGONAL[layout] = diag
    return bands, groups


_DIAGONAL = {}


class _Exact:
    """The transform of a layout from its definition, in float64 on a device."""

    def __init__(self, layout, device):
        bands, self.groups = _bank(layout)
        diag = _DIAGONAL[layout]
        bins, win, dual = [], [], []
        for c, w, m in bands:
            j = np.arange(-(w // 2), w - w // 2)
            g = 0.5 + 0.5 * np.cos(2 * np.pi * j / w)
            k, a, d = np.zeros(m, dtype=np.int64), np.zeros(m), np.zeros(m)
            k[j % m], a[j % m], d[j % m] = (c + j) % N, g, m * g / diag[(c + j) % N]
            bins.append(k)
            win.append(a)
            dual.append(np.where(k <= N // 2, d, 0.0))
        t = lambda v: torch.as_tensor(np.concatenate(v), device=device)  # noqa: E731
        self.bins, self.win, self.dual = t(bins), t(win), t(dual)
        self.pos = torch.where(self.bins <= N // 2, self.bins, 0)

    def parts(self, k):
        return [k[..., o:o + b * m].unflatten(-1, (b, m)) for b, m, o in self.groups]

    def analysis(self, x):
        """[..., N] -> [..., ncoef]"""
        taps = torch.fft.fft(x)[..., self.bins] * self.win
        return torch.cat([torch.fft.ifft(p).flatten(-2) for p in self.parts(taps)], -1)

    def synthesis(self, k):
        """[..., ncoef] -> [..., N]"""
        taps = torch.cat([torch.fft.fft(p).flatten(-2) for p in self.parts(k)], -1) * self.dual
        half = torch.zeros(*k.shape[:-1], N // 2 + 1, dtype=k.dtype, device=k.device)
        return torch.fft.irfft(half.index_add(-1, self.pos, taps), n=N)


def _num_slices(length):
    return (-(-length // H) + 1) // 2 + 1


def _tukey(device):
    r = 0.5 - 0.5 * torch.cos(math.pi * torch.arange(H, device=device, dtype=torch.float64) / H)
    w = torch.zeros(N, device=device, dtype=torch.float64)
    w[H - H // 2:H + H // 2] = r
    w[H + H // 2:3 * H - H // 2] = 1
    w[3 * H - H // 2:3 * H + H // 2] = 1 - r
    return w


def _exact_sliced(e, x):
    """Per slice: (coefficient parts [B, S, b, M] with the octave blocks rolled
    back) and the overlap-added inverse [B, S * N / 2] of signals x [B, L]."""
    b, length = x.shape
    s = _num_slices(length)
    pad = torch.zeros(b, (s + 1) * 2 * H, dtype=x.dtype, device=x.device)
    pad[:, 2 * H:2 * H + length] = x
    sl = pad.unfold(-1, N, 2 * H) * _tukey(x.device)
    turn = [H if i % 2 else -H for i in range(s)]
    k = torch.stack([e.analysis(torch.roll(sl[:, i], turn[i], -1)) for i in range(s)], 1)
    out = torch.zeros_like(pad)
    for i in range(s):
        out[:, 2 * H * i:2 * H * i + N] += torch.roll(e.synthesis(k[:, i]), -turn[i], -1)
    parts = e.parts(k)
    for g, p in enumerate(parts[:-2]):
        q = p.shape[-1] // 4
        parts[g] = torch.stack([torch.roll(p[:, i], -q if i % 2 else q, -1) for i in range(s)], 1)
    return parts, out[:, 2 * H:]


def exact(case, seed):
    dev = _device()
    kind, b = case["kind"], case["batch"]
    d = _inputs(case, seed, dev)
    e = _Exact(case["layout"], dev)
    if kind == "bwd":
        return e.synthesis(torch.complex(d["kr"].double(), d["ki"].double()))
    x = d["x"].double()
    if kind in ("fwd", "rt", "graph"):
        ks, ys = [], []
        for rows in x.split(64):                     # in pieces: the double-precision spectra are large
            k = e.analysis(rows)
            ks.append(k)
            if kind != "fwd":
                ys.append(e.synthesis(k))
        k = torch.cat(ks)
        return (k.real, k.imag) + ((torch.cat(ys),) if ys else ())
    if kind in ("train", "eq"):
        target = d["target"].double()
        wrt = [x] if kind == "train" else [g.double() for g in d["gains"]]
        for v in wrt:
            v.requires_grad_(True)
        k = e.analysis(x)
        if kind == "eq":
            p = e.parts(k)
            k = torch.cat([(c * g).flatten(-2) for c, g in zip(p, wrt)] + [c.flatten(-2) for c in p[-2:]], -1)
        y = e.synthesis(k)
        loss = torch.nn.functional.mse_loss(y, target)
        got = torch.autograd.grad(loss, wrt)
        return (loss.detach(), got[0]) if kind == "train" else (loss.detach(), y.detach(), list(got))
    if kind == "sliced":
        length = case["length"]
        parts, out = _exact_sliced(e, x.view(b, length))
        s = _num_slices(length)
        blocks = [p.transpose(1, 2).reshape(b, 1, p.shape[2], s * p.shape[3]) for p in parts[:-2]]
        return blocks, [p.unsqueeze(1) for p in parts[-2:]], out[:, None, :length]
    hops = case["hops"]
    parts, out = _exact_sliced(e, x.view(b, hops * 2 * H))
    coefs = [[p[:, i].unsqueeze(1) for p in parts] for i in range(hops + 1)]
    return coefs, [out[:, None, 2 * H * i:2 * H * (i + 1)] for i in range(hops)]
