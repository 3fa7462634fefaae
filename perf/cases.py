"""The work a user of this framework has it do, as measurable cases.

Each case is one call sequence of a drift-rate search through the public
Python entry points (``fdrt_hip``), on the sizes such searches have: one
coarse channel of 2^16 to 2^22 fine channels, tens to hundreds of time steps,
tens to about a thousand drift rates, plus the small and the awkward
(non-power-of-two, odd) shapes that cut-outs and other instruments give.  A
spectrogram is Exponential(1) noise (detected power) with a few drifting
tones; everything is Float32, the framework's one data type.

kind      one pass
zdt       zdtfdr!(dest, ws, spectrogram): input! and one batch of rates
batches   the same spectrogram against several batches of rates (batchrates)
steps     input!, preprocess!, convolve!, postprocess!, output! one by one
fftfdr    the Fourier-shift FDR for a list of arbitrary rates
detect    an FDR to its statistics, proto-hits and clustered hits
plan      several channels of uneven shapes in one captured plan launch
stream    spectrograms from pinned host memory to proto-hits

Preparation holds what a program keeps between calls: the workspace, plan or
stream, the output matrices and the inputs.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "frequencydriftratetransforms.jl_amd"))

import fdrt_hip as F  # noqa: E402

TONES = 4  # drifting tones per spectrogram


def listed():
    return [
        # a cut-out around one candidate: all latency and launches
        {"name": "zdt_4096x16x33", "kind": "zdt", "Nf": 4096, "Nt": 16, "Nr": 33, "rmax": 2.0, "window": ""},
        # a narrow coarse channel (the repository's small test configuration)
        {"name": "zdt_2p16x16x33", "kind": "zdt", "Nf": 1 << 16, "Nt": 16, "Nr": 33, "rmax": 4.0, "window": ""},
        # the headline configuration: a 2^20-channel coarse channel, rates -4:1/16:4
        {"name": "zdt_2p20x16x129", "kind": "zdt", "Nf": 1 << 20, "Nt": 16, "Nr": 129, "rmax": 4.0, "window": ""},
        # a band that is no power of two, with the Hamming taper
        {"name": "zdt_1e6x16x129", "kind": "zdt", "Nf": 1000000, "Nt": 16, "Nr": 129, "rmax": 4.0,
         "window": "hamming"},
        # an odd number of channels and ragged time and rate counts
        {"name": "zdt_99225x21x77", "kind": "zdt", "Nf": 99225, "Nt": 21, "Nr": 77, "rmax": 2.5, "window": ""},
        # the longest channel of the ragged workload: 60 time steps, rates -4:1/60:4
        {"name": "zdt_2p20x60x481", "kind": "zdt", "Nf": 1 << 20, "Nt": 60, "Nr": 481, "rmax": 4.0, "window": ""},
        # one batch of the long-integration search
        {"name": "zdt_2p22x64x257", "kind": "zdt", "Nf": 1 << 22, "Nt": 64, "Nr": 257, "rmax": 2.0, "window": ""},
        # a time-resolution product: few channels, many time steps, two batches of rates
        {"name": "batches_2p16x279x257", "kind": "batches", "Nf": 1 << 16, "Nt": 279, "Nr": 257, "rmax": 4.0, "nb": 2},
        # arbitrary (not evenly spaced) rates by Fourier shifts
        {"name": "fftfdr_2p18x16x64", "kind": "fftfdr", "Nf": 1 << 18, "Nt": 16, "Nr": 64, "rmax": 4.0},
        # the end of a search: an FDR to hits at SNR 8
        {"name": "detect_2p20x129", "kind": "detect", "Nf": 1 << 20, "Nt": 16, "Nr": 129, "rmax": 4.0, "nb": 1,
         "snr": 8.0},
        # coarse channels of uneven shapes in one launch (the ragged workload's shapes)
        {"name": "plan_6ch", "kind": "plan", "channels": "262144x16,524288x32,262144x60,1048576x16,524288x16,262144x32"},
        # the streamed search, host copies included
        {"name": "stream_2p20x16x257", "kind": "stream", "Nf": 1 << 20, "Nt": 16, "Nr": 257, "rmax": 8.0, "nspec": 2},
    ]


# ---------------------------------------------------------------- ranges


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth(n):
    for p in (2, 3, 5, 7, 11, 13):
        while n % p == 0:
            n //= p
    return n == 1


def _channels(rng, lo, hi):
    """A channel count in [lo, hi]: a power of two, an even smooth number or an odd one."""
    u = rng.random()
    n = _log_int(rng, lo, hi)
    if u < 0.5:
        return 1 << max(int(round(math.log2(n))), int(math.ceil(math.log2(lo))))
    if u < 0.8:
        n += n % 2
        while not _smooth(n):
            n += 2
        return n
    n |= 1
    while not _smooth(n):
        n += 2
    return n


def _cost(Nf, Nt, Nr):
    """Rough relative cost of a batch, for the upper end of draw()."""
    k = 1.0 + Nt / 32.0
    if Nf & (Nf - 1) or Nf < (1 << 16):
        k *= 12.0 if Nf % 2 else 4.0
    return Nf * (Nr + Nt) * k


_MOST = _cost(1 << 22, 64, 257)


def draw(rng):
    while True:
        kind = rng.choices(["zdt", "batches", "steps", "fftfdr", "detect", "plan", "stream"],
                           [50, 12, 4, 8, 12, 8, 6])[0]
        if kind == "plan":
            chans = []
            for _ in range(rng.randint(3, 8)):
                chans.append("%dx%d" % (1 << rng.randint(16, 20), rng.choice([8, 16, 21, 32, 60])))
            if sum(_cost(nf, nt, 8 * nt + 1) for nf, nt in map(_nf_nt, chans)) > _MOST:
                continue
            return {"kind": kind, "channels": ",".join(chans)}
        Nf = _channels(rng, 2000, 1 << 22)
        Nt = _log_int(rng, 5, 300)
        Nr = _log_int(rng, 9, 600)
        rmax = round(rng.uniform(1.0, 8.0), 2)
        case = {"kind": kind, "Nf": Nf, "Nt": Nt, "Nr": Nr, "rmax": rmax}
        cost = _cost(Nf, Nt, Nr)
        if kind == "zdt":
            case["window"] = rng.choice(["", "", "hamming"])
        elif kind == "batches":
            case["nb"] = rng.randint(2, 4)
            cost *= case["nb"]
        elif kind == "steps":
            cost *= 8
        elif kind == "fftfdr":
            cost *= 4
        elif kind == "detect":
            case["Nt"] = rng.randint(8, 32)
            case["nb"] = rng.randint(1, 3)
            case["snr"] = rng.choice([6.0, 8.0, 10.0])
            if Nf * Nr * case["nb"] > 1 << 28:
                continue
        elif kind == "stream":
            case["nspec"] = rng.randint(1, 3)
            cost *= 2 * case["nspec"]
        if cost <= _MOST:
            return case


def _nf_nt(text):
    nf, nt = text.split("x")
    return int(nf), int(nt)


# ---------------------------------------------------------------- inputs


def _spectrogram(gen, Nf, Nt, rmax):
    """(Nf, Nt) column-major on the GPU: noise plus TONES tones of total SNR 15 to 60."""
    s = torch.empty((Nt, Nf), device="cuda").exponential_(1.0, generator=gen)
    u = torch.rand((3, TONES), generator=gen, device="cuda")
    t = torch.arange(Nt, device="cuda")
    chan = torch.round(u[0, :, None] * Nf + (2.0 * u[1, :, None] - 1.0) * rmax * t[None, :]).long() % Nf
    amp = (15.0 + 45.0 * u[2]) / math.sqrt(Nt)
    s.index_put_((t[None, :].expand(TONES, Nt).reshape(-1), chan.reshape(-1)),
                 amp[:, None].expand(TONES, Nt).reshape(-1).contiguous(), accumulate=True)
    return s.t()


def _spec(case, seed, i=0):
    gen = torch.Generator(device="cuda").manual_seed(1000 * seed + i)
    return _spectrogram(gen, case["Nf"], case["Nt"], case["rmax"])


def _rates(case, b=0):
    """(r0, dr) of batch b as Float32 values: nb batches of Nr rates span -rmax .. rmax."""
    n = case["Nr"] * case.get("nb", 1)
    dr = np.float32(2.0 * case["rmax"] / max(n - 1, 1))
    return np.float32(np.float32(-case["rmax"]) + np.float32(b * case["Nr"]) * dr), dr


def _any_rates(case, seed):
    r = np.random.default_rng(seed).uniform(-case["rmax"], case["rmax"], case["Nr"])
    return np.sort(r).astype(np.float32)


def _plan_channels(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    shapes = [_nf_nt(c) for c in case["channels"].split(",")]
    specs = [_spectrogram(gen, nf, nt, 4.0) for nf, nt in shapes]
    return specs, [(-4.0, 1.0 / nt, 8 * nt + 1) for _, nt in shapes]


def _fdr64(spec, rates, window=""):
    """The FDR of a spectrogram by its definition, in 64 bits: (Nf, len(rates)), column-major."""
    Nf, Nt = spec.shape
    X = torch.fft.rfft(spec.t().double(), dim=1)  # (Nt, Nk)
    k = torch.arange(X.shape[1], device=X.device, dtype=torch.float64)
    w = 0.53836 + 0.46164 * torch.cos(2.0 * math.pi * k / Nf) if window == "hamming" else None
    out = torch.empty((len(rates), Nf), device=X.device, dtype=torch.float64)
    z = torch.empty_like(X[0])
    for j, r in enumerate(rates):
        acc = X[Nt - 1].clone()
        ph = torch.remainder(k * (float(r) / Nf), 1.0) * (2.0 * math.pi)
        torch.complex(torch.cos(ph), torch.sin(ph), out=z)
        for t in range(Nt - 2, -1, -1):
            acc.mul_(z).add_(X[t])
        out[j] = torch.fft.irfft(acc if w is None else acc * w, n=Nf)
    return out.t()


def _table(cap, width, dtype=np.int64):
    """A program's table of found hits: cap rows, -1 where there is none, and the rows in use."""
    return {"rows": np.full((cap, width) if width else cap, -1, dtype), "used": 0}


def _record(tables, found):
    """Puts each list found in its table; rows of the pass before that are no longer in use are cleared."""
    out = []
    for t, x in zip(tables, found):
        n = min(len(x), len(t["rows"]))
        t["rows"][:n] = x[:n]
        t["rows"][n:t["used"]] = -1
        t["used"] = n
        out.append((t["rows"], len(x)))
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "plan":
        specs, rates = _plan_channels(case, seed)
        plan = F.RaggedPlan(specs, rates, autotune=False)
        plan.bind(10.0, snr=True, cap=1 << 14)
        return {"kind": kind, "plan": plan, "tables": [_table(1 << 14, 2) for _ in range(plan.nch)]}
    Nf, Nt, Nr = case["Nf"], case["Nt"], case["Nr"]
    if kind == "stream":
        specs = []
        for i in range(case["nspec"]):
            p = F.pinned_spectrogram(Nf, Nt)
            p.t().copy_(_spec(case, seed, i).t())
            specs.append(p)
        r0, dr = _rates(case)
        return {"kind": kind, "specs": specs, "search": F.StreamSearch(Nf, Nt, (r0, dr, Nr)),
                "tables": [_table(1 << 16, 2) for _ in specs]}
    if kind == "detect":
        # an FDR by its definition, rounded to Float32
        spec = _spec(case, seed)
        fdrs = []
        for b in range(case["nb"]):
            r0, dr = _rates(case, b)
            fdrs.append(_fdr64(spec, float(r0) + float(dr) * np.arange(Nr)).float())
        return {"kind": kind, "fdrs": fdrs[0] if len(fdrs) == 1 else fdrs, "snr": case["snr"],
                "tables": [_table(1 << 16, 2), _table(1 << 15, 2), _table(1 << 15, 0, np.float32), _table(1 << 15, 0),
                           _table(1 << 15, 4), _table(1 << 16, 0)]}
    spec = _spec(case, seed)
    if kind == "fftfdr":
        return {"kind": kind, "spec": spec, "ws": F.fftfdr_workspace(spec), "rates": _any_rates(case, seed),
                "dest": F.create_fdr(spec, Nr)}
    r0, dr = _rates(case)
    st = {"kind": kind, "spec": spec, "ws": F.ZDTWorkspace(spec, r0, dr, Nr)}
    if kind == "batches":
        st["dests"] = [F.create_fdr(spec, Nr) for _ in range(case["nb"])]
        st["r0s"] = [_rates(case, b)[0] for b in range(case["nb"])]
    else:
        st["dest"] = F.create_fdr(spec, Nr)
        st["window"] = case.get("window", "")
    return st


def run(st):
    kind = st["kind"]
    if kind == "zdt":
        if st["window"]:
            return F.zdtfdr_(st["window"], st["dest"], st["ws"], st["spec"])
        return F.zdtfdr_(st["dest"], st["ws"], st["spec"])
    if kind == "batches":
        return F.zdtfdr_(st["dests"], st["ws"], st["spec"], r0=st["r0s"])
    if kind == "steps":
        F.input_(st["ws"], st["spec"])
        F.preprocess_(st["ws"])
        F.convolve_(st["ws"])
        F.postprocess_(st["ws"])
        return F.output_(st["dest"], st["ws"])
    if kind == "fftfdr":
        F.fftfdr_workspace_(st["ws"], st["spec"])
        return F.fftfdr_(st["dest"], st["ws"], st["rates"])
    if kind == "detect":
        protohits, hits = F.findhits(st["fdrs"], st["snr"], snr=True)
        return _record(st["tables"], [protohits, *hits])
    if kind == "plan":
        plan = st["plan"]
        plan.launch()
        return plan.dests, _record(st["tables"], [plan.hits(c) for c in range(plan.nch)])
    hits, thr = st["search"].search(st["specs"], snr=10.0)
    # the threshold is a statistic of Float32 cells
    return _record(st["tables"], hits), thr.astype(np.float32)


# ---------------------------------------------------------------- yardsticks


def _batch_flops(Nf, Nt, Nr):
    """Real transforms of the Nt inputs and Nr outputs, and per bin the cheaper
    of the direct sum and the fast convolution of length Nt+Nr-1."""
    Nk, Nl = Nf // 2 + 1, Nt + Nr - 1
    czt = min(8.0 * Nt * Nr, 10.0 * Nl * math.log2(max(Nl, 2)) + 6.0 * (Nl + Nt + Nr))
    return 2.5 * Nf * math.log2(Nf) * (Nt + Nr) + Nk * czt


def work(case):
    kind = case["kind"]
    if kind == "plan":
        shapes = [_nf_nt(c) for c in case["channels"].split(",")]
        return {"bytes": sum(4.0 * nf * (nt + 8 * nt + 1) for nf, nt in shapes),
                "flops": sum(_batch_flops(nf, nt, 8 * nt + 1) for nf, nt in shapes)}
    Nf, Nt, Nr = case["Nf"], case["Nt"], case["Nr"]
    if kind == "detect":
        # the cells read once; their sums and one comparison each
        cells = float(Nf) * Nr * case["nb"]
        return {"bytes": 4.0 * cells, "flops": 4.0 * cells}
    if kind == "stream":
        # the spectrograms read once; the FDR need not leave the device's caches
        return {"bytes": 4.0 * Nf * Nt * case["nspec"], "flops": case["nspec"] * _batch_flops(Nf, Nt, Nr)}
    nb = case.get("nb", 1)
    return {"bytes": 4.0 * Nf * (Nt + nb * Nr), "flops": _batch_flops(Nf, Nt, nb * Nr)}


def exact(case, seed):
    """What run() returns, in 64 bits; None in the places of hits (whole numbers)."""
    kind = case["kind"]
    if kind in ("detect", "stream"):
        return None
    if kind == "plan":
        specs, rates = _plan_channels(case, seed)
        fdrs = []
        for s, (r0, dr, Nr) in zip(specs, rates):
            fdrs.append(_fdr64(s, float(np.float32(r0)) + float(np.float32(dr)) * np.arange(Nr)))
        return fdrs, [(None, None)] * len(specs)
    spec = _spec(case, seed)
    if kind == "fftfdr":
        return _fdr64(spec, [float(r) for r in _any_rates(case, seed)])
    out = []
    for b in range(case.get("nb", 1)):
        r0, dr = _rates(case, b)
        # the workspace keeps batch 0's dr, and each batch its own Float32 r0
        out.append(_fdr64(spec, float(r0) + float(dr) * np.arange(case["Nr"]), case.get("window", "")))
    return out if kind == "batches" else out[0]
