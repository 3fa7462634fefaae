"""The most rates a workspace takes (2^24) on a few channels, where the product
of rate groups and parts passes 32 bits: every column is written, and sampled
ones match the definition in FP64.  Normwise bar 2e-6, as in the other parity
tests."""
import numpy as np
import pytest

from oracle import synth

pytestmark = pytest.mark.gpu


def test_every_rate_is_written(gpu):
    import torch

    import fdrt_hip as F
    Nf, Nt, Nr = 16, 4, 1 << 24
    r0, dr = np.float32(-0.5), np.float32(2.0 ** -24)
    print(f"many rates Nf={Nf} Nt={Nt} Nr={Nr}", flush=True)
    s = synth.spectrogram(Nf, Nt, [(5.0, 0.25, 25.0)], seed=8)
    ws = F.ZDTWorkspace(s, r0, dr, Nr)
    dest = F.create_fdr(s, Nr)
    dest.fill_(float("nan"))
    F.zdtfdr_(dest, ws)
    assert not bool(torch.isnan(dest).any())
    j = np.unique(np.concatenate([np.arange(5), [5581481, 5581482, 5592405, 8388607, 8388608, Nr - 1],
                                  np.random.default_rng(1).integers(0, Nr, 2000)]))
    X = np.fft.rfft(s.astype(np.float64), axis=0)
    k, t = np.arange(Nf // 2 + 1)[:, None, None], np.arange(Nt)[None, :, None]
    rates = float(r0) + float(dr) * j
    ref = np.fft.irfft((X[:, :, None] * np.exp(2j * np.pi * k * t * rates / Nf)).sum(axis=1), n=Nf, axis=0)
    out = dest[:, torch.from_numpy(j).to(dest.device)].cpu().numpy().astype(np.float64)
    assert np.max(np.abs(out - ref)) <= 2e-6 * np.max(np.abs(ref))
