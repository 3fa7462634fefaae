"""The fused output's chunks of rates (fast_out_run): rate counts on both sides
of one chunk, columns at the ends and on both sides of every chunk boundary
against the FP64 oracle (normwise <= 2e-6), and the statistics, threshold and
hits that ride on the chunked k3 against the FDR itself."""
from fractions import Fraction

import numpy as np
import pytest

from oracle import synth
from oracle import zdt_oracle as Z

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def F(gpu):
    import fdrt_hip
    return fdrt_hip


def spectrogram(Nf, Nt, seed):
    return synth.spectrogram(Nf, Nt, [(Nf * 0.31, 0.6, 25.0), (Nf * 0.77, -0.7, 40.0)], seed=seed)


# 1 MB of spectra per rate at 2^18, 2 at 2^19, 8 at 2^21: one chunk up to 252
# MB, then equal chunks of at most 224 MB rounded up to 8 (4) rates
@pytest.mark.parametrize("Nf,Nr,bounds", [(1 << 18, 252, []), (1 << 18, 253, [128]), (1 << 18, 449, [152, 304]),
                                          (1 << 19, 127, [64]), (1 << 21, 35, [20])])
def test_chunked_columns(F, Nf, Nr, bounds):
    import torch
    Nt, r0, dr = 17, -1.0, 1.0 / 128
    print(f"chunks Nf={Nf} Nr={Nr}", flush=True)
    s = spectrogram(Nf, Nt, Nr)
    ws = F.ZDTWorkspace(s, r0, dr, Nr)
    assert ws.path == "fused-output"
    dest = F.create_fdr(s, Nr)
    dest.fill_(float("nan"))
    F.zdtfdr_(dest, ws)
    assert bool(torch.isfinite(dest).all())
    cols = sorted({0, 1, Nr // 3, Nr - 2, Nr - 1} | {b - 1 for b in bounds} | set(bounds))
    ref = Z.fdr64(s, None, rates=[Fraction(r0) + Fraction(dr) * j for j in cols])
    out = dest[:, cols].cpu().numpy().astype(np.float64)
    assert np.max(np.abs(out - ref)) <= 2e-6 * np.max(np.abs(ref))
    # without a destination every rate's spectra stay for output!
    F.zdtfdr_(ws)
    late = F.create_fdr(s, Nr)
    F.output_(late, ws)
    assert bool((late == dest).all())


def test_chunked_statistics_and_hits(F):
    Nf, Nt, Nr = 1 << 18, 20, 261
    s = spectrogram(Nf, Nt, 3)
    plan = F.RaggedPlan([s], [(-1.0, 1.0 / 128, Nr)], autotune=False)
    plan.bind(8.0, snr=True, cap=1 << 16)
    plan.launch()
    fdr = plan.fdr(0)
    f64 = fdr.double()
    thr = 8.0 * float(f64.std(dim=0).min()) + float(f64[:, 0].mean())
    assert abs(plan.thresholds()[0] - thr) <= 1e-9 * thr
    want = (f64.t().reshape(-1) >= plan.thresholds()[0]).nonzero()[:, 0].cpu().numpy()
    hits = plan.hits(0)
    assert len(want) > 0 and np.array_equal((hits[:, 0] - 1) + Nf * (hits[:, 1] - 1), want)
    plan.close()
