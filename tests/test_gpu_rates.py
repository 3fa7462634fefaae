"""fftfdr over arbitrary rates through the fused output's kernels (power-of-two
lengths from 2^16 on) and the generic ones, against the FP64 oracle: every
register block of the sum (Nt at its edges), more rates than one launch or one
piece of kept spectra takes, a repeated call with more and with fewer rates, and
the other uses of the workspace's input beside it.  Normwise bar 2e-6, as in the
other tests of fftfdr."""
import numpy as np
import pytest

from oracle import synth
from oracle import zdt_oracle as Z

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def F(gpu):
    import fdrt_hip
    return fdrt_hip


def rates_of(n, seed=0):
    r = np.random.default_rng(seed).uniform(-6.0, 6.0, n).astype(np.float32)
    r[: min(n, 3)] = [0.0, -2.5, 1.0][: min(n, 3)]
    return r


def close(out, s, rates):
    ref = Z.fftfdr64(s, rates)
    assert np.max(np.abs(out.cpu().numpy().astype(np.float64) - ref)) <= 2e-6 * np.max(np.abs(ref))


@pytest.mark.parametrize("Nf,Nt,Nr", [
    (1 << 16, 1, 1), (1 << 16, 4, 5), (1 << 16, 5, 129), (1 << 16, 16, 300), (1 << 16, 17, 8), (1 << 16, 32, 9),
    (1 << 16, 64, 17), (1 << 16, 65, 3), (1 << 17, 16, 31), (1 << 18, 20, 2), (1 << 19, 3, 7), (1 << 20, 16, 61),
    (1 << 21, 2, 3), (1 << 22, 2, 17), (1 << 16, 1030, 2), (30000, 16, 131), (9375, 33, 7), (250, 64, 257), (1 << 15, 17, 3)])
def test_rates(F, Nf, Nt, Nr):
    print(f"rates Nf={Nf} Nt={Nt} Nr={Nr}", flush=True)
    s = synth.spectrogram(Nf, Nt, [(Nf * 0.4, 1.0, 25.0), (Nf * 0.8, -2.5, 30.0)], seed=Nf % 1000 + Nt)
    r = rates_of(Nr)
    d = F.create_fdr(s, Nr)
    d.fill_(float("nan"))
    close(F.fftfdr_(d, F.fftfdr_workspace(s), r), s, r)


@pytest.mark.parametrize("Nf", [1 << 16, 6000])
def test_repeated_calls(F, Nf):
    s = synth.spectrogram(Nf, 12, [(Nf * 0.4, 1.0, 25.0)], seed=3)
    s2 = synth.spectrogram(Nf, 12, [(Nf * 0.6, -1.0, 25.0)], seed=4)
    ws = F.fftfdr_workspace(s)
    for n in (3, 40, 7):
        close(F.fftfdr(ws, rates_of(n, n)), s, rates_of(n, n))
    ref = np.fft.rfft(s.astype(np.float64), axis=0)
    Fd = ws.dest_rfft.cpu().numpy()
    assert Fd.shape == ref.shape and np.max(np.abs(Fd - ref)) <= 2e-6 * np.max(np.abs(ref))
    sh = F.fdshift(ws, 1.0).cpu().numpy()
    ref = Z.fdshift64(s, 1.0)
    assert np.max(np.abs(sh - ref)) <= 2e-6 * np.max(np.abs(ref))
    ws = F.fftfdr_workspace_(ws, s2)
    close(F.fftfdr(ws, rates_of(9)), s2, rates_of(9))
    sh = F.fdshift(ws, -1.0).cpu().numpy()
    ref = Z.fdshift64(s2, -1.0)
    assert np.max(np.abs(sh - ref)) <= 2e-6 * np.max(np.abs(ref))
    with pytest.raises(RuntimeError):
        F.fftfdr(ws, [1.0, float("inf")])
