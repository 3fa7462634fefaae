"""The LDS transforms of the generic path (fft_generic.hip): lengths on both
sides of the one-kernel limit, every radix, odd lengths with one, two and an odd
number of columns packed in pairs, radix caps, and both directions (the input
spectrum F against numpy's FP64 rfft, the FDR against the FP64 oracle).
Normwise bars as the other parity tests: 2e-6."""
import numpy as np
import pytest

from oracle import synth
from oracle import zdt_oracle as Z

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def F(gpu):
    import fdrt_hip
    return fdrt_hip


def check(F, Nf, Nt, Nr, **kw):
    print(f"lds fft Nf={Nf} Nt={Nt} Nr={Nr} {kw}", flush=True)
    s = synth.spectrogram(Nf, Nt, [(Nf * 0.31, 0.5, 25.0), (Nf * 0.77, -0.75, 40.0)], seed=Nf % 1000 + Nr)
    ws = F.ZDTWorkspace(s, -0.5, 0.25, Nr, generic=True, **kw)
    Fd = ws.F.cpu().numpy().astype(np.complex128)
    ref = np.fft.rfft(s.astype(np.float64), axis=0)
    assert np.max(np.abs(Fd - ref)) <= 2e-6 * np.max(np.abs(ref))
    dest = F.create_fdr(s, Nr)
    dest.fill_(float("nan"))
    out = F.zdtfdr_(dest, ws).cpu().numpy().astype(np.float64)
    ref = Z.fdr64(s, -0.5, 0.25, Nr)
    assert np.max(np.abs(out - ref)) <= 2e-6 * np.max(np.abs(ref))


# even: half lengths 2..16 and products of single radices, 4096 and just past it,
# the four-step split at its smallest and largest
@pytest.mark.parametrize("Nf", [4, 6, 8, 10, 12, 14, 16, 18, 20, 22, 24, 26, 28, 30, 32, 338, 242, 2 * 13 * 11 * 7, 2 * 3375,
                                2 * 2744, 2 * 4095, 8192, 2 * 4116, 8400, 50000, 2 * 59049, 2 * 1000000 // 2, 1 << 21])
def test_even_lengths(F, Nf):
    check(F, Nf, 3, 5)


@pytest.mark.parametrize("Nf", [3, 5, 7, 9, 11, 13, 15, 105, 1001, 3375, 4095, 4125, 15625, 99225, 823543, 1003275])
@pytest.mark.parametrize("Nr", [1, 2, 5])
def test_odd_lengths(F, Nf, Nr):
    check(F, Nf, 2, Nr)


# many short transforms per block, with a remainder
@pytest.mark.parametrize("Nf,Nt,Nr", [(64, 37, 1031), (250, 5, 4099), (63, 9, 2051)])
def test_many_transforms(F, Nf, Nt, Nr):
    s = synth.spectrogram(Nf, Nt, [(Nf * 0.4, 0.1, 10.0)], seed=1)
    out = F.zdtfdr(F.ZDTWorkspace(s, -1.0, 1.0 / 1024, Nr, generic=True)).cpu().numpy()
    ref = Z.fdr64(s, -1.0, 1.0 / 1024, Nr)
    assert np.max(np.abs(out - ref)) <= 2e-6 * np.max(np.abs(ref))


# the blocks of fs_cols: 125 x 16 and 147 x 16 elements in few and in many blocks, 243 x 16,
# 315 x 16, 576 x 8, each with a partial last block of columns and rows
@pytest.mark.parametrize("Nf,Nt,Nr", [(15625, 3, 7), (15625, 3, 141), (21609, 2, 151), (2 * 15625, 70, 2), (59049, 2, 9),
                                      (99225, 2, 3), (2 * 589824, 2, 3)])
def test_blocks_of_columns(F, Nf, Nt, Nr):
    s = synth.spectrogram(Nf, Nt, [(Nf * 0.4, 0.1, 10.0)], seed=2)
    out = F.zdtfdr(F.ZDTWorkspace(s, -1.0, 1.0 / 64, Nr, generic=True)).cpu().numpy()
    ref = Z.fdr64(s, -1.0, 1.0 / 64, Nr)
    assert np.max(np.abs(out - ref)) <= 2e-6 * np.max(np.abs(ref))


@pytest.mark.parametrize("Nf", [4096, 30000, 99225])
def test_radix_cap(F, Nf):
    check(F, Nf, 2, 3, radix_cap=8)


def test_one_bad_time_step_stays_alone(F):
    """fdshift of an odd-length spectrogram: a time step that is not finite
    leaves the other time steps' columns untouched."""
    s = synth.spectrogram(1001, 6, [(300.0, 0.5, 20.0)], seed=4)
    good = F.fdshift(F.fftfdr_workspace(s), 0.75).cpu().numpy()
    bad = s.copy()
    bad[17, 2] = np.inf
    got = F.fdshift(F.fftfdr_workspace(bad), 0.75).cpu().numpy()
    keep = [t for t in range(6) if t != 2]
    assert np.array_equal(got[:, keep], good[:, keep]) and not np.isfinite(got[:, 2]).all()
