"""The chirp-Z of few time steps: one step is the same for every rate to the last
bit, and the edges between the Horner sums (5 steps), a centred block (15) and a
full one (16), alone and behind the 1280 steps one launch takes, agree with the
FP64 oracle.  Normwise bar 2e-6, as in the other parity tests."""
import numpy as np
import pytest

from oracle import synth
from oracle import zdt_oracle as Z

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def F(gpu):
    import fdrt_hip
    return fdrt_hip


@pytest.mark.parametrize("Nf", [6000, 30000, 9375, 1 << 21])
def test_one_step_is_rate_free(F, Nf):
    print(f"short Nf={Nf}", flush=True)
    s = synth.spectrogram(Nf, 1, [(Nf * 0.3, 0.0, 25.0)], seed=1)
    # even lengths: one rate alone; odd ones: also the two of a transform
    out = F.zdtfdr(F.ZDTWorkspace(s, -1.7, 0.3, 6)).cpu().numpy()
    assert np.array_equal(out, out[:, [0, 1] * 3])
    if Nf % 2 == 0:
        assert np.array_equal(out[:, 0], out[:, 1])
    ref = s.astype(np.float64)
    assert np.max(np.abs(out - ref)) <= 2e-6 * np.max(np.abs(ref))


@pytest.mark.parametrize("Nf", [2002, 1 << 21])
@pytest.mark.parametrize("Nt", [3, 4, 5, 6, 7, 9, 14, 15])
def test_edges(F, Nf, Nt):
    s = synth.spectrogram(Nf, Nt, [(Nf * 0.31, 0.5, 25.0)], seed=Nt)
    out = F.zdtfdr(F.ZDTWorkspace(s, -0.9, 0.35, 4)).cpu().numpy()
    ref = Z.fdr64(s, -0.9, 0.35, 4)
    assert np.max(np.abs(out - ref)) <= 2e-6 * np.max(np.abs(ref))


@pytest.mark.parametrize("Nt", [1281, 1285, 1286, 1295, 1296, 1297])
def test_remainder_of_a_long_sum(F, Nt):
    s = synth.spectrogram(250, Nt, [(100.0, 0.01, 5.0)], seed=Nt)
    out = F.zdtfdr(F.ZDTWorkspace(s, -0.02, 0.011, 3)).cpu().numpy()
    ref = Z.fdr64(s, -0.02, 0.011, 3)
    assert np.max(np.abs(out - ref)) <= 2e-6 * np.max(np.abs(ref))
