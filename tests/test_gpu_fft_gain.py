"""The gain of the generic transforms (r2c and c2r together) on a tone: the constants
of the radices, rounded to 32 bits and the same in every pass, must not add up.
One time step at one rate returns its input, so the value at a channel of
power 1 is the gain there.  Its mean over 64 channels is held to 7e-8: the output
scale's rounding (3e-8), the passes' tables (2e-8) and three deviations of the mean
(2e-8)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nf", [2000, 2187, 4096, 9375, 10000, 59049, 78125, 250000, 300000, 500000, 1000000])
def test_gain_of_a_tone(gpu, Nf):
    import fdrt_hip as F
    print(f"gain Nf={Nf}", flush=True)
    rng = np.random.default_rng(Nf)
    ws, gains = None, []
    for n in rng.integers(0, Nf, 64):
        s = np.zeros((Nf, 1), np.float32)
        s[n] = 1.0
        if ws is None:
            ws = F.ZDTWorkspace(s, 0.0, 1.0, 1, generic=True)
        out = F.zdtfdr_(F.create_fdr(s, 1), ws, s)
        gains.append(float(out[int(n), 0].double()) - 1.0)
    assert abs(np.mean(gains)) <= 7e-8


@pytest.mark.parametrize("Nf", [2000, 9375, 500000, 1000000])
def test_gain_of_the_mean(gpu, Nf):
    """A constant (bin 0 alone) meets no rounded constant: each element comes back
    within the scale's and the sums' rounding, 2^-22."""
    import fdrt_hip as F
    s = np.ones((Nf, 1), np.float32)
    out = F.zdtfdr(F.ZDTWorkspace(s, 0.0, 1.0, 1)).cpu().numpy()
    assert np.max(np.abs(out - 1.0)) <= 2.0 ** -22
