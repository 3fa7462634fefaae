"""The folded chirp-Z (czt_fold.h) at the edges of its 16-step blocks, of the
blocks a lane holds and of the lanes that share a bin, for even, odd and single
rate counts, on the fused output and on the generic kernels, against the FP64
oracle (normwise <= 2e-6, as the other parity tests)."""
import numpy as np
import pytest

from oracle import synth
from oracle import zdt_oracle as Z

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def F(gpu):
    import fdrt_hip
    return fdrt_hip


def check(F, Nf, Nt, Nr, r0, dr, path, **kw):
    print(f"fold Nf={Nf} Nt={Nt} Nr={Nr} r0={r0} dr={dr} {kw}", flush=True)
    s = synth.spectrogram(Nf, Nt, [(Nf * 0.31, 1.5, 25.0), (Nf * 0.77, -1.75, 40.0)], seed=Nt + Nr)
    ws = F.ZDTWorkspace(s, r0, dr, Nr, **kw)
    assert ws.path == path
    dest = F.create_fdr(s, Nr)
    dest.fill_(float("nan"))
    out = F.zdtfdr_(dest, ws).cpu().numpy().astype(np.float64)
    ref = Z.fdr64(s, r0, dr, Nr)
    assert np.max(np.abs(out - ref)) <= 2e-6 * np.max(np.abs(ref))


# one lane: 2..5 blocks; two, four, eight and sixteen lanes
@pytest.mark.parametrize("Nt,Nr", [(17, 1), (32, 2), (33, 3), (48, 5), (49, 8), (64, 9), (65, 4), (80, 7), (81, 3), (96, 2),
                                   (128, 6), (160, 5), (161, 3), (256, 4), (320, 7), (321, 2), (640, 3), (641, 5),
                                   (1023, 2), (1024, 3)])
def test_fold_fused_output(F, Nt, Nr):
    check(F, 1 << 16, Nt, Nr, -0.75, 0.375, "fused-output")


# rates not symmetric about 0 and a step that is not dyadic: the coefficients'
# pre-rotation; the rate pairs split over blocks
@pytest.mark.parametrize("Nt,Nr,r0,dr", [(21, 75, -2.0, 0.05), (60, 131, 0.5, 0.01), (100, 97, 1.0, -0.03)])
def test_fold_rates(F, Nt, Nr, r0, dr):
    check(F, 1 << 16, Nt, Nr, r0, dr, "fused-output")


# Nf > 2^20 takes the fused output at Nt <= 16 too (one block)
@pytest.mark.parametrize("Nt", [1, 2, 15, 16])
def test_fold_one_block(F, Nt):
    check(F, 1 << 21, Nt, 3, -1.25, 1.0, "fused-output")


# the generic kernels, more steps than the lanes of a bin hold at once included
@pytest.mark.parametrize("Nf,Nt,Nr", [(2187, 1, 3), (2000, 2, 1), (2002, 5, 4), (4096, 16, 33), (6000, 17, 9),
                                      (3125, 80, 6), (1001, 81, 35), (1024, 333, 8), (512, 700, 5), (250, 1280, 3),
                                      (250, 1281, 4), (64, 3000, 5)])
def test_fold_generic(F, Nf, Nt, Nr):
    check(F, Nf, Nt, Nr, -0.4, 0.25, "generic")
