"""The column-pair kernels with their rate or time groups split over several
blocks (group_parts): rate counts around the edges of the groups and parts,
where a part's first or last group could be lost, doubled or started at the
wrong phase.  Same bar as the other parity tests: normwise <= 2e-6 of the
FP64 oracle."""
import sys

import numpy as np
import pytest

from oracle import synth
from oracle import zdt_oracle as Z

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def F(gpu):
    import fdrt_hip
    return fdrt_hip


def check(F, Nf, Nt, Nr, r0, dr, path):
    print(f"split Nf={Nf} Nt={Nt} Nr={Nr}", flush=True)
    sys.stdout.flush()
    s = synth.spectrogram(Nf, Nt, [(Nf * 0.31, 1.5, 25.0), (Nf * 0.77, -1.75, 40.0)], seed=Nt + Nr)
    ws = F.ZDTWorkspace(s, r0, dr, Nr)
    assert ws.path == path
    dest = F.create_fdr(s, Nr)
    dest.fill_(float("nan"))
    out = F.zdtfdr_(dest, ws).cpu().numpy().astype(np.float64)
    ref = Z.fdr64(s, r0, dr, Nr)
    assert np.max(np.abs(out - ref)) <= 2e-6 * np.max(np.abs(ref))


# paired rates (Nt > 8; groups of two pairs, from one group a part on) and single
# rates (groups of four), N1 = 64 and 128
@pytest.mark.parametrize("Nf,Nt,Nr", [(1 << 16, 16, n) for n in (1, 2, 11, 12, 13, 23, 24, 25, 47, 131)]
                         + [(1 << 16, 5, n) for n in (1, 4, 11, 12, 13, 24, 25, 131)]
                         + [(1 << 17, 12, 26), (1 << 17, 2, 49), (1 << 18, 16, 38), (1 << 18, 3, 27)])
def test_split_fused(F, Nf, Nt, Nr):
    check(F, Nf, Nt, Nr, -2.25, 0.0625, "fused")


# the fused output: time groups of the input and rate groups of the c2r
@pytest.mark.parametrize("Nf,Nt,Nr", [(1 << 16, 17, 1), (1 << 16, 33, 7), (1 << 16, 65, 8), (1 << 16, 279, 9),
                                      (1 << 16, 21, 131), (1 << 17, 18, 17), (1 << 18, 37, 19), (1 << 19, 25, 21)])
def test_split_fused_output(F, Nf, Nt, Nr):
    check(F, Nf, Nt, Nr, -1.0, 0.03125, "fused-output")
