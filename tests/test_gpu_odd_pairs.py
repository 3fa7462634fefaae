"""The c2r of odd lengths takes two rates a transform where neither can reach the
other's column: a rate whose spectrum overflows, or a column of Y that is not
finite, leaves its neighbours as they are, as do runs before and after one with
such values.  Odd lengths of one kernel and of two, odd and even rate counts."""
import ctypes as C

import numpy as np
import pytest

from oracle import synth
from oracle import zdt_oracle as Z

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def F(gpu):
    import fdrt_hip
    return fdrt_hip


LENGTHS = [1001, 9375]


def run(F, ws, s):
    d = F.create_fdr(s, ws.Nr)
    d.fill_(7.0)
    return F.zdtfdr_(d, ws, s).cpu().numpy()


# two time steps whose spectra (one bin near Nf/2) cancel at even rates and pass
# the Float32 range at odd ones
@pytest.mark.parametrize("Nf", LENGTHS)
@pytest.mark.parametrize("Nr", [2, 3, 4])
def test_overflowing_rate(F, Nf, Nr):
    print(f"odd pairs Nf={Nf} Nr={Nr}", flush=True)
    n = np.arange(Nf)
    x = 1.9e38 / (Nf / 2) * np.cos(2 * np.pi * ((Nf // 2 * n) % Nf) / Nf)
    s = np.asfortranarray(np.stack([x, -x], axis=1).astype(np.float32))
    out = run(F, F.ZDTWorkspace(s, 0.0, 1.0, Nr), s)
    assert np.isfinite(out[:, 0::2]).all()
    assert not np.isfinite(out[:, 1]).all()


# past the bound from which rates are kept apart, without overflow: the values
# themselves; then the same workspace on ordinary values
@pytest.mark.parametrize("Nf", LENGTHS)
@pytest.mark.parametrize("Nr", [1, 6, 9])
def test_large_values(F, Nf, Nr):
    s = synth.spectrogram(Nf, 21, [(Nf * 0.4, 0.5, 25.0)], seed=Nr)
    ws = F.ZDTWorkspace(s, -0.5, 0.125, Nr)
    good = run(F, ws, s)
    for scale in (1e26, 1e31):
        big = np.asfortranarray(s * np.float32(scale))
        ref = Z.fdr64(big, -0.5, 0.125, Nr)
        assert np.max(np.abs(run(F, ws, big) - ref)) <= 2e-6 * np.max(np.abs(ref))
        for _ in range(3):
            assert np.array_equal(run(F, ws, s), good)


# a captured run, replayed after other runs have moved on to the other flag
@pytest.mark.parametrize("Nf", LENGTHS)
@pytest.mark.parametrize("others", [0, 1, 2])
def test_overflow_in_a_replay(F, Nf, others):
    import torch
    n = np.arange(Nf)
    x = 1.9e38 / (Nf / 2) * np.cos(2 * np.pi * ((Nf // 2 * n) % Nf) / Nf)
    big = np.asfortranarray(np.stack([x, -x], axis=1).astype(np.float32))
    s = synth.spectrogram(Nf, 2, [(Nf * 0.4, 0.5, 25.0)], seed=5)
    ws = F.ZDTWorkspace(s, 0.0, 1.0, 4)
    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    ws.set_stream(st.cuda_stream)

    def run_on(spec):  # on the workspace's stream, which torch's own does not wait for
        d = F.create_fdr(spec, 4)
        torch.cuda.synchronize()
        F.zdtfdr_(d, ws, spec)
        torch.cuda.synchronize()
        return d.cpu().numpy()

    s, big = (torch.from_numpy(np.ascontiguousarray(v.T)).cuda().t() for v in (s, big))
    good = run_on(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        F.zdtfdr_(ws)
    for spec in (big, s, big, s):
        for _ in range(others):
            run_on(s)
        F.input_(ws, spec)
        torch.cuda.synchronize()
        g.replay()
        out = F.create_fdr(s, 4)
        torch.cuda.synchronize()
        F.output_(out, ws)
        torch.cuda.synchronize()
        out = out.cpu().numpy()
        if spec is s:
            assert np.max(np.abs(out - good)) <= 2e-6 * np.max(np.abs(good))
        else:
            assert np.isfinite(out[:, 0::2]).all() and not np.isfinite(out[:, 1]).all()


@pytest.mark.parametrize("Nf", LENGTHS)
def test_bad_column_of_Y(F, Nf):
    import torch

    from fdrt_hip import _device, _lib
    s = synth.spectrogram(Nf, 4, [(Nf * 0.4, 0.5, 25.0)], seed=2)
    ws = F.ZDTWorkspace(s, -0.5, 0.125, 5)
    F.input_(ws, s)
    F.preprocess_(ws)
    F.convolve_(ws)
    F.postprocess_(ws)
    good = F.output_(F.create_fdr(s, 5), ws).cpu().numpy()
    p, rows = C.c_void_p(), C.c_int64()
    _lib.check(_lib.lib().zdt_buffer(ws.handle, _lib.ZDT_BUF_Y, C.byref(p), C.byref(rows), None))
    bad = torch.full((2,), float("nan"))
    dst = C.c_void_p(p.value + 8 * (2 * rows.value + 17))  # bin 17 of column 2
    torch.cuda.synchronize()
    assert _device._hiprt().hipMemcpyAsync(dst, C.c_void_p(bad.data_ptr()), 8, 1, C.c_void_p(0)) == 0
    torch.cuda.synchronize()
    out = F.output_(F.create_fdr(s, 5), ws).cpu().numpy()
    keep = [0, 1, 3, 4]
    assert np.array_equal(out[:, keep], good[:, keep]) and not np.isfinite(out[:, 2]).all()
