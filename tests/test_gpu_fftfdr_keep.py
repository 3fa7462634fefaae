"""The spectra that fftfdr and fdshift keep with the workspace: captured graphs of the
workspace outlive later calls with more rates, and calls on another stream do not
share them.  Power-of-two lengths (the fused output's kernels) and others (the
generic ones)."""
import numpy as np
import pytest

from oracle import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def F(gpu):
    import fdrt_hip
    return fdrt_hip


def spec(Nf, Nt, seed):
    return synth.spectrogram(Nf, Nt, [(Nf * 0.4, 1.0, 25.0)], seed=seed)


def rates_of(n, seed):
    return np.random.default_rng(seed).uniform(-4.0, 4.0, n).astype(np.float32)


def replays(g, dest, want, between):
    import torch
    for _ in range(4):
        dest.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(dest, want)
        between()
        torch.cuda.synchronize()


def capture(ws, st, call):
    import torch
    ws.set_stream(st.cuda_stream)
    call()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        call()
    torch.cuda.synchronize()
    return g


# a graph of zdtfdr! and fftfdr! calls with more rates than its scratch holds
@pytest.mark.parametrize("Nf", [6000, 9375, 1 << 16])
def test_graph_of_zdtfdr(F, Nf):
    import torch
    print(f"keep zdtfdr Nf={Nf}", flush=True)
    s = spec(Nf, 12, 1)
    ws = F.ZDTWorkspace(s, -1.0, 0.25, 9, generic=Nf == 1 << 16)
    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    dest = F.create_fdr(s, 9)
    g = capture(ws, st, lambda: F.zdtfdr_(dest, ws))
    want = dest.clone()
    more = iter((20, 70, 300, 5))

    def between():
        n = next(more)
        F.fftfdr_(F.create_fdr(s, n), ws_of(ws), rates_of(n, n))

    replays(g, dest, want, between)


def ws_of(ws):
    """fftfdr! on a plain workspace."""
    from types import SimpleNamespace
    return SimpleNamespace(ws=ws, Nf=ws.Nf, Nt=ws.Nt)


# a graph of fftfdr! and later calls with more rates
@pytest.mark.parametrize("Nf", [6000, 9375, 1 << 16, 1 << 18])
def test_graph_of_fftfdr(F, Nf):
    import torch
    print(f"keep fftfdr Nf={Nf}", flush=True)
    s = spec(Nf, 12, 2)
    ws = F.fftfdr_workspace(s)
    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    r = rates_of(6, 0)
    dest = F.create_fdr(s, 6)
    g = capture(ws.ws, st, lambda: F.fftfdr_(dest, ws, r))
    want = dest.clone()
    size0 = ws.ws.nbytes
    more = iter((20, 70, 300, 5))

    def between():
        n = next(more)
        F.fftfdr_(F.create_fdr(s, n), ws, rates_of(n, n))
        F.fdshift(ws, 0.5)

    replays(g, dest, want, between)
    assert ws.ws.nbytes - size0 <= 2 * (480 << 20)


@pytest.mark.parametrize("Nf", [30000, 1 << 18])
def test_two_streams(F, Nf):
    import torch
    print(f"keep streams Nf={Nf}", flush=True)
    s = spec(Nf, 16, 3)
    ws = F.fftfdr_workspace(s)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(3)]
    rates = [rates_of(40, i) for i in range(3)]
    want = []
    for r in rates:
        want.append(F.fftfdr(ws, r))
        torch.cuda.synchronize()
    dest = [F.create_fdr(s, 40) for _ in range(3)]
    torch.cuda.synchronize()
    for _ in range(8):
        for st, r, d in zip(streams, rates, dest):
            ws.ws.set_stream(st.cuda_stream)
            F.fftfdr_(d, ws, r)
    torch.cuda.synchronize()
    for d, w in zip(dest, want):
        assert torch.equal(d, w)


# fdshift! between fftfdr! calls, in the same buffer
@pytest.mark.parametrize("Nf", [6000, 9375, 1 << 16])
def test_fdshift_beside_fftfdr(F, Nf):
    import torch
    s = spec(Nf, 12, 4)
    ws, ws2 = F.fftfdr_workspace(s), F.fftfdr_workspace(s)
    want = F.fdshift(ws2, 1.25)
    for n in (3, 90, 5):
        fdr = F.fftfdr(ws, rates_of(n, n))
        sh = F.fdshift(ws, 1.25)
        assert torch.equal(sh, want)
        assert torch.equal(fdr, F.fftfdr(F.fftfdr_workspace(s), rates_of(n, n)))
