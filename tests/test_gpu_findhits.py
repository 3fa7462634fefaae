"""zdt_findhits (findhits and findprotohits) against fdrstats, zdt_findprotohits
and zdt_clusterprotohits called one after the other, exactly: the maxima of 4096
rows by which tiles are passed over (columns that end inside a tile, tiles across
columns, strided and unaligned matrices, NaN and infinite cells), and the limits of
the one-workgroup clustering and of the buffers."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def F(gpu):
    import fdrt_hip
    return fdrt_hip


def matrices(Nf, Nr, nb, seed, pad=0, skew=0):
    import torch
    rng = np.random.default_rng(seed)
    host, dev = [], []
    for _ in range(nb):
        a = rng.exponential(1.0, size=(Nr, Nf + pad)).astype(np.float32)
        for _ in range(12):
            j, i = int(rng.integers(Nr)), int(rng.integers(Nf))
            a[j, i:i + 3] += 30.0
        a[:, Nf:] = 1e9  # outside the matrix
        flat = torch.empty(Nr * (Nf + pad) + skew, dtype=torch.float32, device="cuda")
        flat[skew:] = torch.from_numpy(a.reshape(-1)).cuda()
        dev.append(torch.as_strided(flat, (Nf, Nr), (1, Nf + pad), skew))
        host.append(a[:, :Nf].T)
    return host, dev


def steps(F, dev, threshold, snr, di=1, dj=1):
    from fdrt_hip import fdrutils as U
    thr = F.fdrdenormalize(threshold, dev) if snr else threshold
    buf, n, Nf, Nr, ld, arr = U._protohits_device(dev, thr, 1 << 20)
    hits = U._cluster_device(buf, n, arr, len(dev), Nf, Nr, ld, di, dj, 1 << 16)
    lin = buf[:n].cpu().numpy()
    return thr, np.stack([lin % Nf + 1, lin // Nf + 1], axis=1), hits


def same(a, b):
    for x, y in zip(a, b):
        assert x.dtype == y.dtype and np.array_equal(x, y)


@pytest.mark.parametrize("Nf,Nr,nb,pad,skew", [
    (4096, 5, 1, 0, 0), (4097, 7, 2, 0, 0), (8192, 3, 1, 5, 0), (16384, 4, 1, 0, 0), (16383, 9, 1, 0, 1),
    (20000, 9, 3, 0, 0), (65536 + 4100, 6, 1, 0, 3), (4095, 8, 1, 0, 0), (100, 300, 1, 0, 0), (1, 40, 1, 0, 0),
    (1 << 18, 17, 1, 0, 0), (1 << 16, 1, 2, 4, 0)])
@pytest.mark.parametrize("snr", [False, True])
def test_as_the_steps(F, Nf, Nr, nb, pad, skew, snr):
    host, dev = matrices(Nf, Nr, nb, Nf + Nr, pad, skew)
    threshold = 7.5 if snr else 14.0
    thr, cells, hits = steps(F, dev, threshold, snr)
    if Nf > 1 or not snr:
        assert np.array_equal(cells, np.argwhere((np.hstack(host) >= thr).T)[:, ::-1] + 1)
    p, h = F.findhits(dev, threshold, snr=snr)
    assert np.array_equal(p, cells)
    same(h, hits)
    assert np.array_equal(F.findprotohits(dev, threshold, snr=snr), cells)


@pytest.mark.parametrize("di,dj", [(0, 0), (3, 1), (1, 4)])
def test_radii(F, di, dj):
    _, dev = matrices(9000, 11, 2, 5)
    _, cells, hits = steps(F, dev, 5.0, True, di, dj)
    p, h = F.findhits(dev, 5.0, snr=True, di=di, dj=dj)
    assert np.array_equal(p, cells)
    same(h, hits)


def test_nan_and_infinite_cells(F):
    import torch
    host, dev = matrices(12288, 6, 1, 9)
    d = dev[0]
    d[100, 1] = float("nan")
    d[5000:9000, 2] = float("nan")
    d[7, 3] = float("inf")
    d[4096:8192, 4] = -float("inf")
    x = d.cpu().numpy()
    for thr in (14.0, float("-inf"), float("inf"), float("nan"), 0.0):
        want = np.argwhere((x >= np.float64(thr)).T)[:, ::-1] + 1
        assert np.array_equal(F.findprotohits(dev, thr), want)
    # the statistics of a matrix with NaN are NaN, and nothing reaches a NaN threshold
    p, h = F.findhits(dev, 5.0, snr=True)
    assert len(p) == 0 and len(h.size) == 0 and h.peak.shape == (0, 2) and h.box.shape == (0, 4)


@pytest.mark.parametrize("n,hits", [(0, 0), (16384, 1), (16385, 1), (2730, 2730), (2731, 2731), (520, 400)])
def test_limits_of_one_workgroup(F, n, hits):
    import torch
    Nf, Nr = 1 << 15, 2
    d = torch.zeros((Nr, Nf), dtype=torch.float32, device="cuda").t()
    if hits == n:
        d[0:3 * n:3, 0] = 5.0
    elif hits == 1:
        d[:n, 1] = 5.0
    else:  # words beyond the first copy
        d[0:3 * hits:3, 0] = 5.0
        d[3 * hits - 3:3 * hits - 3 + n - hits + 1, 0] = 5.0
    _, cells, ref = steps(F, [d], 1.0, False)
    assert len(cells) == n and len(ref.size) == hits
    p, h = F.findhits(d, 1.0)
    assert np.array_equal(p, cells)
    same(h, ref)
    p, h = F.findhits(d, 1.0, capacity=max(n // 2, 1))  # found again with room for all
    assert np.array_equal(p, cells)
    same(h, ref)
    assert np.array_equal(F.findprotohits(d, 1.0, capacity=0), cells)


def test_refusals(F):
    from fdrt_hip import _lib
    _, dev = matrices(5000, 3, 1, 2)
    with pytest.raises(_lib.ZDTError):
        F.findhits(dev, 5.0, di=-1)
    with pytest.raises(_lib.ZDTError):
        F.findhits(dev, 5.0, snr=True, dj=-2)
    with pytest.raises((_lib.ZDTError, RuntimeError)):
        F.findprotohits(dev, 5.0, capacity=-1)
    L = _lib.lib()
    b, w = C.c_int64(), C.c_int64()
    assert L.zdt_findhits_scratch(1, 1 << 16, 1 << 15, 1, C.byref(b), C.byref(w)) == _lib.ZDT_ENOTSUP
    assert L.zdt_findhits_scratch(1, 5000, 3, 1, C.byref(b), C.byref(w)) == _lib.ZDT_OK
    arr = (C.c_void_p * 1)(dev[0].data_ptr())
    n, nh, thr = C.c_int64(), C.c_int64(), C.c_double()
    assert L.zdt_findhits(arr, 1, 5000, 3, 5000, 5.0, 1, 1, 1, None, 0, None, 0, None, C.byref(n), C.byref(nh),
                          C.byref(thr), None) == _lib.ZDT_EINVAL


@pytest.mark.parametrize("tiles,nb", [(1, 1), (17, 2), (2047, 1), (2048, 1), (2049, 1), (1500, 3), (4097, 2), (131072, 1),
                                      (131073, 1)])
def test_scan_of_tile_counts(F, tiles, nb):
    """Proto-hits at the ends of tiles and everywhere in a few, around the chunks of
    the scan and on both sides of the most chunks that the write pass adds up."""
    import torch
    rng = np.random.default_rng(tiles)
    Nf = 4096
    fdrs, want = [], []
    for b in range(nb):
        d = torch.zeros((tiles, Nf), dtype=torch.float32, device="cuda")
        pick = np.unique(np.concatenate([rng.integers(0, tiles, 40), [0, tiles - 1], np.arange(2046, 2050) % tiles]))
        full = pick[:3].repeat(Nf) * Nf + np.tile(np.arange(Nf), len(pick[:3]))
        lin = np.unique(np.concatenate([pick * Nf, pick * Nf + Nf - 1, full]))
        d.view(-1)[torch.from_numpy(lin).cuda()] = 2.0
        fdrs.append(d.t())
        want.append(np.stack([lin % Nf + 1, lin // Nf + 1 + b * tiles], axis=1))
    want = np.concatenate(want)
    assert np.array_equal(F.findprotohits(fdrs, 1.0), want)
    assert np.array_equal(F.findprotohits(fdrs, 1.0, capacity=100), want)
