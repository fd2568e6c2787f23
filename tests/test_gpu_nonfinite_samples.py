"""Samples that are zero, NaN or infinite in the band forms of the coherence and
of the ESD (coherence_band.hpp), against the 16 x 64 tiles, which serve the same
windows on smaller rasters and bands (EstCoh.cu:413-456, EstESD.cu:914-1217): the
same outputs are lost and no others, and no window takes anything from a sample
outside it."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _scene(rng, h, w):
    z = rng.normal(0, 300, (h, w, 2))
    m = np.round(z).astype(np.int16)
    s = (0.9 * z + 0.3 * rng.normal(0, 300, z.shape)).astype(np.float32)
    return m, s


def _spoil(rng, m, s, n, values=(np.nan, np.inf, -np.inf, 1e30, 0.0)):
    """n samples each of those values (zeros in both rasters)."""
    h, w = s.shape[:2]
    for v in values:
        for _ in range(n):
            r, c = rng.integers(0, h), rng.integers(0, w)
            s[r, c, rng.integers(0, 2)] = v
            if v == 0.0:
                s[r, c] = 0.0
                m[r, c] = 0


@pytest.mark.parametrize("wa,wr", [(2, 8), (3, 10), (4, 9), (5, 20), (6, 24), (7, 20), (8, 32)])
def test_coherence_bands_lose_what_the_tiles_lose(tops, dev, wa, wr):
    """480 x 1984 samples take the tiles (30 x 31 of them, fewer than 4 per CU);
    three times as wide they take the bands."""
    N = tops.native
    L = N.load()
    rng = np.random.default_rng(wa * 100 + wr)
    m, s = _scene(rng, 480, 1984)
    _spoil(rng, m, s, 12)
    dx, dy = (wr - 1) // 2, (wa - 1) // 2

    def run(m, s):
        h, w = m.shape[:2]
        dm, ds, out = dev.put(m), dev.put(s), dev.empty(4 * h * w)
        N.check(L.tops_coherence(dm.data_ptr(), ds.data_ptr(), w, h, dx, dy, wr, wa,
                                 out.data_ptr(), N.MODE_FAST, None))
        return dev.get(out, np.float32, (h, w)).copy()

    tile = run(m, s)
    band = run(*(np.ascontiguousarray(np.concatenate([a, a, a], 1)) for a in (m, s)))
    inner = slice(wr, 1984 - wr)   # windows inside the small raster
    band = band[:, 1984:2 * 1984][:, inner]
    tile = tile[:, inner]
    lost = ~np.isfinite(tile)
    assert np.array_equal(np.isnan(band), np.isnan(tile))
    assert np.array_equal(np.isposinf(band), np.isposinf(tile))
    assert np.array_equal(band == 0.0, tile == 0.0) and (tile == 0.0).sum() > 0
    # both round their sums of up to 256 products at 2^-24: 256 * 2^-24 at most
    assert np.abs(band[~lost] - tile[~lost]).max() <= 256 * 2.0 ** -24


@pytest.mark.parametrize("wa,wr", [(3, 10), (5, 20), (8, 32)])
def test_esd_bands_lose_what_the_tiles_lose(tops, dev, wa, wr):
    """12 overlaps of 60 x 8000 samples take the bands (4 x 125 tiles each, over
    10 per CU in all), one overlap at a time the tiles.  The first six overlaps
    hold samples that are not finite, which leave their sums NaN, all of them
    zeros."""
    N = tops.native
    L = N.load()
    rng = np.random.default_rng(wa)
    n, lines, w = 12, 60, 8000
    arrays = []
    for _ in range(2):
        m, s = _scene(rng, n * lines, w)
        _spoil(rng, m, s, 60, (0.0,))
        _spoil(rng, m[:6 * lines], s[:6 * lines], 10)
        arrays += [m, s]
    mf, sf, mb, sb = (dev.put(a) for a in arrays)

    def run(first, count):
        sizes = np.full(count, lines, np.int32)
        shifts, sums = np.zeros(count), np.zeros(2 * count)
        at = lambda t, size: t.data_ptr() + first * lines * w * size
        N.check(L.tops_esd_shifts(at(mf, 4), at(mb, 4), at(sf, 8), at(sb, 8),
                                  sizes.ctypes.data_as(C.POINTER(C.c_int)), count, w, wa, wr, 0.3,
                                  5e3, 2e-3, N.ptr(shifts), N.ptr(sums), None))
        return sums

    bands = run(0, n).reshape(n, 2)
    tiles = np.concatenate([run(i, 1).reshape(1, 2) for i in range(n)])
    print("  bands", bands[:2], "tiles", tiles[:2], flush=True)
    assert np.array_equal(np.isnan(bands), np.isnan(tiles))
    ok = ~np.isnan(tiles)
    assert not ok.all()
    # 480000 unit phasors, each rounded at 2^-22 in either form; none lies near
    # the thresholds of 0.3 and 1 but at the spoilt samples (at most 50 windows'
    # worth of phasors near them, hence the 2)
    assert ok.any() and np.abs(bands[ok] - tiles[ok]).max() <= lines * w * 2.0 ** -22 + 2.0
