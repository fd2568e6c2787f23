"""The band form of the coherence against the oracle's FP64 window sums
(EstCoh.cu:101-139, 413-456 semantics), at the edges of its ranges: the lowest,
tallest, narrowest and widest windows, every remainder of the window width by
4, off-centre windows, rasters that end inside a thread's 4 columns or a
band's last one, odd widths (unaligned rows), and samples below the amplitude
threshold.  A window sum takes at most 8 + 64 / 4 + 6 roundings in a row, each
2^-24 of its sum of magnitudes; the coherence of three such sums is within
3 * 30 * 2^-24 = 5.4e-6, and 1e-5 with the square roots."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _inputs(h, w, seed):
    rng = np.random.default_rng(seed)
    M = rng.integers(-800, 800, (h, w, 2), dtype=np.int16)
    S = (M[..., 0] + 1j * M[..., 1]) * np.exp(0.3j) + rng.normal(0, 300, (h, w)) \
        + 1j * rng.normal(0, 300, (h, w))
    S = S.astype(np.complex64)
    S[rng.random((h, w)) < 0.02] = 0      # masked outputs
    S[h // 2, :] *= 1e-6
    return M, S


# (window lines, samples), (lines before, samples before), (lines, samples); the
# rasters have more tiles of 16 x 64 than run at once, so they take the bands
# (3 x 10 on 700 x 1019 has 704, which still run at once: the tiles)
@pytest.mark.parametrize("win,off,shape", [
    ((2, 4), (0, 1), (1301, 1000)),
    ((2, 8), (1, 7), (33, 25001)),
    ((3, 10), (1, 4), (700, 1019)),
    ((3, 10), (2, 9), (65, 16001)),
    ((4, 9), (1, 4), (48, 25002)),
    ((4, 16), (0, 0), (640, 2023)),
    ((5, 7), (2, 3), (531, 2011)),
    ((5, 20), (4, 19), (18, 50003)),
    ((6, 24), (2, 11), (700, 3001)),
    ((6, 25), (5, 0), (37, 64000)),
    ((7, 31), (3, 15), (801, 2817)),
    ((8, 32), (3, 15), (1000, 2305)),
    ((8, 64), (7, 63), (20, 99999)),
])
def test_band_windows(tops, orc, dev, win, off, shape):
    N = tops.native
    L = N.load()
    (wa, wr), (dy, dx), (h, w) = win, off, shape
    M, S = _inputs(h, w, wa * 100 + wr)
    ref = orc.coherence(M, S.astype(np.complex128), dx, dy, wr, wa)
    dm, ds, dc = dev.put(M), dev.put(S), dev.empty(h * w * 4)
    N.check(L.tops_coherence(dm.data_ptr(), ds.data_ptr(), w, h, dx, dy, wr, wa, dc.data_ptr(),
                             0, None))
    got = dev.get(dc, np.float32, (h, w))
    zero = np.abs(S) < 0.0009
    assert not got[zero].any()
    e = float(np.max(np.abs(got - ref)))
    print(f"  {wa} x {wr} from ({dy}, {dx}) on {h} x {w}: {e:.2e}", flush=True)
    assert e <= TOL


@pytest.mark.parametrize("wa,wr", [(3, 10), (6, 24)])
def test_band_split_independent(tops, dev, wa, wr):
    """A raster's coherence does not depend on its split into bands and row
    blocks: the lower part of a raster, taken alone, has the same bits away
    from its first lines."""
    N = tops.native
    L = N.load()
    h, w, cut = 1500, 2301, 333
    M, S = _inputs(h, w, 7)
    dx, dy = (wr - 1) // 2, (wa - 1) // 2

    def run(m, s, n):
        dm, ds, dc = dev.put(np.ascontiguousarray(m)), dev.put(np.ascontiguousarray(s)), \
            dev.empty(n * w * 4)
        N.check(L.tops_coherence(dm.data_ptr(), ds.data_ptr(), w, n, dx, dy, wr, wa,
                                 dc.data_ptr(), 0, None))
        return dev.get(dc, np.float32, (n, w))

    whole, part = run(M, S, h), run(M[cut:], S[cut:], h - cut)
    assert np.array_equal(whole[cut + wa:], part[wa:])


@pytest.mark.parametrize("shape", [(1100, 1019), (33, 25001), (1487, 769)])
def test_default_window_in_bands(tops, orc, dev, shape):
    """The 3 x 10 window at its default centre on rasters of more than 4 tiles of
    16 x 64 per CU."""
    N = tops.native
    L = N.load()
    h, w = shape
    assert -(-h // 16) * -(-w // 64) > 4 * dev.torch.cuda.get_device_properties(
        0).multi_processor_count
    M, S = _inputs(h, w, h)
    ref = orc.coherence(M, S.astype(np.complex128), 4, 1, 10, 3)
    dm, ds, dc = dev.put(M), dev.put(S), dev.empty(h * w * 4)
    N.check(L.tops_coherence(dm.data_ptr(), ds.data_ptr(), w, h, 4, 1, 10, 3, dc.data_ptr(), 0,
                             None))
    got = dev.get(dc, np.float32, (h, w))
    assert not got[np.abs(S) < 0.0009].any()
    assert float(np.max(np.abs(got - ref))) <= TOL
