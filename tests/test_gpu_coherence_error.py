"""Rounding of the band coherence (coherence_band.hpp) against that of the
16 x 64 tiles, which serve the same windows on smaller rasters: the same
samples once as a small raster and once as the middle of a wide one, both
against FP64 window sums.  The bands' RMS error must not be larger (2 % for the
statistics of 0.9 M samples).  Emulated in FP32 the bands' is 0.1 to 4 % below
the tiles'; one left-to-right chain per window is 3 to 8 % above."""
import numpy as np
import pytest

H, W = 480, 1984   # 30 x 31 tiles: fewer than 4 per CU; three times that are more than 8


def _sums(v, wa, wr):
    a = np.cumsum(np.pad(v, ((1, 0), (0, 0))), 0)
    a = a[wa:] - a[:-wa]
    a = np.cumsum(np.pad(a, ((0, 0), (1, 0))), 1)
    return a[:, wr:] - a[:, :-wr]


@pytest.mark.gpu
@pytest.mark.parametrize("wa,wr", [(6, 24), (8, 32), (7, 20), (4, 16), (5, 20)])
def test_band_error_is_not_above_the_tiles(tops, dev, wa, wr):
    N = tops.native
    L = N.load()
    rng = np.random.default_rng(10 * wa + wr)
    z = rng.normal(0, 300, (H, W, 2))
    m = np.round(z).astype(np.int16)
    s = (0.8 * z + 0.6 * rng.normal(0, 300, z.shape)).astype(np.float32)
    dx, dy = (wr - 1) // 2, (wa - 1) // 2

    def run(m, s):
        h, w = m.shape[:2]
        dm, ds, out = dev.put(m), dev.put(s), dev.empty(4 * h * w)
        N.check(L.tops_coherence(dm.data_ptr(), ds.data_ptr(), w, h, dx, dy, wr, wa,
                                 out.data_ptr(), N.MODE_FAST, None))
        return dev.get(out, np.float32, (h, w)).copy()

    tile = run(m, s)
    band = run(*(np.ascontiguousarray(np.concatenate([a, a, a], 1)) for a in (m, s)))[:, W:2 * W]
    mc = m[..., 0].astype(np.float64) + 1j * m[..., 1]
    sc = s[..., 0].astype(np.float64) + 1j * s[..., 1]
    p = mc * sc.conj()
    ref = np.hypot(_sums(p.real, wa, wr), _sums(p.imag, wa, wr)) / np.sqrt(
        _sums(np.abs(sc) ** 2, wa, wr) * _sums(np.abs(mc) ** 2, wa, wr))
    # windows inside the small raster: output (r + dy, c + dx) is window (r, c)
    n, k = ref.shape
    rms = [float(np.sqrt(np.mean((v[dy:dy + n, dx:dx + k] - ref) ** 2))) for v in (band, tile)]
    print(f"  {wa} x {wr}: RMS error bands {rms[0]:.3e}, tiles {rms[1]:.3e}", flush=True)
    assert rms[0] <= 1.02 * rms[1]
