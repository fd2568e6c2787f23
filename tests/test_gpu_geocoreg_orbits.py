"""Zero-Doppler solves from a tile's orbit polynomial against the oracle's
Newton solve per post (Geocoreg_cuda.cu:272-307), on DEMs whose last tiles are
ragged, with orbits whose fifth-order term takes none, a part or most of the
posts beyond the polynomial's range, to the full iteration.  Lines and pixels agree to 1e-3, what the FP32 projection of a
post (under a millimetre) leaves room for; the lines, whose error has no part of
the projection's beyond its share along the track, to 1e-4."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# fifth: metres per (10 s)^5; the polynomial's range is (2e-12 / fifth)^0.25 x 10 s,
# where its velocity is within 1e-12 m/s: 1.2e-3 s at 1e4, 2.1e-4 s at 1e7, where a
# tile of 1 arcsec reaches 1e-2 s (test_tiles_in_part: 1.2e-2 s at 1, 6.7e-3 at 10)
@pytest.mark.parametrize("fifth", [0.0, 1e4, 1e7])
@pytest.mark.parametrize("rows,cols", [(1, 1), (4, 64), (5, 65), (61, 333)])
def test_orbit_polynomials(tops, orc, dev, fifth, rows, cols):
    N = tops.native
    L = N.load()
    pair = tops.synth.single_burst_small()
    gm, gs, keep = [], [], []
    for sw, orbit in ((pair.master, pair.morbit), (pair.slave, pair.sorbit)):
        t, x, y, z = tops.synth.orbit_polyfit_inputs(orbit)
        c = [np.array(a, np.float64) for a in N.polyfit_orbit(t, x, y, z)]
        for a in c:
            assert len(a) <= 6
        c = [np.concatenate([a, np.zeros(6 - len(a))]) for a in c]
        c[1][5] += fifth
        first, last = sw.burst_first_line_time[0], sw.burst_last_line_time[0]
        args = (t[len(t) // 2], sw.az_time_interval, first, sw.slr_time_first_pixel,
                sw.range_spacing, 0.5 * (first + last))
        keep.append(c)
        gm.append(N.OrbitGeom(N.ptr(c[0]), N.ptr(c[1]), N.ptr(c[2]), 6, *args, 0))
        gs.append(orc.orbit_geom(c, *args, 0))
    la0, la1, lo0, lo1 = pair.master.burst_ll[0]
    step = 1.0 / 3600
    lat0, lon0 = 0.5 * (la0 + la1) + rows * step / 2, 0.5 * (lo0 + lo1) - cols * step / 2
    rng = np.random.default_rng(rows)
    dem = rng.integers(0, 1500, (rows, cols)).astype(np.int32)
    dem[rng.random((rows, cols)) < 0.05] = -32768
    box = [0, pair.master.samples_per_burst - 1, 0, pair.master.lines_per_burst - 1]
    d, lp = dev.put(dem), dev.empty(4 * dem.size * 8)
    ca, cr, used = np.zeros(6), np.zeros(6), C.c_int64(0)
    rc = L.tops_geocoreg(d.data_ptr(), rows, cols, lat0, lon0, step, step, -32768, C.byref(gm[0]),
                         C.byref(gm[1]), *box, N.ptr(ca), N.ptr(cr), C.byref(used), lp.data_ptr(),
                         None)
    if rc != N.TOPS_ERR_NOT_PD:
        N.check(rc)
    L.tops_clear_error()
    got = dev.get(lp, np.float64, (4, rows, cols))
    for k in range(2):
        line, pix = orc.ell2lp(dem, lat0, lon0, step, step, -32768, gs[k])
        el = float(np.max(np.abs(got[2 * k] - line)))
        ep = float(np.max(np.abs(got[2 * k + 1] - pix)))
        print(f"  {rows} x {cols}, fifth {fifth:g}: line {el:.2e}, pixel {ep:.2e}", flush=True)
        assert el <= 1e-4 and ep <= 1e-3


@pytest.mark.parametrize("fifth", [1.0, 3.0, 10.0])
def test_tiles_in_part(tops, orc, dev, fifth):
    """Fifth-order terms whose range ends inside a tile: some of its posts take
    the polynomial, some the full iteration."""
    test_orbit_polynomials(tops, orc, dev, fifth, 61, 333)
