"""The resample walker's row groups against the FP64 oracle
(DerampAndResample.cu:348-520 semantics) in launches so small that every strip is
one group: groups of fewer rows, several azimuth keys a row, and the two forms of
the phase.  (Strips of many groups: test_gpu_resample_walk.py.)  Samples agree to max|dz|/RMS|z| <= 1e-5, the tolerance of
the resampled samples everywhere: FP32 sums of 24 terms of magnitude up to
the largest sample reach 24 * 2^-24 * max/RMS, about 6e-6."""
import ctypes as C

import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _run(tops, dev, d, kaz, krg, mbox, sbox, az_shift, ca, cr, kt, tref, fdc):
    N = tops.native
    L = N.load()
    ctx = L.tops_ctx_create(N.ptr(kaz, C.c_float), N.ptr(krg, C.c_float), 12)
    assert ctx, N.last_error()
    try:
        g = N.BurstGeom((C.c_int * 4)(*mbox), (C.c_int * 4)(*sbox), 0, len(kt), d["dt"],
                        az_shift, (C.c_double * 6)(*ca), (C.c_double * 6)(*cr))
        bufs = [dev.put(a) for a in (d["S"], kt, tref, fdc)]
        ml, mp = mbox[3] - mbox[2] + 1, mbox[1] - mbox[0] + 1
        out = dev.empty(ml * mp * 8)
        N.check(L.tops_resample_burst(ctx, C.byref(g), *[b.data_ptr() for b in bufs],
                                      out.data_ptr(), 0, None))
        return dev.get(out, np.complex64, (ml, mp))
    finally:
        L.tops_ctx_destroy(ctx)


@pytest.fixture(scope="module")
def d(tops, orc):
    pair = tops.synth.single_burst_small()
    m = pair.master
    kt, tref, fdc, _ = pair.params()
    kaz, krg = orc.lut(prf=m.prf, abw=m.azimuth_bandwidth, rsr2x=2 * m.range_sampling_rate)
    ca, cr = pair.cpm(0)
    return dict(S=pair.burst(0, "slave"), kt=kt[0].copy(), tref=tref[0].copy(),
                fdc=fdc[0].copy(), kaz=kaz, krg=krg, ca=np.array(ca), cr=np.array(cr),
                L=m.lines_per_burst, P=m.samples_per_burst, dt=m.az_time_interval)


# (rows, columns) of the top-left of the burst that are resampled at about one
# slave line a row: part of a group .. 17 of them one below the other
@pytest.mark.parametrize("rows,cols", [(1, 52), (3, 53), (5, 64), (31, 105), (33, 157), (67, 300)])
@pytest.mark.parametrize("form", ["smooth", "rough", "taps"])
def test_groups(tops, orc, dev, d, rows, cols, form):
    """smooth: the arrays as they are (the phase as a quadratic of the
    column); rough: FM rate and Doppler centroid with noise of 1e-6 and a step
    in the middle of a strip; taps: range taps whose rows do not sum to 1.
    The last two take the FP64 phases column by column."""
    L, P = d["L"], d["P"]
    mbox, sbox = [20, 20 + cols - 1, 30, 30 + rows - 1], [0, P - 1, 0, L - 1]
    # positions of the burst's polynomials: y = line + 1.3 - 0.35 of the
    # width's fraction, so that a strip holds up to a dozen keys a row
    ca = np.array([30 + (rows - 1) / 2 + 1.3, (rows - 1) / 4, 0.0875, 0, 0, 0])
    cr = np.array([20 + (cols - 1) / 2 + 0.6, 0.05, (cols - 1) / 4, 0, 0, 0])
    kt, tref, fdc, krg = d["kt"].copy(), d["tref"].copy(), d["fdc"].copy(), d["krg"]
    if form == "rough":
        rng = np.random.default_rng(5)
        kt *= 1 + 1e-6 * rng.standard_normal(P)
        fdc += 1e-3 * rng.standard_normal(P)
        fdc[45:] += 0.5
    if form == "taps":
        k2 = np.asarray(krg, np.float32).reshape(-1, 12)
        krg = (k2 * np.linspace(0.9, 1.1, len(k2), dtype=np.float32)[:, None]).reshape(krg.shape)
    ref = orc.resample(d["S"], mbox, sbox, 0, d["dt"], 0.21, ca, cr, d["kaz"], krg, kt, tref, fdc)
    got = _run(tops, dev, d, d["kaz"], krg, mbox, sbox, 0.21, ca, cr, kt, tref, fdc)
    if rows == 1:   # a box of one line has no normalised line (0 / 0): every output is 0
        assert not ref.any() and not got.any()
        return
    e = rel_err(got, ref)
    print(f"  {form} {rows} x {cols}: {e:.3e}", flush=True)
    assert e <= TOL
