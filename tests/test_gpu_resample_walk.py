"""The resample walker over strips of many row groups, against the FP64 oracle
(DerampAndResample.cu:348-520 semantics): strips that end at, before and past
the 32 rows of a position table, tall strips with low ones after them, slave
lines that advance by other than one a row, lines that change along a row, and
phase arrays that are not finite.  A one-burst plan fixes the strip height.
Samples agree to max|dz|/RMS|z| <= 1e-5, as everywhere: FP32 sums of 24 terms of
magnitude up to the largest sample reach 24 * 2^-24 * max/RMS, about 6e-6."""
import ctypes as C

import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.fixture(scope="module")
def d(tops, orc):
    pair = tops.synth.single_burst_small()
    m = pair.master
    kt, tref, fdc, _ = pair.params()
    kaz, krg = orc.lut(prf=m.prf, abw=m.azimuth_bandwidth, rsr2x=2 * m.range_sampling_rate)
    return dict(S=pair.burst(0, "slave"), kt=kt[0].copy(), tref=tref[0].copy(),
                fdc=fdc[0].copy(), kaz=kaz, krg=krg, L=m.lines_per_burst, P=m.samples_per_burst,
                dt=m.az_time_interval)


def _arrays(d, form):
    """smooth: the arrays as they are (the phase as a quadratic of the column);
    rough: FM rate and Doppler centroid with noise and a step; taps: range taps
    whose rows do not sum to 1.  The last two take FP64 phases by column."""
    kt, tref, fdc, krg = d["kt"].copy(), d["tref"].copy(), d["fdc"].copy(), d["krg"]
    if form == "rough":
        rng = np.random.default_rng(5)
        kt *= 1 + 1e-6 * rng.standard_normal(len(kt))
        fdc += 1e-3 * rng.standard_normal(len(kt))
        fdc[45:] += 0.5
    if form == "taps":
        k2 = np.asarray(krg, np.float32).reshape(-1, 12)
        krg = (k2 * np.linspace(0.9, 1.1, len(k2), dtype=np.float32)[:, None]).reshape(krg.shape)
    return kt, tref, fdc, krg


def _both(tops, orc, dev, d, rows, cols, strip_rows, rate, shear, line, arrays):
    """(plan, oracle) of rows x cols outputs whose slave line is
    line + rate * row + shear * column."""
    N = tops.native
    L = N.load()
    kt, tref, fdc, krg = arrays
    mbox, sbox = [20, 19 + cols, 30, 29 + rows], [0, d["P"] - 1, 0, d["L"] - 1]
    ca = [line + rate * (rows - 1) / 2 + shear * (cols - 1) / 2, rate * (rows - 1) / 4,
          shear * (cols - 1) / 4, 0, 0, 0]
    cr = [20 + (cols - 1) / 2 + 0.6, 0.05, (cols - 1) / 4, 0, 0, 0]
    ref = orc.resample(d["S"], mbox, sbox, 0, d["dt"], 0.21, ca, cr, d["kaz"], krg, kt, tref, fdc)
    ctx = L.tops_ctx_create(N.ptr(d["kaz"], C.c_float), N.ptr(krg, C.c_float), 12)
    assert ctx, N.last_error()
    g = N.BurstGeom((C.c_int * 4)(*mbox), (C.c_int * 4)(*sbox), 0, d["P"], d["dt"], 0.21,
                    (C.c_double * 6)(*ca), (C.c_double * 6)(*cr))
    bufs = [dev.put(a) for a in (d["S"], kt, tref, fdc)]
    out = dev.empty(rows * cols * 8)
    item = (N.BurstItem * 1)(N.BurstItem(g, *[b.data_ptr() for b in bufs], out.data_ptr(), None,
                                         None))
    plan = L.tops_plan_create(ctx, item, 1, 3, 10, strip_rows)
    assert plan, N.last_error()
    N.check(L.tops_plan_run(plan, None))
    got = dev.get(out, np.complex64, (rows, cols)).copy()
    L.tops_plan_destroy(plan)
    L.tops_ctx_destroy(ctx)
    return got, ref


@pytest.mark.parametrize("strip_rows", [8, 32, 36, 68, 200])
@pytest.mark.parametrize("form", ["smooth", "rough", "taps"])
def test_strips_of_many_groups(tops, orc, dev, d, form, strip_rows):
    """One line a row; 203 rows leave a last group of 3 and, for the taller
    strips, low strips after the tall ones."""
    got, ref = _both(tops, orc, dev, d, 203, 157, strip_rows, 1.0, 2e-4, 31.3, _arrays(d, form))
    e = rel_err(got, ref)
    print(f"  {form}, strips of {strip_rows}: {e:.3e}", flush=True)
    assert e <= TOL


@pytest.mark.parametrize("rate", [0.5, 0.8, 0.99, 1.1, 1.25, 1.5, 1.8, 2.0, 2.9, -1.0, 0.0])
@pytest.mark.parametrize("shear", [0.0, 0.03, -0.08])
def test_line_rates_and_shear(tops, orc, dev, d, rate, shear):
    """Groups whose slave lines advance by other than 4, spread over more lines
    than the window reaches, or run backwards, with up to 12 lines along a
    strip's row."""
    line = 40.4 + (150 * -rate if rate < 0 else 0) + (105 * -shear if shear < 0 else 0)
    for form in ("smooth", "rough"):
        got, ref = _both(tops, orc, dev, d, 150, 105, 68, rate, shear, line, _arrays(d, form))
        e = rel_err(got, ref)
        print(f"  {form}, {rate} lines a row, {shear} a column: {e:.3e}", flush=True)
        assert np.abs(ref).min() > 0 or rate == 0.0   # interior throughout
        assert e <= TOL


@pytest.mark.parametrize("rate", [1.0, 2.0])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_phase_arrays_that_are_not_finite(tops, orc, dev, d, rate, bad):
    """A column without a finite phase spoils the outputs whose taps hold it and
    no others."""
    kt, tref, fdc, krg = _arrays(d, "smooth")
    fdc[100] = bad
    got, ref = _both(tops, orc, dev, d, 150, 157, 36, rate, 0.0, 31.3, (kt, tref, fdc, krg))
    lost = ~np.isfinite(ref)
    assert 0 < lost.sum() <= 13 * 150
    assert np.array_equal(~np.isfinite(got), lost)
    assert rel_err(got[~lost], ref[~lost]) <= TOL


def test_fitted_phase_rounds_like_the_sum(tops, orc, dev, d):
    """The phase fitted over a strip's columns against the FP64 sum of its 12
    columns, which one range row whose taps sum to 1 + 4e-6 makes the walker take:
    the RMS error of the samples must be the same within 0.3 %.  The reference
    time bends the phase by 2.1e-8 rad (1.4e-8 RMS) from a quadratic over 64
    columns, which would be 0.7 % of the samples' 1.16e-7 if it were left out."""
    kt, tref, fdc, krg = _arrays(d, "smooth")
    bend = 2.4e-8 / (2 * np.pi * np.abs(kt * tref).mean() * 0.38 * 30.0 ** 3)
    bend = bend * (np.arange(len(kt)) - 100.0) ** 3
    tref, fdc = tref + bend, fdc + kt * bend   # kt tref - fdc stays
    uneven = np.array(krg, np.float32).reshape(-1, 12)
    uneven[1023] *= np.float32(1 + 4e-6)
    rms = []
    for k in (krg, uneven.reshape(np.shape(krg))):
        got, ref = _both(tops, orc, dev, d, 400, 417, 68, 1.0, 2e-4, 31.3, (kt, tref, fdc, k))
        rms.append(float(np.sqrt(np.mean(np.abs(got - ref) ** 2) / np.mean(np.abs(ref) ** 2))))
    print(f"  RMS error: fitted {rms[0]:.5e}, summed {rms[1]:.5e}", flush=True)
    assert rms[0] <= 1.003 * rms[1]
