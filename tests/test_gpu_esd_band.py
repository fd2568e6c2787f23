"""The band form of the ESD sums against the oracle (EstESD.cu:914-1217
semantics): windows of 2 to 8 lines, widths that end inside a thread's 4 columns
or a band's last one, overlaps of few and of different lines (row blocks that
walk up and down, overlaps without lines), zero and extreme samples.  The band
sums agree as the tiles' do: a sample whose coherence is within rounding of the
threshold may fall on either side of it (0.25 of a phasor per overlap allows
none here), and the sums of FP32 phasors otherwise to 1e-6 of their number."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("win", [(2, 4), (3, 10), (4, 16), (5, 21), (6, 20), (7, 31), (8, 32)])
@pytest.mark.parametrize("sizes,pixels", [([1, 40, 0, 97], 24001), ([160], 21003),
                                          ([17, 16, 33, 100, 64], 15002)])
def test_bands(tops, orc, dev, win, sizes, pixels):
    N = tops.native
    L = N.load()
    wa, wr = win
    rng = np.random.default_rng(wa * 7 + len(sizes))
    n = sum(sizes)
    M = [np.round(rng.normal(0, 300, (n, pixels, 2))).astype(np.int16) for _ in range(2)]
    S = []
    for k in range(2):
        mc = M[k][..., 0] + 1j * M[k][..., 1]
        s = mc * np.exp(1j * (0.3 + 0.2 * k)) + rng.normal(0, 60, (n, pixels)) \
            + 1j * rng.normal(0, 60, (n, pixels))
        s = s.astype(np.complex64)
        s[rng.random((n, pixels)) < 0.01] = 0
        # double differences whose square underflows or overflows FP32 (the
        # window sums of both stay inside its range)
        s[:, 100:140] *= np.float32(1e-13)
        s[:, 5000:5040] *= np.float32(1e5)
        S.append(s)
    args = (M[0], M[1], S[0], S[1])
    sz = np.array(sizes, np.int32)
    d = [dev.put(np.ascontiguousarray(a)) for a in args]
    shifts, sums = np.zeros(len(sz)), np.zeros(2 * len(sz))
    N.check(L.tops_esd_shifts(*[x.data_ptr() for x in d], N.ptr(sz, C.c_int), len(sz), pixels, wa,
                              wr, 0.3, 4500.0, 2e-3, N.ptr(shifts), N.ptr(sums), None))
    ref, rsums = orc.esd(*args, sz, pixels, wa, wr, 0.3, 4500.0, 2e-3)
    got, rsums = sums.reshape(-1, 2), np.asarray(rsums).reshape(-1, 2)
    e = np.abs(got - rsums).max(axis=1)
    print(f"  {wa} x {wr}, lines {sizes} x {pixels}: sums |d| {e.max():.2e}", flush=True)
    for i, k in enumerate(sizes):
        assert e[i] <= 0.25 + 1e-6 * k * pixels
        assert k > 0 or not got[i].any()


@pytest.mark.parametrize("win", [(2, 8), (3, 10), (5, 20), (8, 32)])
def test_bands_sum_to_rounding(tops, orc, dev, win):
    """Coherent samples throughout (0.95, none near a threshold, none zero): the
    sums differ from the oracle's by the rounding of the unit phasors alone, at
    most 2^-22 each (a reciprocal square root good to an ulp and a product), and
    as roundings of either sign by about the square root of their number: 32 times
    that is allowed."""
    N = tops.native
    L = N.load()
    wa, wr = win
    sizes, pixels = [97, 60, 33], 15002
    rng = np.random.default_rng(wa)
    n = sum(sizes)
    M, S = [], []
    for k in range(2):
        m = np.round(rng.normal(0, 300, (n, pixels, 2))).astype(np.int16)
        m[(m == 0).all(-1)] = 1
        mc = m[..., 0] + 1j * m[..., 1]
        th = 0.3 + 0.2 * k + 1e-3 * np.arange(pixels) * (1 - 2 * k)
        S.append((mc * np.exp(1j * th) + rng.normal(0, 60, (n, pixels))
                  + 1j * rng.normal(0, 60, (n, pixels))).astype(np.complex64))
        M.append(m)
    args = (M[0], M[1], S[0], S[1])
    sz = np.array(sizes, np.int32)
    d = [dev.put(np.ascontiguousarray(a)) for a in args]
    shifts, sums = np.zeros(len(sz)), np.zeros(2 * len(sz))
    N.check(L.tops_esd_shifts(*[x.data_ptr() for x in d], N.ptr(sz, C.c_int), len(sz), pixels, wa,
                              wr, 0.3, 4500.0, 2e-3, N.ptr(shifts), N.ptr(sums), None))
    _, rsums = orc.esd(*args, sz, pixels, wa, wr, 0.3, 4500.0, 2e-3)
    e = np.abs(sums.reshape(-1, 2) - np.asarray(rsums).reshape(-1, 2)).max(axis=1)
    bound = 32 * 2.0 ** -22 * np.sqrt(sz.astype(float) * pixels)
    print(f"  {wa} x {wr}: sums |d| {e}, allowed {bound}", flush=True)
    assert np.all(e <= bound)
