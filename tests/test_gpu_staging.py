"""Host buffers of the reference-style calls: sizes about the smallest staging
chunk (4 MiB; an eighth of larger uploads, 32 MiB for downloads, two chunks in
flight), unaligned, pinned and pageable, from several threads at once, give the
bytes that the device entry points give."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(tops, orc):
    pair = tops.synth.single_burst_small()
    m = pair.master
    kt, tref, fdc, _ = pair.params()
    kaz, krg = orc.lut(prf=m.prf, abw=m.azimuth_bandwidth, rsr2x=2 * m.range_sampling_rate)
    return m, kt[0], tref[0], fdc[0], kaz, krg


# lines x 1024 samples: the slave (4 bytes a sample) just under, at and over 4
# MiB, the smallest copy that is staged, and of five chunks; the output has twice
# the bytes, up to a chunk and a part of the next
@pytest.mark.parametrize("lines", [1023, 1024, 1025, 5121])
@pytest.mark.parametrize("kind", ["pageable", "unaligned", "pinned"])
def test_sizes_and_kinds(tops, orc, dev, lines, kind):
    N = tops.native
    L = N.load()
    torch = dev.torch
    m, kt, tref, fdc, kaz, krg = _case(tops, orc)
    P = 1024
    kt, tref, fdc = (np.ascontiguousarray(a[:P]) for a in (kt, tref, fdc))
    rng = np.random.default_rng(lines)

    def host(nbytes, dtype, shape):
        if kind == "pinned":
            raw = torch.empty(nbytes, dtype=torch.uint8, pin_memory=True).numpy()
        else:
            off = 12 if kind == "unaligned" else 0
            raw = np.empty(nbytes + 16, np.uint8)[off:off + nbytes]
        return raw.view(dtype).reshape(shape)

    S = host(lines * P * 4, np.int16, (lines, P, 2))
    M = host(lines * P * 4, np.int16, (lines, P, 2))
    S[:] = rng.integers(-900, 900, S.shape)
    M[:] = rng.integers(-900, 900, M.shape)
    out, coh = host(lines * P * 8, np.float32, (lines, P, 2)), host(lines * P * 4, np.float32, (lines, P))
    ca = np.array([(lines - 1) / 2 + 0.2, (lines - 1) / 4, 0.05, 0, 0, 0])
    cr = np.array([(P - 1) / 2 + 0.4, 0.02, (P - 1) / 4, 0, 0, 0])
    box = (C.c_int * 4)(0, P - 1, 0, lines - 1)
    L.tops_clear_error()
    d = L.DerampDemodResample_ESD(S.ctypes.data, N.ptr(ca), N.ptr(cr), 0.0, out.ctypes.data,
                                  N.ptr(kaz, C.c_float), N.ptr(krg, C.c_float), 0, P, lines, box,
                                  box, lines, P, m.az_time_interval, N.ptr(kt), N.ptr(tref),
                                  N.ptr(fdc), 12)
    assert d and L.tops_last_error() == 0, N.last_error()
    L.CoherenceEst_ESD(0, 0, P, lines, 4, 1, 10, 3, M.ctypes.data, d, coh.ctypes.data_as(
        C.POINTER(C.c_float)))
    assert L.tops_last_error() == 0, N.last_error()

    g = N.BurstGeom(box, box, 0, P, m.az_time_interval, 0.0, (C.c_double * 6)(*ca),
                    (C.c_double * 6)(*cr))
    ctx = L.tops_ctx_create(N.ptr(kaz, C.c_float), N.ptr(krg, C.c_float), 12)
    bufs = [dev.put(np.array(a)) for a in (S, kt, tref, fdc, M)]
    do, dc = dev.empty(lines * P * 8), dev.empty(lines * P * 4)
    N.check(L.tops_resample_burst(ctx, C.byref(g), *[b.data_ptr() for b in bufs[:4]],
                                  do.data_ptr(), 0, None))
    N.check(L.tops_coherence(bufs[4].data_ptr(), do.data_ptr(), P, lines, 4, 1, 10, 3,
                             dc.data_ptr(), 0, None))
    assert np.array_equal(out, dev.get(do, np.float32, (lines, P, 2)))
    assert np.array_equal(coh, dev.get(dc, np.float32, (lines, P)))
    L.tops_ctx_destroy(ctx)


def test_sums_from_several_threads(tops, dev):
    """The ESD's band sums land in a pinned block of the call's own: threads on
    streams of their own, with bands of their own, get their own sums."""
    N = tops.native
    L = N.load()
    torch = dev.torch
    rng = np.random.default_rng(3)
    n, P = 40, 600
    sizes = np.array([n, n], np.int32)
    cases = []
    for _ in range(6):
        M = rng.integers(-300, 300, (2, 2 * n, P, 2)).astype(np.int16)
        S = (M + rng.normal(0, 30, M.shape)).astype(np.float32)
        cases.append([torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in
                      (M[0], M[1], S[0], S[1])])

    def call(d, stream):
        shifts, sums = np.zeros(2), np.zeros(4)
        N.check(L.tops_esd_shifts(*[x.data_ptr() for x in d], N.ptr(sizes, C.c_int), 2, P, 6, 24,
                                  0.3, 4500.0, 0.002, N.ptr(shifts), N.ptr(sums), stream))
        return sums

    want = [call(d, None) for d in cases]
    streams = [torch.cuda.Stream() for _ in cases]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        for _ in range(20):
            if not np.array_equal(call(cases[i], C.c_void_p(streams[i].cuda_stream)), want[i]):
                bad.append(i)

    th = [threading.Thread(target=work, args=(i,)) for i in range(len(cases))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad


# bytes: chunks of an eighth up to 256 MiB, then of 32 MiB; downloads in 32 MiB
# chunks, whose two buffers are taken in turn
@pytest.mark.parametrize("nbytes", [(4 << 20) + 4, (70 << 20) + 12, (256 << 20) - 8,
                                    (256 << 20) + 8, (300 << 20) + 20])
@pytest.mark.parametrize("offset", [0, 4])
def test_staged_copies(tops, dev, nbytes, offset):
    """The staging layer's own copies, up and down, of sizes past every change of
    its chunks and with a part of a chunk left."""
    L = tops.native.load()
    up, down = (getattr(L, f"_ZN4tops{len(n)}{n}{a}") for n, a in
                (("staged_upload", "EPvPKvm"), ("staged_download", "EPvPKvm")))
    for f in (up, down):
        f.argtypes, f.restype = [C.c_void_p, C.c_void_p, C.c_size_t], C.c_int
    raw = np.empty(nbytes + 64, np.uint8)
    src = raw[offset:offset + nbytes]
    src[:] = np.arange(nbytes // 4, dtype=np.uint32).view(np.uint8)
    d = dev.empty(nbytes)
    assert up(d.data_ptr(), src.ctypes.data, nbytes) == 0
    got = np.zeros(nbytes + 64, np.uint8)
    assert down(got[offset:].ctypes.data, d.data_ptr(), nbytes) == 0
    assert np.array_equal(got[offset:offset + nbytes], src)
    assert not got[:offset].any() and not got[offset + nbytes:].any()
    assert np.array_equal(d.cpu().numpy(), src)
