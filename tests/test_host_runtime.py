"""Host side of the library on a stand-in HIP runtime (hip_stub.cpp): which
calls it makes, with which tables, and what it does when one fails.  Each test
runs a short program of its own in a process that preloads the stand-in, so
nothing here needs a GPU."""
import os
import subprocess
import sys

import pytest

from conftest import PKG_DIR

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes as C, numpy as np, sys
sys.modules["torch"] = None          # the bindings then load without it
import importlib.util
spec = importlib.util.spec_from_file_location("native", {native!r})
N = importlib.util.module_from_spec(spec)
spec.loader.exec_module(N)
L = N.load()
S = C.CDLL({stub!r})
S.stub_count.restype = S.stub_bad.restype = S.stub_host_blocks.restype = C.c_long
S.stub_fail.argtypes = [C.c_char_p, C.c_long]
S.stub_device_bytes.restype = C.c_size_t
count = lambda what: S.stub_count(what.encode())
lut = np.full(2048 * 12, 1 / 12, np.float32)
ctx = L.tops_ctx_create(N.ptr(lut, C.c_float), N.ptr(lut, C.c_float), 12)
FAKE = 0x10000000                    # a device address: no kernel runs

def geom(lines, pixels):
    g = N.BurstGeom()
    g.master_box[:] = g.slave_box[:] = [0, pixels - 1, 0, lines - 1]
    g.samples_per_burst, g.az_time_interval = pixels, 2e-3
    g.cpm_az[:] = [lines / 2, lines / 4, 0, 0, 0, 0]
    g.cpm_rg[:] = [pixels / 2, 0, pixels / 4, 0, 0, 0]
    return g

def plan(shapes, win=(3, 10), strip_rows=0):
    items = (N.BurstItem * len(shapes))(*[N.BurstItem(geom(h, w), *[FAKE] * 7) for h, w in shapes])
    p = L.tops_plan_create(ctx, items, len(shapes), win[0], win[1], strip_rows)
    assert p, N.last_error()
    return p
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    stub = str(tmp_path_factory.mktemp("stub") / "hip_stub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-w", "-I/opt/rocm/include",
                    os.path.join(HERE, "hip_stub.cpp"), "-o", stub], check=True)
    prelude = PRELUDE.format(native=os.path.join(PKG_DIR, "native.py"), stub=stub)

    def program(text):
        r = subprocess.run([sys.executable, "-c", prelude + text], capture_output=True, text=True,
                           timeout=300, env=dict(os.environ, LD_PRELOAD=stub))
        assert r.returncode == 0, (r.returncode, r.stdout[-2000:], r.stderr[-2000:])
        return r.stdout

    return program


TUNE = """
p = plan([(300 + 40 * i, 2500 + 300 * i) for i in range(7)])
stream = C.c_void_p()
S.hipStreamCreate(C.byref(stream))
best = C.c_int()
N.check(L.tops_plan_tune(p, stream, C.byref(best)))
"""


def test_tune_makes_no_graph(run):
    """Tuning times eager launches: no graph is made, launched and destroyed
    while the plan is being formed."""
    run(TUNE + """
assert L.tops_plan_tune_count(p) > 10 and count("hipGraphInstantiate") == 0
N.check(L.tops_plan_capture_graph(p, stream))
assert count("hipGraphInstantiate") == 1 and S.stub_bad() == 0
""")


def test_coherence_rows_are_the_launched_ones(run):
    """tops_plan_coh_rows and the tuner's entries give the height the batched
    coherence was launched with, 32 included, also in a second tuning."""
    run("""
p = plan([(300 + 40 * i, 2500 + 300 * i) for i in range(7)], strip_rows=64)
N.check(L.tops_plan_run(p, None))
assert S.stub_band_rows() == L.tops_plan_coh_rows(p) == 32 and S.stub_bad() == 0
best = C.c_int()
for _ in range(2):
    N.check(L.tops_plan_tune(p, None, C.byref(best)))
    assert S.stub_bad() == 0
    N.check(L.tops_plan_run(p, None))
    if best.value > 0:
        assert S.stub_band_rows() == L.tops_plan_coh_rows(p)
    # the next tuning starts from a table of another height
    N.check(L.tops_plan_set_groups(p, 1))
""" + """
timed = []
for i in range(L.tops_plan_tune_count(p)):
    v = [C.c_int() for _ in range(4)]
    ms = C.c_float()
    N.check(L.tops_plan_tune_entry(p, i, *[C.byref(x) for x in v], C.byref(ms)))
    timed.append([x.value for x in v])
assert {e[1] for e in timed if e[3] == 2} <= {16, 64, 128, 256} and 32 in {e[1] for e in timed}
""")


def test_coherence_of_very_long_narrow_rasters(run):
    """A raster of more row blocks than a grid has rows is launched with taller
    blocks (3 x 10 windows, one column band)."""
    run("""
for lines in (6_200_000, 6_300_000, 40_000_000):
    N.check(L.tops_coherence(FAKE, FAKE, 5, lines, 4, 1, 10, 3, FAKE, N.MODE_FAST, None))
    assert S.stub_bad() == 0, lines
""")


CALLS = """
import threading
def esd(lines=40, pixels=900):
    n = np.full(3, lines, np.int32)
    sh, su = np.zeros(3), np.zeros(6)
    N.check(L.tops_esd_shifts(*[FAKE] * 4, N.ptr(n, C.c_int), 3, pixels, 6, 24, 0.3, 5e3, 2e-3,
                              N.ptr(sh), N.ptr(su), None))

co = np.array([7e6, 1.0, 0, 0, 0, 0])
og = N.OrbitGeom(*[N.ptr(co)] * 3, 6, 0.0, 2e-3, 0.0, 5e-3, 2.3, 0.0, 0)
def geocoreg(lines, pixels):
    a, r = np.zeros(6), np.zeros(6)
    # (no kernel runs: the sums are not positive definite)
    rc = L.tops_geocoreg(FAKE, lines, pixels, 45.0, 10.0, 3e-4, 3e-4, -32768, C.byref(og),
                         C.byref(og), 0, 99, 0, 99, N.ptr(a), N.ptr(r), None, None, None)
    assert rc in (0, N.TOPS_ERR_NOT_PD), rc
"""


def test_kept_scratch_serves_the_larger_calls_too(run):
    """Idle blocks of small calls give way to a larger one, a call takes the
    smallest block that serves it, and one whose block is not kept takes no
    pinned memory."""
    run(CALLS + """
S.stub_sync_ms(200)
t = [threading.Thread(target=esd) for _ in range(4)]
[x.start() for x in t]; [x.join() for x in t]
S.stub_sync_ms(0)
assert S.stub_host_blocks() == 4
geocoreg(1500, 2200)                 # 5 MB of tile records
made = count("hipMalloc")
for _ in range(5):
    geocoreg(1500, 2200)
    esd()
assert count("hipMalloc") == made, count("hipMalloc") - made
pinned = count("hipHostMalloc")
geocoreg(6000, 6000)                 # 50 MB
assert count("hipHostMalloc") == pinned and S.stub_host_blocks() <= 4
assert S.stub_bad() == 0
""")


def test_kept_scratch_is_given_back(run):
    """Destroying a context gives the idle scratch back."""
    run(CALLS + """
tables = S.stub_device_bytes()
esd(); geocoreg(1500, 2200)
assert S.stub_device_bytes() > tables and S.stub_host_blocks() > 0
L.tops_ctx_destroy(ctx)
assert S.stub_device_bytes() == 0 and S.stub_host_blocks() == 0 and S.stub_bad() == 0
""")


def test_calls_after_a_device_reset(run):
    """Calls that hold nothing of the caller's take new scratch and staging
    buffers when a reset of the device has taken the kept ones."""
    run(CALLS + """
big = np.zeros(3000 * 900 * 2, np.int16)     # a CInt16 raster of 10.8 MB
coh = np.zeros(3000 * 900, np.float32)
def drop_in():
    d = L.ResampleFirstBurst(np.zeros(3000 * 900, np.complex64).ctypes.data, 900, 3000)
    L.CoherenceEst_ESD(0, 0, 900, 3000, 4, 1, 10, 3, big.ctypes.data, d, N.ptr(coh, C.c_float))
    assert L.tops_last_error() == 0
esd(); drop_in()
S.stub_reset()
esd(); drop_in(); geocoreg(300, 300)
assert S.stub_bad() == 0
""")


def test_staging_pool_is_tried_again(run):
    """A pool that could not be made leaves a copy to the runtime, once."""
    run(CALLS + """
S.stub_fail(b"hipHostMalloc", 1)
x = np.zeros(2000 * 900, np.complex64)       # 14.4 MB
L.ResampleFirstBurst(x.ctypes.data, 900, 2000)
assert L.tops_last_error() == 0 and count("hipMemcpyAsync") == 0 and S.stub_host_blocks() == 0
L.ResampleFirstBurst(x.ctypes.data, 900, 2000)
assert L.tops_last_error() == 0 and count("hipMemcpyAsync") > 0 and S.stub_host_blocks() == 2
""")
