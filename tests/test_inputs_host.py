"""
The host side of the input read-back (``d4_inputs_begin``/``d4_inputs_wait``)
and the errors it meets, without a GPU: the library runs in a process of its
own against a stand-in for the HIP runtime with two devices that refuses what
the runtime refuses (an event recorded on a stream of another device) and
fails where the test tells it to.
"""

import os
import shutil
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

RUNTIME = r"""
#include <cstdlib>
#include <cstring>
#include <cstddef>
extern "C" {
// what the test reads and sets
int fake_device = 0, fake_last = 0, fake_launches = 0, fake_launch_device = -1;
int fake_pinned = 0, fake_freed = 0, fake_syncs = 0;
int fail_query = 0, fail_record = 0, fail_wait = 0, fail_sync = 0;

static int err(int e) { if (e) fake_last = e; return e; }
static int take(int* f) { int e = *f; *f = 0; return err(e); }
struct Event { int device; };
// stream handles: 0x1000 * (device + 1) + k; null: the current device's
static int device_of(void* s) { return s ? (int)((size_t)s / 0x1000) - 1 : fake_device; }

int hipGetDevice(int* d) { *d = fake_device; return 0; }
int hipSetDevice(int d) { if (d < 0 || d > 1) return err(101); fake_device = d; return 0; }
int hipMalloc(void** p, size_t n) { *p = malloc(n); return 0; }
int hipFree(void* p) { free(p); return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int) { memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { memcpy(d, s, n); return 0; }
int hipGetSymbolAddress(void** p, const void*) { static char scratch[64]; *p = scratch; return 0; }
int hipHostMalloc(void** p, size_t n, unsigned) { ++fake_pinned; *p = malloc(n); return 0; }
int hipHostFree(void* p) { ++fake_freed; free(p); return 0; }
int hipEventCreateWithFlags(void** e, unsigned) { *e = new Event{fake_device}; return 0; }
int hipEventDestroy(void* e) { delete (Event*)e; return 0; }
int hipEventRecord(void* e, void* s) {
  if (fail_record) return take(&fail_record);
  return err(((Event*)e)->device == device_of(s) ? 0 : 400);
}
int hipEventSynchronize(void*) { return take(&fail_wait); }
int hipStreamIsCapturing(void*, int* st) { *st = 0; return take(&fail_query); }
int hipStreamSynchronize(void*) { ++fake_syncs; return take(&fail_sync); }
int hipGetLastError() { int e = fake_last; fake_last = 0; return e; }
const char* hipGetErrorString(int) { return "stand-in error"; }
int hipLaunchKernel(const void*, size_t, size_t, size_t, size_t, void**, size_t, void*) { return 0; }
void* __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*,
                           void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
// the launch configuration carries the stream
int __hipPushCallConfiguration(size_t, size_t, size_t, size_t, size_t, void* s) {
  ++fake_launches;
  fake_launch_device = device_of(s);
  return 0;
}
int __hipPopCallConfiguration(void*, void*, size_t*, void**) { return 0; }
}
"""

PRELUDE = r"""
import ctypes, importlib.util, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
spec = importlib.util.spec_from_file_location("_lib", sys.argv[2])
L = importlib.util.module_from_spec(spec)
spec.loader.exec_module(L)
lib = ctypes.CDLL(str(L.LIB_PATH))
for name, (res, args) in L.SIGNATURES.items():
    getattr(lib, name).restype, getattr(lib, name).argtypes = res, args
def var(name):
    return ctypes.c_int.in_dll(fake, name)
zeros = (ctypes.c_double * (104 * 104 * 49))()
izeros = (ctypes.c_int32 * (104 * 7))()
tb = L.Tables()
for name, kind in L.Tables._fields_:
    if name not in ("wfpair", "alpha", "refslot"):
        setattr(tb, name, ctypes.cast(zeros if kind is L._dp else izeros, kind))
def context(device):
    out = ctypes.c_void_p()
    assert lib.d4_context_create(device, ctypes.byref(tb), ctypes.byref(out)) == 0
    return out
numbers = (ctypes.c_int64 * 4)(1, 6, 7, 8)
def begin(ctx, stream):
    t = ctypes.c_void_p()
    rc = lib.d4_inputs_begin(ctx, stream, 4, ctypes.cast(numbers, ctypes.c_void_p), 0, None, None,
                             ctypes.byref(t))
    return rc, t
def wait(ctx, t):
    return lib.d4_inputs_wait(ctx, t, None, None)
DEV0, DEV1 = 0x1000, 0x2000  # streams of the two devices
"""


@pytest.fixture(scope="module")
def runtime_so(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("hip")
    (d / "hip.cpp").write_text(RUNTIME)
    so = d / "libstandin.so"
    subprocess.run([cxx, "-std=c++17", "-O1", "-shared", "-fPIC", "-w", str(d / "hip.cpp"),
                    "-o", str(so)], check=True)
    return so


def _run(so, body):
    env = dict(os.environ, PYTHONDONTWRITEBYTECODE="1")
    run = subprocess.run([sys.executable, "-c", PRELUDE + body, str(so),
                          str(ROOT / "tad_dftd4_amd" / "_lib.py")],
                         capture_output=True, text=True, timeout=60, env=env)
    assert run.returncode == 0, run.stderr


def test_device_that_is_not_current(runtime_so):
    """The read-back runs on the context's device, whichever is current, and
    leaves the current device as it was; a null stream is that device's."""
    _run(runtime_so, r"""
for device, stream in ((1, DEV1), (1, None), (0, DEV0), (0, None)):
    ctx = context(device)
    for current in (0, 1):
        var("fake_device").value = current
        for k in range(2):  # a new event, then the same one again
            rc, t = begin(ctx, stream)
            assert rc == 0, (device, stream, current, lib.d4_last_error())
            assert var("fake_launch_device").value == device
            assert var("fake_device").value == current
            assert wait(ctx, t) == 0
    lib.d4_context_destroy(ctx)
""")


def test_failed_query_leaves_no_error(runtime_so):
    """A capture query that fails is reported by its own call; the next call's
    launches do not find its error."""
    _run(runtime_so, r"""
ctx = context(0)
var("fail_query").value = 906
rc, t = begin(ctx, DEV0)
assert rc == L.D4_ERR_DEVICE and not t.value
assert var("fake_last").value == 0
rc, t = begin(ctx, DEV0)
assert rc == 0 and wait(ctx, t) == 0
""")


@pytest.mark.parametrize("sync", [0, 700])
def test_failed_record(runtime_so, sync):
    """An event that cannot be recorded behind the launched read: its host memory
    is used again only after the stream was waited for."""
    _run(runtime_so, r"""
ctx = context(0)
var("fail_record").value = 400
var("fail_sync").value = %d
syncs, pinned, launches = (var(k).value for k in ("fake_syncs", "fake_pinned", "fake_launches"))
rc, t = begin(ctx, DEV0)
assert rc == L.D4_ERR_DEVICE and not t.value and var("fake_last").value == 0
assert var("fake_launches").value == launches + 1 and var("fake_syncs").value == syncs + 1
rc, t = begin(ctx, DEV0)
assert rc == 0 and wait(ctx, t) == 0
# a stream that could not be waited for may still write: new memory then
assert var("fake_pinned").value == pinned + (2 if %d else 1)
lib.d4_context_destroy(ctx)
assert var("fake_freed").value == var("fake_pinned").value
""" % (sync, sync))


def test_failed_wait(runtime_so):
    """A wait that fails is reported, and the host memory that the read may
    still write is not given to the next call."""
    _run(runtime_so, r"""
ctx = context(0)
rc, t = begin(ctx, DEV0)
pinned = var("fake_pinned").value
var("fail_wait").value = 900
assert wait(ctx, t) == L.D4_ERR_DEVICE and var("fake_last").value == 0
rc, t = begin(ctx, DEV0)
assert rc == 0 and var("fake_pinned").value == pinned + 1 and wait(ctx, t) == 0
lib.d4_context_destroy(ctx)
assert var("fake_freed").value == var("fake_pinned").value
""")
