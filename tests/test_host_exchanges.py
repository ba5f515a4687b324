"""Host logic of the exchanges with host memory, on a stand-in HIP runtime:
memory is the host's, kernels do nothing, and every stream and event belongs to
the device that was current when it was made.  An event recorded on another
device's stream, or none at all, is an error, as in HIP.

Each check is a program of its own with the stand-in preloaded.
"""
import os
import subprocess
import sys

import pytest

import caviar_amd

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RUNTIME = r"""
#include <cstdlib>
#include <cstring>
#include <cstddef>
typedef struct { unsigned x, y, z; } dim3_t;
struct Obj { int device; };
static thread_local int current = 0;
static int pinned_left = 1 << 30;
static Obj none{0};
static Obj *stream(void *s) { return s ? (Obj *)s : &none; }
extern "C" {
void fake_current(int d) { current = d; }
void fake_pinned(int left) { pinned_left = left; }
int hipGetDeviceCount(int *n) { *n = 2; return 0; }
int hipSetDevice(int d) { current = d; return 0; }
int hipGetLastError() { return 0; }
int hipMalloc(void **p, size_t n) { *p = calloc(n ? n : 1, 1); return 0; }
int hipFree(void *p) { free(p); return 0; }
int hipHostMalloc(void **p, size_t n, unsigned)
{
  if (pinned_left-- <= 0) return 2;
  return hipMalloc(p, n);
}
int hipHostFree(void *p) { free(p); return 0; }
int hipHostGetDevicePointer(void **d, void *h, unsigned) { *d = h; return 0; }
int hipMemset(void *p, int v, size_t n) { memset(p, v, n); return 0; }
int hipMemsetAsync(void *p, int v, size_t n, void *) { return hipMemset(p, v, n); }
int hipMemcpy(void *d, const void *s, size_t n, int) { if (n) memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *) { return hipMemcpy(d, s, n, k); }
int hipStreamCreate(void **s) { *s = new Obj{current}; return 0; }
int hipStreamCreateWithFlags(void **s, unsigned) { return hipStreamCreate(s); }
int hipStreamDestroy(void *s) { delete (Obj *)s; return 0; }
int hipStreamSynchronize(void *) { return 0; }
int hipStreamWaitEvent(void *, void *e, unsigned) { return e ? 0 : 400; }
int hipEventCreate(void **e) { *e = new Obj{current}; return 0; }
int hipEventCreateWithFlags(void **e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void *e) { delete (Obj *)e; return 0; }
int hipEventRecord(void *e, void *s)
{
  return e && ((Obj *)e)->device == stream(s)->device ? 0 : 400;
}
int hipEventSynchronize(void *e) { return e ? 0 : 400; }
int hipLaunchKernel(const void *, dim3_t, dim3_t, void **, size_t, void *) { return 0; }
int __hipPushCallConfiguration(dim3_t, dim3_t, size_t, void *) { return 0; }
int __hipPopCallConfiguration(dim3_t *, dim3_t *, size_t *, void **) { return 0; }
}
"""

HEAD = """
import ctypes, numpy as np
import caviar_amd
from caviar_amd import Engine, configs
fake = ctypes.CDLL(None)
lib = caviar_amd.load_library()
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    if not os.path.exists(caviar_amd.LIB_PATH):
        from caviar_amd import build
        build.build()
    d = tmp_path_factory.mktemp("hip")
    src, so = str(d / "fake.cpp"), str(d / "libfake.so")
    with open(src, "w") as f:
        f.write(RUNTIME)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-w", src, "-o", so], check=True)
    return so


def run(runtime, body):
    preload = ":".join(filter(None, [runtime, os.environ.get("LD_PRELOAD")]))
    env = dict(os.environ, LD_PRELOAD=preload, PYTHONPATH=ROOT)
    p = subprocess.run([sys.executable, "-c", HEAD + body], env=env, cwd=ROOT, capture_output=True,
                       text=True, timeout=120)
    assert p.returncode == 0, p.stdout + p.stderr


def test_download_of_no_atoms(runtime):
    """A context without atoms gives nothing and no error, as does one of none."""
    run(runtime, """
h = ctypes.c_void_p()
assert lib.cav_create(0, ctypes.byref(h)) == 0
out = np.zeros(3)
p = out.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
for which in range(4):
    assert lib.cav_download(h, which, p) == 0, lib.cav_last_error(h)
    assert lib.cav_upload(h, which, p) == 0, lib.cav_last_error(h)
""")


SETUP = """
def engine(device):
    s = configs.ions(n=64, rho=0.3, kmax=2, seed=1)
    e = Engine(s, device=device)
    e.setup()
    return e
"""


def test_staging_belongs_to_the_contexts_device(runtime):
    """Each call that may be an engine's first exchange, while another device is
    current, and the ones that follow it."""
    run(runtime, SETUP + """
first = dict(virial=lambda e: e.virial(), get=lambda e: e.get("pos"),
             set=lambda e: e.set("pos", e.system.pos), energy=lambda e: e.energy(),
             points=lambda e: e.point_field("r", e.system.pos),
             adjoint=lambda e: e.adjoint(np.ones((e.n, 3))))
for name, call in first.items():
    a, b = engine(0), engine(1)
    for e, other in ((a, 1), (b, 0)):
        fake.fake_current(other)
        call(e)
        for later in first.values():
            fake.fake_current(other)
            later(e)
""")


def test_exchanges_without_pinned_memory(runtime):
    """Where no pinned memory is to be had, every exchange takes plain copies."""
    run(runtime, SETUP + """
e = engine(0)
fake.fake_pinned(0)
e.virial()
e.energy()
e.get("pos")
e.set("pos", e.system.pos)
e.point_field("r", e.system.pos)
e.point_field("k", e.system.pos)
e.adjoint(np.ones((e.n, 3)))
""")
