"""Host logic (exchanges with host memory, launch shapes) on a stand-in HIP
runtime: memory is the host's, kernels only leave their name and grid, and every
stream and event belongs to the device that was current when it was made.  An
event recorded on another device's stream, or none at all, is an error, as in HIP.

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
#include <map>
#include <string>
typedef struct { unsigned x, y, z; } dim3_t;
struct Obj { int device; };
static thread_local int current = 0;
static int pinned_left = 1 << 30;
static int crowd = 0, malloc_device = -1;
static Obj none{0};
struct Call { dim3_t grid, block; size_t shared; void *stream; };
static thread_local Call call;
static std::map<const void *, std::string> &names()
{
  static std::map<const void *, std::string> m;
  return m;
}
static std::string launches;  // "name x y z" lines
static Obj *stream(void *s) { return s ? (Obj *)s : &none; }
extern "C" {
void fake_current(int d) { current = d; }
void fake_pinned(int left) { pinned_left = left; }
void fake_crowd(int most) { crowd = most, malloc_device = -1; }  // F_MAXCELL of flags read back
int fake_malloc_device() { return malloc_device; }
int hipGetDeviceCount(int *n) { *n = 2; return 0; }
int hipSetDevice(int d) { current = d; return 0; }
int hipGetLastError() { return 0; }
int hipMalloc(void **p, size_t n) { malloc_device = current; *p = calloc(n ? n : 1, 1); return 0; }
int hipFree(void *p) { free(p); return 0; }
int hipGetSymbolAddress(void **p, const void *)
{
  static void *scratch = calloc(64 << 20, 1);
  *p = scratch;
  return 0;
}
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
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *)
{
  hipMemcpy(d, s, n, k);
  if (crowd && k == 2 && n == 16 * sizeof(int)) ((int *)d)[13] = crowd;
  return 0;
}
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
int hipLaunchKernel(const void *f, dim3_t g, dim3_t, void **, size_t, void *)
{
  launches += names()[f] + " " + std::to_string(g.x) + " " + std::to_string(g.y) + " " +
              std::to_string(g.z) + "\n";
  return 0;
}
const char *fake_launches() { return launches.c_str(); }
void fake_forget() { launches.clear(); }
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t n, void *s)
{
  call = Call{g, b, n, s};
  return 0;
}
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *n, void **s)
{
  *g = call.grid, *b = call.block, *n = call.shared, *s = call.stream;
  return 0;
}
int hipFuncSetAttribute(const void *, int, int) { return 0; }
void **__hipRegisterFatBinary(const void *) { static void *p; return &p; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *)
{
  names()[host] = name;
}
}
"""

HEAD = """
import ctypes, numpy as np
import caviar_amd
from caviar_amd import Engine, configs
fake = ctypes.CDLL(None)
fake.fake_launches.restype = ctypes.c_char_p
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
                       text=True, timeout=60)
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


def test_mixed_chunks_keep_their_length(runtime):
    """The mixed form sums 32-bit products over one chunk of atoms, so its
    chunks are no longer than an even deal of 512 workgroups of eight waves,
    nor than 4096 atoms: the last few row tiles of a group, and past a million
    atoms."""
    run(runtime, """
from caviar_amd import EwaldKSettings, System
for n, kmax, longest in ((30000, 13, 64), (100003, 13, 224), (30000, 16, 128), (2000000, 16, 4096),
                         (3000000, 6, 4096)):
    rng = np.random.default_rng(1)
    box = (n / 0.3) ** (1 / 3)
    s = System(lower=[0] * 3, upper=[box] * 3, bc=[1] * 3, ghost_cutoff=4.0, mass=[1.0], charge=[1.0],
               pos=rng.uniform(0, box, (n, 3)), vel=np.zeros((n, 3)), types=np.zeros(n, dtype=np.int32),
               ewald_k=EwaldKSettings.cube(0.9, kmax, 2.0))
    fake.fake_forget()
    e = Engine(s, precision="mixed")
    e.setup()
    grids = [l.split() for l in fake.fake_launches().decode().splitlines() if "k_sk_h" in l]
    assert len(grids) == 1, grids
    tiles = -(-(kmax + 1) * (2 * kmax + 1) // 16)
    chunks = int(grids[0][1]) // -(-tiles // 21)     # at least: the grid is rounded up by chunks of 8
    assert n / chunks <= longest, (n, kmax, n / chunks)
    e.close()
""")


@pytest.mark.parametrize("kmax,most", [(3, 484263), (16, 462549)])
def test_fixed_scratch_serves_the_same_systems(runtime, kmax, most):
    """The largest system of two types that cav_adjoint_noalloc takes."""
    run(runtime, f"""
from caviar_amd import CaviarError, EwaldKSettings, System
for n in ({most}, {most} + 1):
    s = System(lower=[0] * 3, upper=[100.0] * 3, bc=[1] * 3, ghost_cutoff=4.0, mass=[1.0, 1.0],
               charge=[1.0, -1.0], pos=np.zeros((n, 3)), vel=np.zeros((n, 3)),
               types=np.zeros(n, dtype=np.int32), ewald_k=EwaldKSettings.cube(0.9, {kmax}, 2.0))
    e = Engine(s)
    e.setup()
    try:
        e.adjoint_noalloc(np.zeros((n, 3)))
        assert n == {most}
    except CaviarError as err:
        assert n > {most} and err.code == 5
""")


def test_steps_that_do_not_run_are_an_error(runtime):
    """Queued steps whose kernels leave no trace end the call, not an endless
    repetition (here no kernel runs)."""
    run(runtime, SETUP + """
e = engine(0)
try:
    e.step(0.001, 3)
    assert False
except caviar_amd.CaviarError as err:
    assert err.code == 2
""")


def test_cell_buckets_grow_on_the_contexts_device(runtime):
    """Flags read back while another device is current: larger buckets are
    still the context's own device's."""
    run(runtime, SETUP + """
e = engine(0)
fake.fake_crowd(1000)
fake.fake_current(1)
n = ctypes.c_int()
assert lib.cav_num_ghosts(e.h, ctypes.byref(n)) == 0
assert fake.fake_malloc_device() == 0
""")
