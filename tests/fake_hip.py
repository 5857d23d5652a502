"""Host logic of libmset_amd.so without a device: runs a piece of Python in a child process in which
tests/fake_hip.cpp stands in for the HIP runtime (kernels are recorded, not run)."""
import os
import subprocess
import sys
import textwrap

from tests.conftest import ROOT

PRELUDE = '''
import ctypes as C
import sys
fake = C.CDLL(%(so)r, mode=C.RTLD_GLOBAL)
fake.fake_log.restype = fake.fake_kernels.restype = C.c_char_p
fake.fake_bytes.restype = fake.fake_peak.restype = C.c_size_t
fake.fake_fail_malloc.argtypes = fake.fake_device_memory.argtypes = [C.c_size_t]
fake.fake_occupancy.argtypes = [C.c_char_p, C.c_int]
sys.path.insert(0, %(root)r)
import numpy as np
from mset_amd import lib, physics


def launches(part=''):
    """(kernel, grid x, grid y, threads, captured) of every launch since the last fake_reset"""
    rows = [l.rsplit('|', 4) for l in fake.fake_log().decode().splitlines()]
    return [(r[0], int(r[1]), int(r[2]), int(r[3]), r[4] == '1') for r in rows if part in r[0]]


def state(n, nz, npos, seed=0, separable=True):
    rng = np.random.default_rng(seed)
    prop = physics.propagator(n, 0.5, physics.electron_wavelength(300e3), 1)
    if not separable:
        prop = prop * np.exp(0.5j * rng.uniform(-1, 1, (n, n)))
    return dict(V=rng.uniform(0, 1, (nz, n, n)).astype(np.float32), probe=np.ones((n, n), np.complex64), prop=prop,
                x=np.full(npos, n / 2, np.float32), y=np.full(npos, n / 2, np.float32),
                M=np.ones((npos, n, n), np.float32))


def upload(ctx, n, nz, npos, binning=1, steps=(1., 1., 1.), mode=0, **kw):
    s = state(n, nz, npos, **kw)
    ctx.upload(s['V'], s['probe'], s['prop'], s['x'], s['y'], s['M'], 1e-3, 0.5, slice_binning=binning, step_size=steps,
               grad_mode=mode)


def recon(n, nz, npos, steps=(1., 1., 1.), angles=(0., 30.)):
    """tilts of `npos` positions (a number, or one per tilt)"""
    per = [npos] * len(angles) if np.isscalar(npos) else list(npos)
    s = state(n, nz, 1)
    r = lib.Recon(s['V'], s['prop'], len(per), 1e-3, 0.5, step_size=steps)
    for j, k in enumerate(per):
        t = state(n, nz, k, seed=j)
        r.set_tilt(j, (0., angles[j], 0.), t['probe'] * (j + 1), t['x'] + j, t['y'] - j, t['M'])
    return r
'''

_BUILT = {}


def build(tmp):
    """the stand-in library, built once per test session"""
    if 'so' not in _BUILT:
        so = os.path.join(str(tmp), 'libfake_hip.so')
        rocm = os.environ.get('ROCM_PATH', '/opt/rocm')
        subprocess.run(['g++', '-std=c++17', '-O1', '-w', '-shared', '-fPIC', '-I' + os.path.join(rocm, 'include'),
                        os.path.join(ROOT, 'tests', 'fake_hip.cpp'), '-o', so], check=True)
        _BUILT['so'] = so
    return _BUILT['so']


def run(tmp, body):
    """Runs `body` after PRELUDE in a child process; its assertion or crash fails the test."""
    code = PRELUDE % dict(so=build(tmp), root=ROOT) + textwrap.dedent(body)
    r = subprocess.run([sys.executable, '-c', code], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
    return r.stdout


FAIL_SOURCE = '''
#include <dlfcn.h>
#include <stddef.h>
static size_t size;
static int count;
void fail_malloc(size_t n) { size = n; }
int failed(void) { return count; }
int hipMalloc(void** p, size_t n) {
    static int (*real)(void**, size_t);
    if (!real) real = (int (*)(void**, size_t))dlsym(dlopen("libamdhip64.so.7", RTLD_NOW), "hipMalloc");
    if (size && n == size) {
        *p = 0;
        ++count;
        return 2;            /* hipErrorOutOfMemory */
    }
    return real(p, n);
}
'''

FAIL_PRELUDE = '''
import ctypes as C
import sys
shim = C.CDLL(%(so)r, mode=C.RTLD_GLOBAL)
shim.fail_malloc.argtypes = [C.c_size_t]
fail_malloc, failed = shim.fail_malloc, shim.failed
sys.path.insert(0, %(root)r)
import numpy as np
from mset_amd import lib
'''


def run_failing_malloc(tmp, body):
    """Runs `body` in a child process on the real runtime, where device allocations of exactly fail_malloc(n) bytes
    report that the device is out of memory; failed() counts them."""
    so, c = os.path.join(str(tmp), 'libfail_malloc.so'), os.path.join(str(tmp), 'fail_malloc.c')
    with open(c, 'w') as fh:
        fh.write(FAIL_SOURCE)
    subprocess.run(['gcc', '-O1', '-shared', '-fPIC', c, '-o', so, '-ldl'], check=True)
    code = FAIL_PRELUDE % dict(so=so, root=ROOT) + textwrap.dedent(body)
    r = subprocess.run([sys.executable, '-c', code], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
