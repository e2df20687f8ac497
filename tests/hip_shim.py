"""A library that stands between libmgcfd and the HIP runtime: loaded into the
global scope before libmgcfd, its definitions of a few calls are the ones that
libmgcfd binds to.  It can refuse allocations, and it can show the one device
as two, counting calls made while another than the chosen one is current.
Used by scripts that tests run in a process of their own."""
import ctypes as C
import os
import subprocess
import sys

SOURCE = r"""
#include <dlfcn.h>
#include <stddef.h>

static void* hip(const char* name)
{
    static void* h = dlopen("/opt/rocm/lib/libamdhip64.so", RTLD_NOW | RTLD_LOCAL);
    return dlsym(h, name);
}
#define REAL(name, ...) (reinterpret_cast<int (*)(__VA_ARGS__)>(hip(#name)))

struct Dim { unsigned x, y, z; };
static int refuse_device = 0, pinned_left = -1, devices = 0, expect = -1, misplaced = 0;
static thread_local int current = 0;
static long long shapes[4096][2];
static int n_shapes = 0, watch = 0;
static void placed() { if (expect >= 0 && current != expect) __atomic_add_fetch(&misplaced, 1, __ATOMIC_SEQ_CST); }

extern "C" {
// 1: device allocations fail
void shim_refuse_device(int on) { refuse_device = on; }
// pinned allocations that still succeed (-1: all)
void shim_pinned_left(int n) { pinned_left = n; }
// devices shown (0: as they are), and the one every call below has to be made on (-1: any)
void shim_devices(int n) { devices = n; }
void shim_expect(int d) { expect = d; }
int shim_misplaced(void) { return misplaced; }
// shapes of the launches made while watching: {workgroups, threads per workgroup} each, once
void shim_watch(int on) { watch = on; if (on) n_shapes = 0; }
int shim_shapes(long long* out)
{
    for (int i = 0; i < n_shapes; i++) { out[2 * i] = shapes[i][0]; out[2 * i + 1] = shapes[i][1]; }
    return n_shapes;
}

int hipMalloc(void** p, size_t n)
{
    placed();
    if (refuse_device) return 2;
    return REAL(hipMalloc, void**, size_t)(p, n);
}
int hipHostMalloc(void** p, size_t n, unsigned f)
{
    placed();
    if (pinned_left == 0) return 2;
    if (pinned_left > 0) pinned_left--;
    return REAL(hipHostMalloc, void**, size_t, unsigned)(p, n, f);
}
int hipLaunchKernel(const void* f, Dim g, Dim b, void** a, size_t l, void* s)
{
    placed();
    int i = 0;
    while (i < n_shapes && (shapes[i][0] != g.x || shapes[i][1] != b.x)) i++;
    if (watch && i == n_shapes && n_shapes < 4096) { shapes[i][0] = g.x; shapes[i][1] = b.x; n_shapes++; }
    return REAL(hipLaunchKernel, const void*, Dim, Dim, void**, size_t, void*)(f, g, b, a, l, s);
}
int hipGetDeviceCount(int* n)
{
    const int rc = REAL(hipGetDeviceCount, int*)(n);
    if (!rc && devices) *n = devices;
    return rc;
}
int hipSetDevice(int d)
{
    if (!devices) return REAL(hipSetDevice, int)(d);
    current = d;
    return REAL(hipSetDevice, int)(0);
}
int hipGetDevice(int* d)
{
    if (!devices) return REAL(hipGetDevice, int*)(d);
    *d = current;
    return 0;
}
int hipGetDevicePropertiesR0600(void* p, int d)
{
    return REAL(hipGetDevicePropertiesR0600, void*, int)(p, devices ? 0 : d);
}
}
"""


def build(folder) -> str:
    src, out = folder / "hip_shim.cpp", folder / "hip_shim.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-o", str(out), str(src), "-ldl"], check=True)
    return str(out)


def load(path) -> C.CDLL:
    return C.CDLL(path, mode=C.RTLD_GLOBAL)


def launch_shapes(shim, f) -> set:
    """The (workgroups, threads) of the kernels launched by f(); one thread at a time may launch."""
    shim.shim_watch(1)
    f()
    shim.shim_watch(0)
    out = (C.c_longlong * 8192)()
    n = shim.shim_shapes(out)
    return {(out[2 * i], out[2 * i + 1]) for i in range(n)}


def run_script(folder, body, **env) -> str:
    """body in a process of its own, with the shim loaded as 'shim' ahead of
    libmgcfd; it has to end by printing "ok".  Returns what it printed."""
    here = os.path.dirname(os.path.abspath(__file__))
    package = os.path.join(os.path.dirname(here), "mg-cfd-app-op2_amd")
    script = folder / "script.py"
    script.write_text(f"""
import sys
sys.path[:0] = {[here, package]!r}
import numpy as np
import hip_shim
shim = hip_shim.load({build(folder)!r})
""" + body)
    r = subprocess.run([sys.executable, "-u", str(script)], env=dict(os.environ, **env), capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.split()[-1] == "ok"
    return r.stdout
