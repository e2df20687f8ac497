"""A library that stands between libmgcfd and the HIP runtime: loaded into the
global scope before libmgcfd, its definitions of a few calls are the ones that
libmgcfd binds to.  It can refuse allocations, and it can show the one device
as two, counting calls made while another than the chosen one is current.
Used by scripts that tests run in a process of their own."""
import ctypes as C
import subprocess

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
