"""A HIP runtime for CPU tests of the library's host code: the calls that
libdsv4_gpu.so makes to bring itself up and to launch, replaced by ones that
allocate host memory and launch nothing. A launch can be made to fail, and the
first eight kernels and the second launch's second argument are kept. `run`
starts a child process with it in place; the child sees no device, so nothing
runs on a GPU wherever the test does. In the child `shim` is this library and
`L` the backend."""
import os
import shutil
import subprocess
import sys

import pytest

import common

SOURCE = r"""
#include <stdlib.h>
#include <string.h>
typedef struct { unsigned x, y, z; } D3;
static int launches, fail_at = -1, last, frees, capturing;
static void *arg1;
static const void *ran[8];
static struct { const void *f; const char *name; } *kernels;
static int n_kernels;
/* launch number `at` of the next call fails (-1: none); its stream is or is
 * not being captured */
void shim_reset(int at, int cap) { launches = 0; last = 0; arg1 = NULL; fail_at = at; capturing = cap; }
int shim_launches(void) { return launches; }
int shim_frees(void) { return frees; }
void *shim_arg1(void) { return arg1; }
/* the mangled name of the call's kernel number k */
const char *shim_kernel(int k)
{
    for (int i = 0; i < n_kernels; i++)
        if (k < launches && k < 8 && kernels[i].f == ran[k]) return kernels[i].name;
    return "";
}
void __hipRegisterFunction(void **m, const void *f, char *d, const char *name, unsigned t, void *a,
                           void *b, void *c, void *e, int *w)
{
    (void)m; (void)d; (void)t; (void)a; (void)b; (void)c; (void)e; (void)w;
    if ((n_kernels & 255) == 0)
        kernels = realloc(kernels, (n_kernels + 256) * sizeof *kernels);
    kernels[n_kernels].f = f;
    kernels[n_kernels++].name = strdup(name);
}
int hipLaunchKernel(const void *f, D3 g, D3 b, void **a, size_t l, void *s)
{
    (void)g; (void)b; (void)l; (void)s;
    if (launches < 8) ran[launches] = f;
    if (launches == 1) arg1 = *(void **)a[1];
    if (launches++ == fail_at) { last = 719; return 719; }
    return 0;
}
int hipGetLastError(void) { const int e = last; last = 0; return e; }
int __hipPushCallConfiguration(D3 g, D3 b, size_t l, void *s)
{
    (void)g; (void)b; (void)l; (void)s;
    return 0;
}
int __hipPopCallConfiguration(D3 *g, D3 *b, size_t *l, void **s)
{
    const D3 one = {1, 1, 1};
    *g = *b = one; *l = 0; *s = NULL;
    return 0;
}
int hipGetDeviceCount(int *n) { *n = 1; return 0; }
int hipSetDevice(int d) { (void)d; return 0; }
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipMemGetInfo(size_t *f, size_t *t) { *f = *t = 0; return 0; }
int hipStreamCreateWithFlags(void **s, unsigned fl) { (void)fl; *s = &launches; return 0; }
int hipGetSymbolAddress(void **p, const void *sym) { (void)sym; *p = &launches; return 0; }
int hipDeviceSynchronize(void) { return 0; }
int hipMalloc(void **p, size_t n) { *p = malloc(n); return *p ? 0 : 2; }
int hipMemset(void *p, int v, size_t n) { memset(p, v, n); return 0; }
int hipFree(void *p) { (void)p; frees++; return 0; }
int hipHostMalloc(void **p, size_t n, unsigned fl) { (void)fl; *p = malloc(n); return *p ? 0 : 2; }
int hipHostGetDevicePointer(void **d, void *h, unsigned fl) { (void)fl; *d = h; return 0; }
int hipMemcpy(void *d, const void *s, size_t n, int k) { (void)k; memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st)
{
    (void)k; (void)st;
    memcpy(d, s, n);
    return 0;
}
int hipStreamSynchronize(void *st) { (void)st; return 0; }
int hipStreamIsCapturing(void *s, int *st) { (void)s; *st = capturing; return 0; }
int hipDeviceGetAttribute(int *v, int attr, int d)
{
    (void)d;
    *v = attr == ATTR_CU ? 256 : 163840;         /* 256 CUs, 160 KB of LDS */
    return 0;
}
int hipFuncGetAttributes(void *a, const void *f) { (void)a; (void)f; return 1; }
int hipFuncSetAttribute(const void *f, int at, int v) { (void)f; (void)at; (void)v; return 0; }
int hipGetDevicePropertiesR0600(void *p, int d) { (void)d; memset(p, 0, PROP); return 0; }
"""

# before torch and the backend, whose calls then find it first
PRELUDE = r"""
import ctypes
import sys
import numpy as np
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
shim.shim_arg1.restype = ctypes.c_void_p
shim.shim_kernel.restype = ctypes.c_char_p
import common
D = common.load_pkg()
L = D.lib()
"""

_CU = r"""
#include <hip/hip_runtime_api.h>
#include <cstdio>
static_assert(sizeof(hipDeviceAttribute_t) == sizeof(int), "");
int main()
{
    printf("-DATTR_CU=%d -DPROP=%d", (int)hipDeviceAttributeMultiprocessorCount,
           (int)sizeof(hipDeviceProp_t));
}
"""


def run(tmp_path, child, env=None):
    """The child's standard output, its exit status checked."""
    hip = "/opt/rocm/include"
    if not (shutil.which("gcc") and shutil.which("g++") and os.path.isdir(hip)):
        pytest.skip("no compiler or no HIP headers")
    cu, exe, src, lib = (str(tmp_path / n) for n in ("cu.cpp", "cu", "shim.c", "shim.so"))
    with open(cu, "w") as f:
        f.write(_CU)
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run(["g++", "-D__HIP_PLATFORM_AMD__", "-w", "-I", hip, cu, "-o", exe], check=True)
    defs = subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split()
    subprocess.run(["gcc", "-shared", "-fPIC", "-Wall", "-Werror"] + defs + [src, "-o", lib], check=True)
    e = dict(os.environ, HIP_VISIBLE_DEVICES="-1", **(env or {}))
    e["PYTHONPATH"] = os.pathsep.join([os.path.join(common.ROOT, "tests"), common.ROOT,
                                       e.get("PYTHONPATH", "")])
    r = subprocess.run([sys.executable, "-c", PRELUDE + child, lib], env=e, capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
