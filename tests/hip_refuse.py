"""Runs a test body in a child process in which chosen HIP runtime calls are
refused: a small library, loaded before libgeauxdock_amd.so, stands in for them
and hands the others on.  Nothing that is refused reaches the device."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
#include <string.h>
typedef struct { unsigned x, y, z; } dim;
static long g_pass = -1;                 /* launches of the stepping kernel until one is refused (-1: none is) */
static const void *g_step;               /* the stepping kernel's host function */
static size_t g_host = (size_t)-1, g_dev = (size_t)-1;  /* most bytes of a pinned / device allocation */
static int g_err, g_n_host, g_n_dev;
void refuse_stepping_after(long n) { g_pass = n; }
void refuse_pinned_over(size_t n) { g_host = n; g_n_host = 0; }
void refuse_device_over(size_t n) { g_dev = n; g_n_dev = 0; }
int refused_pinned(void) { return g_n_host; }
int refused_device(void) { return g_n_dev; }
static void *real(const char *name) {
  static void *h;
  if (!h) h = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
  return h ? dlsym(h, name) : 0;
}
void __hipRegisterFunction(void *m, const void *host, char *device, const char *name, unsigned n, void *tid, void *bid,
                           dim *block, dim *grid, int *size) {
  typedef void (*fn)(void *, const void *, char *, const char *, unsigned, void *, void *, dim *, dim *, int *);
  if (strstr(name, "gd_chain_kernel")) g_step = host;
  ((fn)real("__hipRegisterFunction"))(m, host, device, name, n, tid, bid, block, grid, size);
}
int hipLaunchKernel(const void *f, dim grid, dim block, void **args, size_t lds, void *s) {
  static int (*r)(const void *, dim, dim, void **, size_t, void *);
  if (f == g_step && g_pass == 0) { g_pass = -1; return g_err = 9; }
  if (f == g_step && g_pass > 0) --g_pass;
  if (!r) r = (int (*)(const void *, dim, dim, void **, size_t, void *))real("hipLaunchKernel");
  return r(f, grid, block, args, lds, s);
}
int hipGetLastError(void) {
  static int (*r)(void);
  if (g_err) { const int e = g_err; g_err = 0; return e; }
  if (!r) r = (int (*)(void))real("hipGetLastError");
  return r();
}
int hipHostMalloc(void **p, size_t n, unsigned flags) {
  static int (*r)(void **, size_t, unsigned);
  if (n > g_host) { ++g_n_host; return g_err = 2; }
  if (!r) r = (int (*)(void **, size_t, unsigned))real("hipHostMalloc");
  return r(p, n, flags);
}
int hipMalloc(void **p, size_t n) {
  static int (*r)(void **, size_t);
  if (n > g_dev) { ++g_n_dev; return g_err = 2; }
  if (!r) r = (int (*)(void **, size_t))real("hipMalloc");
  return r(p, n);
}
"""

HEAD = """
import ctypes as C, sys
import numpy as np
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
shim.refuse_stepping_after.argtypes = [C.c_long]
shim.refuse_pinned_over.argtypes = [C.c_size_t]
shim.refuse_device_over.argtypes = [C.c_size_t]
NONE = 2 ** 64 - 1
import geauxdock_amd as g
from geauxdock_amd import abi
FIELDS = ("energy", "movematrix", "idx_tmp", "n_accept", "n_exchange", "best_energy", "is_accept", "n_swap_lig",
          "n_swap_prt")
def same(a, b):
    for f in FIELDS:
        assert np.array_equal(getattr(a, f), getattr(b, f)), f
ene = g.load_enepara()
"""


def run(tmp_path, body, timeout=100):
    """The body (Python source, after HEAD) in a child process."""
    src, lib = os.path.join(tmp_path, "refuse.c"), os.path.join(tmp_path, "refuse.so")
    with open(src, "w") as f:
        f.write(SHIM)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", src, "-o", lib, "-ldl"], check=True)
    r = subprocess.run([sys.executable, "-u", "-c", HEAD + body, lib], cwd=ROOT, capture_output=True, text=True,
                       timeout=timeout)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
