"""Child processes whose library allocates device memory through a probe: every
new block filled with 0xFF bytes (a NaN as FP64, -1 as int), so that a value read
before it is written shows, allocations refused from a chosen one on, or a device of
little room.

The probe defines hipMalloc and hipFree itself and is loaded with global symbols
before the library, whose calls then go through it."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_SOURCE = r"""
#include <cstddef>
#include <dlfcn.h>
#include <map>
namespace {
long calls = 0, limit = -1;  // limit < 0: no call is refused
long live = 0, room = -1;    // bytes; room < 0: the device's own
std::map<void*, size_t> size;
bool fill = false;
template <typename F> F real(const char* name) {
  static void* hip = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
  return reinterpret_cast<F>(dlsym(hip, name));
}
}
extern "C" {
int hipMalloc(void** p, size_t n) {
  if ((limit >= 0 && calls >= limit) || (room >= 0 && live + (long)n > room)) return 2;  // hipErrorOutOfMemory
  ++calls;
  const int e = real<int (*)(void**, size_t)>("hipMalloc")(p, n);
  if (!e) live += size[*p] = n;
  if (e || !fill) return e;
  const int f = real<int (*)(void*, int, size_t)>("hipMemset")(*p, 0xFF, n);
  return f ? f : real<int (*)()>("hipDeviceSynchronize")();
}
int hipFree(void* p) {
  live -= size[p];
  size.erase(p);
  return real<int (*)(void*)>("hipFree")(p);
}
void probe_fill(int on) { fill = on; }
void probe_limit(long n) { calls = 0; limit = n; }  // n more calls succeed; < 0: all
void probe_room(long bytes) { room = bytes; }
long probe_live() { return live; }
}
"""

_PREAMBLE = """
import ctypes, os, sys
sys.path[:0] = [%r, %r]
import torch
probe = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)
probe.probe_limit.argtypes = [ctypes.c_long]
probe.probe_room.argtypes = [ctypes.c_long]
probe.probe_live.restype = ctypes.c_long
import numpy as np
from dftcxx_amd import gridlib as G
from dftcxx_amd import molecule as M
from systems import random_density
"""


def run(tmp_path, code, timeout=100):
    """Runs code after the preamble above in a child; its output, after checking its status."""
    src, so = tmp_path / "probe.cpp", tmp_path / "probe.so"
    src.write_text(_SOURCE)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", str(src), "-o", str(so), "-ldl"], check=True)
    head = _PREAMBLE % (ROOT, os.path.join(ROOT, "tests"), str(so))
    r = subprocess.run([sys.executable, "-u", "-c", head + code], capture_output=True, text=True, timeout=timeout)
    print(r.stdout, r.stderr[-2000:], flush=True)
    assert r.returncode == 0
    return r.stdout
