"""The store of compiled modules (matjes_amd/csrc/mj_modcache.h) on the host, with
counters in a module's place (the same source serves the library)."""
import ctypes
import os
import subprocess

from conftest import REPO

SRC = r'''
#include "mj_modcache.h"
static int loads = 0;
static ModCache<int> cache;
extern "C" int get(int device, const char *src, int fail)
{
    int m = -1;
    if (cache.get(device, src, &m, [&](int *out) { if (fail) return 7; *out = ++loads; return 0; })) return -1;
    return m;
}
'''


def _lib(tmp_path):
    cpp = tmp_path / "m.cpp"
    cpp.write_text(SRC)
    so = tmp_path / "m.so"
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-I",
                           os.path.join(REPO, "matjes_amd", "csrc"), str(cpp), "-o", str(so)])
    return ctypes.CDLL(str(so))


def test_a_module_per_device_and_source(tmp_path):
    L = _lib(tmp_path)
    a0, a1, b0 = L.get(0, b"a", 0), L.get(1, b"a", 0), L.get(0, b"b", 0)
    assert len({a0, a1, b0}) == 3                      # the same source on another device is another module
    assert [L.get(0, b"a", 0), L.get(1, b"a", 0), L.get(0, b"b", 0)] == [a0, a1, b0]
    assert L.get(1, b"b", 1) == -1                     # a failure is not kept
    assert L.get(1, b"b", 0) not in (-1, b0)
