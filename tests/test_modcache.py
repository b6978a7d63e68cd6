"""The store of compiled modules (matjes_amd/csrc/mj_modcache.h) on the host, with
counters in a module's place (the same source serves the library)."""
import ctypes
import os
import subprocess

from conftest import REPO

SRC = r'''
#include <atomic>
#include <thread>
#include <vector>
#include "mj_modcache.h"
static std::atomic<int> loads{0}, live{0};
struct Mod {
    int id;
    Mod() : id(++loads) { ++live; }
    ~Mod() { --live; }
};
static ModCache<Mod> cache(3);
static std::vector<std::shared_ptr<Mod>> held;
static int get_mod(int device, const std::string &src, int fail, std::shared_ptr<Mod> *m)
{
    return cache.get(device, src, m, [&](std::shared_ptr<Mod> *out) {
        if (fail) return 7;
        *out = std::make_shared<Mod>();
        return 0;
    });
}
extern "C" int get(int device, const char *src, int fail)
{
    std::shared_ptr<Mod> m;
    return get_mod(device, src, fail, &m) ? -1 : m->id;
}
extern "C" int hold(int device, const char *src)
{
    held.emplace_back();
    return get_mod(device, src, 0, &held.back()) ? -1 : held.back()->id;
}
extern "C" void release() { held.clear(); }
extern "C" int alive() { return live; }
extern "C" int kept() { long long a, b; cache.stats(&a, &b); return (int)b; }
extern "C" int made() { long long a, b; cache.stats(&a, &b); return (int)a; }
// n threads asking in turn for a few sources each, holding one at a time: wrong answers
extern "C" int race(int n)
{
    std::atomic<int> bad{0};
    std::vector<std::thread> t;
    for (int k = 0; k < n; ++k)
        t.emplace_back([&, k] {
            std::shared_ptr<Mod> a, b;
            for (int i = 0; i < 2000; ++i) {
                const std::string s(1, (char)('a' + (i * 7 + k) % 6));
                if (get_mod(0, s, 0, &a) || get_mod(0, s, 0, &b) || !a || !b) ++bad;
            }
        });
    for (auto &x : t) x.join();
    return bad;
}
'''


def _lib(tmp_path):
    cpp = tmp_path / "m.cpp"
    cpp.write_text(SRC)
    so = tmp_path / "m.so"
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-pthread", "-I",
                           os.path.join(REPO, "matjes_amd", "csrc"), str(cpp), "-o", str(so)])
    return ctypes.CDLL(str(so))


def test_a_module_per_device_and_source(tmp_path):
    L = _lib(tmp_path)
    a0, a1, b0 = L.get(0, b"a", 0), L.get(1, b"a", 0), L.get(0, b"b", 0)
    assert len({a0, a1, b0}) == 3                      # the same source on another device is another module
    assert [L.get(0, b"a", 0), L.get(1, b"a", 0), L.get(0, b"b", 0)] == [a0, a1, b0]
    assert L.get(1, b"b", 1) == -1                     # a failure is not kept
    assert L.get(1, b"b", 0) not in (-1, b0)


def test_modules_are_given_back(tmp_path):
    L = _lib(tmp_path)
    a = L.hold(0, b"a")
    others = [L.get(0, s, 0) for s in (b"b", b"c")]
    assert L.get(0, b"a", 0) == a and L.alive() == 3   # three are kept
    assert L.get(0, b"d", 0) and L.kept() == 3 and L.alive() == 3   # b, the longest unasked, is unloaded
    assert L.get(0, b"c", 0) == others[1] and L.get(0, b"b", 0) not in others
    for s in (b"e", b"f", b"g"):
        L.get(0, s, 0)
    assert L.kept() == 3 and L.alive() == 4            # a is held by its object only
    L.release()
    assert L.alive() == 3                              # and unloaded with it
    assert L.get(0, b"a", 0) != a and L.made() == 9


def test_threads(tmp_path):
    L = _lib(tmp_path)
    assert L.race(8) == 0
    assert L.kept() == 3 and L.alive() == 3
