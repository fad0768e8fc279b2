"""ray-tracer_amd/csrc/host_words.hpp compiled on the host with runtime calls
that fail: page-locked words are kept only together with their device address,
so that no later call hands a kernel a null one."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "host_words.hpp"
int main() {
    int held = 0, fail_alloc = 0, fail_address = 0, calls = 0;
    auto alloc = [&](void** p, size_t n) { calls++; if (fail_alloc) return 2; *p = std::malloc(n); std::memset(*p, 7, n); held++; return 0; };
    auto address = [&](void** d, void* p) { if (fail_address) return 3; *d = (char*)p + 4096; return 0; };
    auto release = [&](void* p) { std::free(p); held--; return 0; };
    rsh::HostWords w;
    auto get = [&]() { return rsh::acquire_words(w, 64, alloc, address, release); };
    auto none = [&]() { return !w.host && !w.dev && held == 0; };
    fail_address = 1;
    if (get() != 3 || !none()) return 1;
    if (get() != 3 || !none()) return 2;         // and again: no half of it was kept
    fail_address = 0; fail_alloc = 1;
    if (get() != 2 || !none()) return 3;
    fail_alloc = 0;
    if (get() != 0 || !w.host || (char*)w.dev != (char*)w.host + 4096 || held != 1) return 4;
    for (int i = 0; i < 16; i++) if (w.host[i]) return 5;
    calls = 0;
    if (get() != 0 || calls != 0) return 6;      // kept
    return 0;
}
"""


def test_words_without_a_device_address_are_given_back(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "ray-tracer_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0
