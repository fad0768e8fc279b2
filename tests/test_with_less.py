"""ray-tracer_amd/csrc/with_less.hpp compiled on the host: a call that failed
for want of memory is made again while something can be given back, and any
other failure or success returns as it is."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "with_less.hpp"
int main() {
    // need: what the call takes; held: what can be given back, one part at a time
    int free_now, held, calls, lacked;
    auto run = [&](int need, int room, int parts, int other) {
        free_now = room; held = parts; calls = 0; lacked = 0;
        return rsh::with_less([&] { calls++; lacked = need > free_now; return lacked ? 2 : other; },
                              [&] { return lacked; },
                              [&] { if (!held) return false; held--; free_now += 10; return true; });
    };
    if (run(5, 10, 2, 0) != 0 || calls != 1 || held != 2) return 1;     // fits
    if (run(15, 10, 2, 0) != 0 || calls != 2 || held != 1) return 2;    // fits with one part less
    if (run(25, 10, 2, 0) != 0 || calls != 3 || held != 0) return 3;    // with both
    if (run(35, 10, 2, 0) != 2 || calls != 3 || held != 0) return 4;    // not at all: its own error
    if (run(5, 10, 2, 7) != 7 || calls != 1 || held != 2) return 5;     // another error
    if (run(15, 10, 2, 7) != 7 || calls != 2 || held != 1) return 6;    // another one after that
    return 0;
}
"""


def test_calls_short_of_memory_are_made_again(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "ray-tracer_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0
