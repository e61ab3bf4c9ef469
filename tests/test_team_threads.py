"""The helper threads of the host copies (csrc/team.h), as a host program without a device: threads
that open, use and close it, with last closes that overlap another thread's open and close."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "team.h"
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>

int main(int argc, char **argv) {
    const int pause = std::atoi(argv[1]), rounds = std::atoi(argv[2]);
    pasc::Team team;
    std::atomic<long> ran{0};
    std::atomic<int> cycle{0};
    std::atomic<bool> over{false};
    const std::function<void()> work = [&] { ran++; };
    // one thread opens, uses and closes a team; the other opens and closes without using it, so
    // that either of them may be the last to close while the other comes and goes
    std::thread other([&] {
        while (!over) {
            team.open();
            if (pause) std::this_thread::sleep_for(std::chrono::microseconds(pause));
            team.close();
            while (cycle == 0 && !over) std::this_thread::yield();
            cycle--;
        }
    });
    for (int i = 0; i < rounds; i++) {
        team.open();
        team.run(pasc::Team::MOST, work);
        cycle = 2;
        team.close();
    }
    over = true;
    other.join();
    // every run is done at least by its caller, and the team works after all of it
    if (ran < rounds) return 1;
    team.open();
    std::atomic<int> n{0};
    team.run(pasc::Team::MOST, [&] { n++; });
    team.close();
    std::printf("%ld runs, %d at the end\n", (long)ran, (int)n);
    return n >= 1 ? 0 : 2;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("team")
    src, exe = d / "team.cpp", d / "team"
    src.write_text(PROGRAM)
    inc = os.path.join(ROOT, "pasc_inference_amd", "csrc")
    r = subprocess.run([shutil.which("g++") or "g++", "-std=c++17", "-O1", "-pthread", "-I", inc,
                        str(src), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return str(exe)


@pytest.mark.parametrize("pause_us", [0, 20, 50])
def test_overlapping_closes_end(program, pause_us):
    # 3000 rounds take under a second; a closer that waits for good ends with the time limit
    r = subprocess.run([program, str(pause_us), "3000"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
