"""The threads that copy host memory, without a GPU: tasks and groups, and what
a forked process does with the pool it inherits."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "hybridhsdla_amd" / "csrc"

PROGRAM = r"""
#include "hostpool.h"

#include <sys/wait.h>
#include <unistd.h>

#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>

using hsgen::HostPool;

int main()
{
    HostPool* pool = new HostPool;
    if (pool->size() == 0) return 3;
    std::atomic<int> ran{0};
    int a, b;
    pool->post(&a, [&] { ++ran; }, 5);
    while (ran.load() < 5) std::this_thread::yield();
    // finish() waits for what runs and withdraws what waits
    std::atomic<bool> go{false};
    std::atomic<int> begun{0}, ended{0};
    pool->post(&b, [&] { ++begun; while (!go.load()) std::this_thread::yield(); ++ended; }, 100);
    while (begun.load() < (int)pool->size()) std::this_thread::yield();
    std::thread opener([&] { std::this_thread::sleep_for(std::chrono::milliseconds(50)); go = true; });
    pool->finish(&a);
    pool->finish(&b);
    if (begun.load() != ended.load()) return 4;
    opener.join();
    std::this_thread::sleep_for(std::chrono::milliseconds(200));    // every thread sleeps again
    const pid_t child = fork();
    if (child == 0) {
        alarm(10);                       // ends a child that waits for threads it has not
        delete pool;
        _exit(0);
    }
    int status = 0;
    if (waitpid(child, &status, 0) != child || !WIFEXITED(status) || WEXITSTATUS(status)) return 5;
    pool->post(&a, [&] { ++ran; }, 1);   // the parent's threads work on
    while (ran.load() < 6) std::this_thread::yield();
    delete pool;
    std::puts("ok");
    return 0;
}
"""


def test_tasks_groups_and_a_forked_process(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not installed")
    src = tmp_path / "pool.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "pool"
    subprocess.run([cxx, "-std=c++17", "-O1", "-pthread", "-I", str(CSRC), str(src), str(CSRC / "hostpool.cpp"), "-o",
                    str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0 and res.stdout.strip() == "ok", res.returncode
