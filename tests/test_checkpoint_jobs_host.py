"""The checkpointing pass's host jobs (csrc/checkpoint_jobs.h, no GPU): every
asked job once, in layer order with a layer's hash first, and every thread in
use whichever kinds are asked for. The jobs of the first `threads` calls wait
for one another, so a thread that never gets one fails the run."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "iris_amd", "csrc")

PROGRAM = r"""
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include "checkpoint_jobs.h"

int main(int, char** v) {
    const uint32_t layers = atoi(v[1]), threads = atoi(v[4]);
    const bool hashes = atoi(v[2]), rows = atoi(v[3]);
    const uint32_t jobs = layers * (hashes + rows), together = std::min(jobs, threads);
    std::mutex m;
    std::condition_variable all;
    uint32_t at = 0;
    bool late = false;
    run_checkpoint_jobs(layers, hashes, rows, threads, [&](uint32_t layer, bool hash) {
        std::unique_lock<std::mutex> l(m);
        printf("%u %d\n", layer, (int)hash);
        at++;
        all.notify_all();
        late |= !all.wait_for(l, std::chrono::seconds(10), [&] { return at >= together || late; });
    });
    return late;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("jobs")
    src, exe = d / "jobs.cpp", d / "jobs"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O1", "-pthread", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True)
    return str(exe)


@pytest.mark.parametrize("threads", [1, 3, 8, 16])
@pytest.mark.parametrize("hashes,rows", [(1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("layers", [1, 2, 32])
def test_every_thread_gets_work(program, layers, hashes, rows, threads):
    r = subprocess.run([program, str(layers), str(hashes), str(rows), str(threads)], capture_output=True, text=True,
                       timeout=60)
    assert r.returncode == 0, r.stdout
    got = [tuple(map(int, line.split())) for line in r.stdout.splitlines()]
    want = [(layer, kind) for layer in range(layers) for kind in (1, 0) if (hashes if kind else rows)]
    assert sorted(got) == sorted(want)
    if threads == 1:
        assert got == want
