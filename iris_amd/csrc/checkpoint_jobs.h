// The host side of a checkpointing pass as jobs: per layer its hash and its
// rows' copy to the caller, those of them that were asked for. Host code only.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <thread>
#include <vector>

// Runs job(layer, hash) for every layer: hash = true where `hashes`, false
// (its rows) where `rows`. At most `most` threads take the jobs in turn, in
// layer order and a layer's hash before its rows, so that whatever mix of
// kinds is left keeps every thread busy. (Dealt round by round to an even
// number of threads, half of them never had a hash, and with one kind asked
// for half had nothing at all: 2048 rows of 4096 through 32 layers, 16
// threads, hashes only 67 -> 52 ms, with rows 65 -> 52; 8 threads with rows
// 91 -> 79.)
template <class Job>
void run_checkpoint_jobs(uint32_t layers, bool hashes, bool rows, uint32_t most, Job&& job) {
    const uint32_t kinds = (uint32_t)hashes + (uint32_t)rows, jobs = kinds * layers;
    std::atomic<uint32_t> next{0};
    std::vector<std::thread> pool;
    for (uint32_t t = 0; t < std::min(jobs, std::max(1u, most)); t++)
        pool.emplace_back([&] {
            for (uint32_t j; (j = next++) < jobs;) job(j / kinds, kinds == 2 ? j % 2 == 0 : hashes);
        });
    for (auto& th : pool) th.join();
}
