// Host check of how many threads a field transfer takes
// (mr-lbm_amd/csrc/transfer.h): no more than there are free processors, also
// while threads of this program spin on all of them. Prints "ok" and exits
// 0 on success.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>

#include "../mr-lbm_amd/csrc/transfer.h"

using namespace mrlbm;

int main() {
    int failures = 0;
    auto expect = [&](int line, int got, int want) {
        if (got == want) return;
        failures++;
        std::printf("line %d: %d workers, not %d\n", line, got, want);
    };
    // free processors: a worker per three chunks, at most eight
    expect(__LINE__, transfer_workers(0, 16, 1, 1), 1);
    expect(__LINE__, transfer_workers(5, 16, 1, 1), 1);
    expect(__LINE__, transfer_workers(6, 16, 1, 1), 2);
    expect(__LINE__, transfer_workers(20, 16, 1, 1), 6);
    expect(__LINE__, transfer_workers(400, 16, 1, 1), 8);
    expect(__LINE__, transfer_workers(400, 4, 1, 1), 4);
    expect(__LINE__, transfer_workers(400, 16, 13, 1), 4);
    // a pool that spins on all of them: the caller alone
    expect(__LINE__, transfer_workers(20, 16, 16, 1), 1);
    expect(__LINE__, transfer_workers(400, 16, 40, 1), 1);
    expect(__LINE__, transfer_workers(400, 16, ~0u, 1), 1);
    expect(__LINE__, transfer_workers(400, 1, 1, 1), 1);
    expect(__LINE__, transfer_workers(400, 0, 1, 1), 1);
    // once it sleeps, more join those that are there; none is sent away
    expect(__LINE__, transfer_workers(400, 16, 3, 3), 8);
    expect(__LINE__, transfer_workers(400, 16, 14, 3), 5);
    expect(__LINE__, transfer_workers(400, 16, 30, 3), 3);
    expect(__LINE__, transfer_workers(3, 16, 3, 3), 3);

    const unsigned cpus = std::thread::hardware_concurrency();
    std::atomic<bool> stop{false};
    std::vector<std::thread> th;
    for (unsigned k = 0; k < cpus; k++) th.emplace_back([&] { while (!stop) {} });
    std::this_thread::sleep_for(std::chrono::milliseconds(50));
    expect(__LINE__, transfer_workers(400, cpus, running_threads(), 1), 1);
    stop = true;
    for (auto& t : th) t.join();
    if (failures) return 1;
    std::printf("ok\n");
    return 0;
}
