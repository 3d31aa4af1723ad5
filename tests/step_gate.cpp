// Exerciser of csrc/step_gate.h, built and run by tests/test_step_gate.py: eight threads count a counter of one to
// eight down at once, as threads do whose steps go layer by layer for a while.  Exactly as many of them as it
// says may find something left, and it ends at zero.
#include <cstdio>
#include <thread>
#include <vector>

#include "../wayruntime_amd/csrc/step_gate.h"

int main()
{
    constexpr int kThreads = 8, kRounds = 20000;
    std::atomic<uint32_t> n{0}, taken{0}, done{0};
    std::atomic<int> round{-1};
    std::vector<std::thread> threads;
    for (int t = 0; t < kThreads; t++)
        threads.emplace_back([&] {
            for (int r = 0; r < kRounds; r++) {
                while (round.load() < r) std::this_thread::yield();
                if (wr::count_down(n)) taken++;
                done++;
            }
        });
    int wrong = 0;
    for (int r = 0; r < kRounds; r++) {
        const uint32_t from = 1 + r % 8;
        n = from;
        taken = 0;
        done = 0;
        round = r;
        while (done.load() < kThreads) std::this_thread::yield();
        if (n.load() != 0 || taken.load() != from) wrong++;
    }
    for (auto& t : threads) t.join();
    std::printf("wrong %d\n", wrong);
    return wrong != 0;
}
