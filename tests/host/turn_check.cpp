// The turns of gh_turn.h on threads: each in its turn adds to plain memory that all share, as
// the wavefronts of k_direct_f64_ring add to the sums of their targets.  Built with
// ThreadSanitizer, which reports any access that the turns do not order.
#include <cstdio>
#include <thread>
#include <vector>

#include "../../gravhopper_amd/csrc/gh_turn.h"

int main()
{
    constexpr int kWorkers = 4, kTurns = 400, kSums = 64;
    int turn = 0;
    double sums[kSums] = {};
    auto work = [&](int w) {
        for (int g = w; g < kTurns; g += kWorkers) {
            while (!gh::turn_is(&turn, g)) std::this_thread::yield();
            for (int k = 0; k < kSums; k++) sums[k] = 0.5 * sums[k] + g;
            gh::turn_pass(&turn, g + 1);
        }
    };
    std::vector<std::thread> workers;
    for (int w = 0; w < kWorkers; w++) workers.emplace_back(work, w);
    for (std::thread& t : workers) t.join();
    double want = 0.0;
    for (int g = 0; g < kTurns; g++) want = 0.5 * want + g;
    int wrong = 0;
    for (double s : sums) wrong += s != want;
    printf("%d wrong\n", wrong);
    return wrong != 0;
}
