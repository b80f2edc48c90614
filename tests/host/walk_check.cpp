// walk_shares (pixienn_amd/csrc/grouped.h) on the host: a workgroup of two waves, only one of which runs at a time, in every
// order that the barriers leave open.  Whatever the order, the waves have to be given the same numbers.
#include "../../pixienn_amd/csrc/grouped.h"

#include <condition_variable>
#include <cstdio>
#include <mutex>
#include <thread>
#include <vector>

namespace {

// Runs one wave up to a barrier or its end, then the other; `first` says, a bit per phase, which of them goes first.
struct Workgroup {
    unsigned first;
    uint32_t word = 0, counter = 0;
    std::mutex mutex;
    std::condition_variable turn;
    int running = -1, phase = 0, arrived = 0;
    bool ended[2] = {}, mismatch = false;

    int leader() const { return first >> (phase % 10) & 1; }
    void wait_turn(std::unique_lock<std::mutex>& lock, int wave) { turn.wait(lock, [&] { return running == wave; }); }
    void arrive(int wave, bool end)
    {
        std::unique_lock<std::mutex> lock(mutex);
        ended[wave] = end;
        ++arrived;
        if (arrived == 2) {      // both are at the barrier, or both at their end
            if (ended[0] != ended[1]) mismatch = true;
            arrived = mismatch ? 1 : 0;
            ++phase;
            running = mismatch ? (ended[0] ? 1 : 0) : leader();
        } else {
            running = 1 - wave;
        }
        turn.notify_all();
        if (!end) wait_turn(lock, wave);
    }
};

struct Wave {
    Workgroup& group;
    int id;
    void sync() const { group.arrive(id, false); }
    void ask() const { if (id == 0) group.word = group.counter++; }
    uint32_t next() const { return group.word; }
};

}  // namespace

int main()
{
    constexpr uint32_t kAll = 7;
    int bad = 0, runs = 0;
    // which shares ask by themselves, as those that form sums do; the others leave that to the walk
    for (uint32_t asking = 0; asking < 1u << kAll; asking += 5)
        for (unsigned first = 0; first < 1u << 10; first += 7, ++runs) {
            Workgroup group{ first };
            std::vector<uint32_t> numbers[2];
            const auto run = [&](int id) {
                Wave wave{ group, id };
                {
                    std::unique_lock<std::mutex> lock(group.mutex);
                    group.wait_turn(lock, id);
                }
                wave.sync();
                wave.ask();
                wave.sync();
                pxh::walk_shares(wave, wave.next(), kAll, [&](uint32_t number) {
                    numbers[id].push_back(number);
                    if (numbers[id].size() > 2 * kAll || !(asking >> (number % kAll) & 1)) return false;
                    wave.sync();
                    if (id == 1) group.word = group.counter++;
                    return true;
                });
                group.arrive(id, true);
            };
            group.running = group.leader();
            std::thread other(run, 1);
            run(0);
            other.join();
            bool good = !group.mismatch && numbers[0] == numbers[1] && numbers[0].size() == kAll;
            for (uint32_t i = 0; good && i < kAll; ++i) good = numbers[0][i] == i;
            if (!good && !bad++) {
                std::printf("asking %x, order %x:", asking, first);
                for (const auto& mine: numbers) {
                    for (uint32_t n: mine) std::printf(" %u", n);
                    std::printf(" /");
                }
                std::printf("%s\n", group.mismatch ? " barriers that do not match" : "");
            }
        }
    std::printf("%d orders, %d failed\n", runs, bad);
    return bad != 0;
}
