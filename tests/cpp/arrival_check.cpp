// CPU check of csrc/hip/arrival.hpp: four threads stand for the waves of a workgroup.  Wave 0 uses the
// LDS word again as soon as last_of returns, as the sum that follows it in the kernel does, and the other
// waves come out of every barrier late.  All of them have to agree on whether the workgroup is the last.
// Prints "OK <workgroups>".
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <mutex>
#include <thread>
#include <vector>

#include "../../cudacompress_amd/csrc/hip/arrival.hpp"

namespace {

constexpr int kWaves = 4;

struct Barrier {
    std::mutex m;
    std::condition_variable cv;
    int waiting = 0, round = 0;
    void wait() {
        std::unique_lock<std::mutex> l(m);
        const int r = round;
        if (++waiting == kWaves) {
            waiting = 0;
            round++;
            cv.notify_all();
        } else {
            cv.wait(l, [&] { return round != r; });
        }
    }
};

struct WaveEx {
    int wave;
    Barrier* b;
    std::atomic<uint32_t>*counter, *word;
    void arrive() const {}
    void barrier() const {
        b->wait();
        if (wave != 0) std::this_thread::sleep_for(std::chrono::milliseconds(3 * wave));
    }
    bool leader() const { return wave == 0; }
    uint32_t count() const { return counter->fetch_add(1u); }
    void put(uint32_t v) const { word->store(v); }
    uint32_t get() const { return word->load(); }
};

}  // namespace

int main() {
    constexpr uint32_t kGroups = 9;
    std::atomic<uint32_t> counter{0};
    for (uint32_t g = 0; g < kGroups; g++) {
        Barrier b;
        std::atomic<uint32_t> word{0xDEADu};
        bool last[kWaves] = {};
        std::vector<std::thread> waves;
        for (int w = 0; w < kWaves; w++)
            waves.emplace_back([&, w] {
                last[w] = cca::last_of(WaveEx{w, &b, &counter, &word}, kGroups);
                if (w == 0) word.store(last[0] ? 0u : kGroups - 1);  // the word's next use, with a misleading value
            });
        for (auto& t : waves) t.join();
        for (int w = 0; w < kWaves; w++)
            if (last[w] != (g == kGroups - 1)) {
                printf("FAIL workgroup %u of %u, wave %d: last = %d\n", g, kGroups, w, (int)last[w]);
                return 1;
            }
    }
    printf("OK %u\n", kGroups);
    return 0;
}
