// CPU check of csrc/host/parallel.hpp: every index once, with all threads, with none to be had and with
// some; and an exception out of the work reaches the caller.  Prints "OK".
#include <cstdio>
#include <cstdlib>
#include <stdexcept>
#include <string>

#include "../../cudacompress_amd/csrc/host/parallel.hpp"

namespace {
int failures = 0;
void expect(bool ok, const char* what) {
    if (!ok) {
        printf("FAIL %s\n", what);
        failures++;
    }
}
bool each_once(size_t n, double work_us, int threads_to_be_had) {
    std::vector<std::atomic<int>> seen(n);
    int started = 0;
    cca::parallel_for(n, work_us, [&](size_t i) { seen[i]++; }, [&](auto& work) {
        if (started++ >= threads_to_be_had) throw std::system_error(std::make_error_code(std::errc::resource_unavailable_try_again));
        return std::thread(std::ref(work));
    });
    for (auto& s : seen)
        if (s != 1) return false;
    return true;
}
}  // namespace

int main() {
    for (size_t n : {0u, 1u, 2u, 7u, 1000u})
        for (double us : {0.0, 80.0, 1e6})
            for (int t : {0, 1, 3, 64}) expect(each_once(n, us, t), "every index once");
    for (double us : {0.0, 1e6}) {
        bool caught = false;
        try {
            cca::parallel_for(500, us, [](size_t i) {
                if (i == 123) throw std::runtime_error("123");
            });
        } catch (const std::runtime_error& e) {
            caught = std::string(e.what()) == "123";
        }
        expect(caught, "the exception");
    }
    if (!failures) printf("OK\n");
    return failures != 0;
}
