// Set-up once on every device (ff_per_device.hpp) without a GPU. Exits with 0 if
// all checks hold.
#include "ff_per_device.hpp"

#include <cstdio>
#include <stdexcept>
#include <thread>
#include <vector>

int main() {
    ffamd::OncePerDevice once;
    int runs[3] = {0, 0, 0};
    bool threw = false;
    try {
        once.run(1, [] { throw std::runtime_error("refused"); });
    } catch (const std::runtime_error&) {
        threw = true;
    }
    std::vector<std::thread> t;
    for (int k = 0; k < 8; ++k)
        t.emplace_back([&] {
            for (int r = 0; r < 1000; ++r) once.run(r % 3, [&] { ++runs[r % 3]; });
        });
    for (auto& x : t) x.join();
    if (threw && runs[0] == 1 && runs[1] == 1 && runs[2] == 1) return 0;
    std::printf("ran %d %d %d times\n", runs[0], runs[1], runs[2]);
    return 1;
}
