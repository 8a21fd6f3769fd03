// Once for each kernel and device, from any thread; a failure is not kept.
#include <atomic>
#include <cstdio>
#include <thread>
#include <vector>

#include "once_per_device.hpp"

int main() {
    lbm::OncePerDevice once;
    const int kernels[2] = {0, 0};
    int fails = 0, calls = 0;
    auto ok = [&](int k, int device, bool works) {
        return once(&kernels[k], device, [&] {
            ++calls;
            return works;
        });
    };
    auto expect = [&](bool got, bool want, int n) {
        if (got != want || calls != n) {
            ++fails;
            printf("FAIL: %d, %d calls; expected %d, %d\n", (int)got, calls, (int)want, n);
        }
    };
    expect(ok(0, 0, true), true, 1);
    expect(ok(0, 0, false), true, 1);   // done
    expect(ok(0, 1, false), false, 2);  // another device is on its own,
    expect(ok(0, 1, true), true, 3);    // and asked again after a failure
    expect(ok(1, 0, true), true, 4);    // as is another kernel
    expect(ok(0, 0, true), true, 4);
    std::atomic<int> set{0};
    std::vector<std::thread> threads;
    for (int t = 0; t < 8; ++t)
        threads.emplace_back([&] {
            for (int d = 0; d < 100; ++d)
                once(&set, d, [&] {
                    ++set;
                    return true;
                });
        });
    for (std::thread &t : threads) t.join();
    if (set != 100) {
        ++fails;
        printf("FAIL: %d of 100\n", set.load());
    }
    if (!fails) printf("once per device: ok\n");
    return fails ? 1 : 0;
}
