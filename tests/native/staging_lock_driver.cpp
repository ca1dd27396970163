// The lock of the shared staging (csrc/gdp_copy_pool.h): while a copy has it, a
// copy of less than 1 MiB goes on without it and a bulk copy waits.  Prints
// "ok" and exits 0.
#include <atomic>
#include <chrono>
#include <cstdio>

#include "gdp_copy_pool.h"

#define CHECK(x)                                       \
    do {                                               \
        if (!(x)) {                                    \
            std::printf("line %d: %s\n", __LINE__, #x); \
            return 1;                                  \
        }                                              \
    } while (0)

int main() {
    std::mutex use;
    std::atomic<bool> held{false}, owned_small{true}, small_done{false}, bulk_done{false};
    use.lock();
    std::thread small([&] {
        owned_small = gdp::staging_lock(use, gdp::kBulkMin - 1).owns_lock();
        small_done = true;
    });
    std::thread bulk([&] {
        const auto lk = gdp::staging_lock(use, gdp::kBulkMin);
        held = lk.owns_lock();
        bulk_done = true;
    });
    for (int i = 0; i < 500 && !small_done; i++) std::this_thread::sleep_for(std::chrono::milliseconds(10));
    const bool in_time = small_done;
    std::this_thread::sleep_for(std::chrono::milliseconds(50));
    const bool bulk_waited = !bulk_done;
    use.unlock();
    small.join();
    bulk.join();
    CHECK(in_time && !owned_small && bulk_waited && held);
    CHECK(gdp::staging_lock(use, 1).owns_lock());
    std::printf("ok\n");
    return 0;
}
