// The pool of pinned blocks (csrc/gdp_host_blocks.h), with ordinary memory in
// place of pinned: a request that fails leaves a block that the next request
// allocates anew; kept blocks are handed out again and bounded.
// Prints "ok" and exits 0.
#include <cstdio>
#include <cstdlib>
#include <stdexcept>

#include "gdp_host_blocks.h"

static int g_live = 0, g_fail = 0;
static void *grab(size_t bytes) {
    if (g_fail > 0 && --g_fail == 0) throw std::runtime_error("no pinned memory");
    g_live++;
    return std::malloc(bytes);
}
static void drop(void *p) {
    g_live--;
    std::free(p);
}
#define CHECK(x)                                       \
    do {                                               \
        if (!(x)) {                                    \
            std::printf("line %d: %s\n", __LINE__, #x); \
            return 1;                                  \
        }                                              \
    } while (0)

int main() {
    gdp::HostBlocks pool(grab, drop);
    {
        gdp::HostBlock b(pool);
        char *first = b.get(1000);
        CHECK(first && b.size == 4096 && b.get(4096) == first);
        g_fail = 1;
        bool threw = false;
        try {
            b.get(5000);
        } catch (const std::runtime_error &) {
            threw = true;
        }
        CHECK(threw);
        CHECK(b.get(5000) != nullptr && b.size == 8192);
        b.p[8191] = 1;
        CHECK(b.get(100) == b.p);
    }
    {
        gdp::HostBlock b(pool), c(pool);
        const int live = g_live;
        CHECK(b.get(1) && c.get(8192) && g_live == live);  // both kept from before
        CHECK(c.get((1u << 20) + 1) && g_live == live + 1);
    }
    {  // 16 MiB are kept, the rest goes back
        gdp::HostBlock *many[40];
        for (auto &m : many) {
            m = new gdp::HostBlock(pool);
            m->get(1u << 20);
        }
        for (auto &m : many) delete m;
        CHECK(g_live <= 16 + 2);
    }
    std::printf("ok\n");
    return 0;
}
