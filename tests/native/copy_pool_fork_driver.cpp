// The copy threads (csrc/gdp_copy_pool.h) stay for the next bulk copy.  A child
// forked meanwhile does not have them and must still end by itself: the
// process-wide object is not destroyed.  Prints "ok" and exits 0.
#include <sys/wait.h>
#include <unistd.h>

#include <chrono>
#include <csignal>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "gdp_copy_pool.h"

int main() {
    std::vector<char> src(4u << 20, 7), dst(src.size());
    gdp::CopyPool &pool = gdp::process_wide<gdp::CopyPool>();
    pool.copy(dst.data(), src.data(), src.size(), 4);
    if (dst != src || pool.threads() != 3 || &pool != &gdp::process_wide<gdp::CopyPool>()) return 1;
    const pid_t child = fork();
    if (child == 0) std::exit(0);
    int status = 0;
    for (int i = 0; i < 500; i++) {
        if (waitpid(child, &status, WNOHANG) == child) {
            if (!WIFEXITED(status) || WEXITSTATUS(status) != 0) return 2;
            std::printf("ok\n");
            return 0;
        }
        std::this_thread::sleep_for(std::chrono::milliseconds(10));
    }
    kill(child, SIGKILL);
    waitpid(child, &status, 0);
    std::printf("the child did not end\n");
    return 3;
}
