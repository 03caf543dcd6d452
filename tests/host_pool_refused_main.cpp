// A worker pool whose threads the system refuses after the first few: it must
// do its passes with those it got, none included.
#include <sys/resource.h>

#include <atomic>
#include <cstdio>
#include <fstream>
#include <string>

#include "rh_pool.h"

static size_t address_space() {
    std::ifstream f("/proc/self/statm");
    size_t pages = 0;
    f >> pages;
    return pages * 4096;
}

int main() {
    for (size_t room : {(size_t)64 << 20, (size_t)1 << 20}) {
        // A thread's stack takes 8 MB or more of address space.
        rlimit old{};
        if (getrlimit(RLIMIT_AS, &old)) return 2;
        rlimit lim = old;
        lim.rlim_cur = address_space() + room;
        if (setrlimit(RLIMIT_AS, &lim)) return 2;
        {
            rhi::HostPool pool(256);
            std::atomic<int> sum{0};
            for (int pass = 0; pass < 3; ++pass) pool.run(100, [&](int k) { sum.fetch_add(k); });
            if (sum.load() != 3 * 4950) return 1;
        }
        if (setrlimit(RLIMIT_AS, &old)) return 2;
    }
    std::puts("pool ok");
    return 0;
}
