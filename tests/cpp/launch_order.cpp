// The bookkeeping of fused launches on several streams (ff_launch_order.hpp)
// without a GPU. Exits with 0 if all checks hold.
#include "ff_launch_order.hpp"

#include <cstdio>

using ffamd::LaunchOrder;

#define CHECK(c)                                                       \
    do {                                                               \
        if (!(c)) {                                                    \
            std::printf("line %d: %s does not hold\n", __LINE__, #c);  \
            return 1;                                                  \
        }                                                              \
    } while (0)

// Only launches that were enqueued count, and a failed one is not the launch
// that the next follows.
static int failed_launches() {
    int streams[3];
    const void *a = &streams[0], *b = &streams[1], *c = &streams[2];
    LaunchOrder o;
    CHECK(!o.follows(a));
    o.launched(a, 10);
    CHECK(o.target == 10 && !o.follows(a) && o.follows(b));
    // (a launch on b fails: nothing is noted)
    CHECK(o.follows(b) && o.follows(c) && !o.follows(a) && o.target == 10);
    o.launched(c, 5);
    CHECK(o.target == 15 && o.follows(a) && !o.follows(c));
    o.finished(a);
    CHECK(o.follows(a));
    o.finished(c);
    CHECK(!o.follows(a) && o.target == 15);
    // modulo 2^32
    o.target = 0xfffffffeu;
    o.launched(a, 5);
    CHECK(o.target == 3u);
    return 0;
}

int main() { return failed_launches(); }
