// CPU check of the host's wait for a published sequence number
// (gip_amd/csrc/gip_wait.h): prints one line per case, "name result queries".
#include <cstdio>
#include <functional>

#include "../gip_amd/csrc/gip_wait.h"

static void run(const char *name, uint64_t have, uint64_t want, const std::function<int(uint64_t &, int)> &query) {
    uint64_t flag = have;
    int asked = 0;
    const int rc = gip::wait_seq(&flag, want, [&]() { return query(flag, ++asked); });
    std::printf("%s %d %d\n", name, rc, asked);
}

int main() {
    const auto done = [](uint64_t &, int) { return 0; };
    run("there", 7, 7, done);
    run("newer", 9, 7, done);
    run("wrapped", 1, ~0ull, done);
    run("missing", 6, 7, done);
    run("arrives", 6, 7, [](uint64_t &f, int n) { if (n == 2) f = 8; return -1; });
    run("last", 6, 7, [](uint64_t &f, int) { f = 7; return 0; });
    run("failed", 6, 7, [](uint64_t &, int) { return 41; });
    return 0;
}
