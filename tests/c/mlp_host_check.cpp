// The surrogate network's host rules (sl_mlp_host.hpp), built without HIP.  Prints the name of
// each rule that does not hold; nothing when all do.
#include "sl_mlp_host.hpp"

#include <cstdio>

using namespace sl;

static void check(bool ok, const char* what)
{
    if (!ok) std::printf("%s\n", what);
}

static void sharing()
{
    const NetKind a{0, true, 21, 256, 9, 4096};
    check(shares_launch(a, a), "nets of one kind share launches");
    NetKind b[6] = {a, a, a, a, a, a};
    b[0].device = 1;
    b[1].chain = false;
    b[2].n_in = 20;
    b[3].width = 128;
    b[4].n_out = 8;
    b[5].max_batch = 64;
    for (const NetKind& x : b) check(!shares_launch(a, x) && !shares_launch(x, a), "nets of another device, form or size do not");
}

// Passes 0 .. n - 1 with issue or collect of pass `bad` failing (-1: none).
static void ahead(long long n, int in_flight, long long bad, bool in_issue)
{
    long long issued = 0, collected = 0, waits = 0;
    bool order = true;
    const int rc = run_ahead(
        n, in_flight,
        [&](long long k) {
            order = order && k == issued && issued - collected < in_flight && waits == 0;
            if (in_issue && k == bad) return -2;
            issued++;
            return 0;
        },
        [&](long long k) {
            order = order && k == collected && k < issued && waits == 0;
            if (!in_issue && k == bad) return -3;
            collected++;
            return 0;
        },
        [&] { waits++; });
    check(order, "passes in order, no more in flight than asked");
    if (bad < 0) {
        check(rc == 0 && issued == n && collected == n && waits == 0, "every pass sent and collected");
    } else {
        check(rc == (in_issue ? -2 : -3), "the first failure is returned");
        check(waits == 1, "after a failure the work in flight is waited for");
        check(in_issue ? issued == bad : collected == bad, "nothing after the failure");
    }
}

static void pinned()
{
    const size_t wide = (size_t)136 << 20, batch = 1 << 20, narrow = 600 << 10;
    check(pinned_bytes(false, batch, wide, 4096) == 4 << 20, "a wide net in the layer form pins a piece of its parameters");
    check(pinned_bytes(false, wide, narrow, 64) == narrow && pinned_bytes(false, wide, narrow, 1 << 20) == 4 << 20,
          "a net in the layer form pins its losses and no batch");
    check(pinned_bytes(true, batch, narrow, 4096) == batch && pinned_bytes(true, narrow, batch, 4096) == batch,
          "a net in the chain form pins what a batch and an exchange need");
}

int main()
{
    sharing();
    pinned();
    for (long long n = 0; n < 6; n++)
        for (int a = 1; a < 3; a++) {
            ahead(n, a, -1, true);
            for (long long bad = 0; bad < n; bad++) {
                ahead(n, a, bad, true);
                ahead(n, a, bad, false);
            }
        }
    return 0;
}
