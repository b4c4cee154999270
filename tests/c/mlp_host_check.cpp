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

int main()
{
    sharing();
    return 0;
}
