// Host-side rules of the surrogate network (sl_mlp.hip) that need no GPU to be checked.
#pragma once

namespace sl {

// What decides whether nets are laid out alike, so that one launch can carry them: a member's
// memory is then the first member's, moved by a distance, on the same device.
struct NetKind {
    int device = 0;
    bool chain = false;   // only the chain form shares launches
    int n_in = 0, width = 0, n_out = 0, max_batch = 0;
};

inline bool shares_launch(const NetKind& a, const NetKind& b)
{
    return a.chain && b.chain && a.device == b.device && a.n_in == b.n_in && a.width == b.width && a.n_out == b.n_out &&
           a.max_batch == b.max_batch;
}

// n passes with `ahead` of them in flight: issue(k) sends pass k, collect(k) waits for it and
// takes its results, in order.  After a failure nothing more is sent and wait() is called, so
// that no launch outlives the call, whose buffers the next call writes.  Returns the first
// nonzero code.
template <class Issue, class Collect, class Wait>
int run_ahead(long long n, int ahead, Issue issue, Collect collect, Wait wait)
{
    int rc = 0;
    for (long long k = 0; k < n && !rc; k++) {
        if (k >= ahead) rc = collect(k - ahead);
        if (!rc) rc = issue(k);
    }
    for (long long k = n > ahead ? n - ahead : 0; k < n && !rc; k++) rc = collect(k);
    if (rc) wait();
    return rc;
}

}  // namespace sl
