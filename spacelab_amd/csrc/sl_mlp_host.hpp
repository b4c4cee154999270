// Host-side rules of the surrogate network (sl_mlp.hip) that need no GPU to be checked.
#pragma once

#include <algorithm>
#include <cstddef>

namespace sl {

// Pinned host memory a net holds for life.  In the chain form: a batch and its results, which the
// kernels read and write there, or the padded parameters during exchanges (at most 4.3 MB,
// CHAIN_MAX wide).  In the layer form a batch's losses or a piece of the parameters: all of
// them are 136 MB at width 4096, more than many nets can pin.  (Through unpinned memory of
// the exchange's own: width 1024 read in 770 us instead of 430, 4096 in 41 ms instead of 11.)
inline size_t pinned_bytes(bool chain, size_t batch_bytes, size_t params_bytes, int max_batch)
{
    const size_t piece = (size_t)4 << 20;
    return chain ? std::max(batch_bytes, params_bytes)
                 : std::max(sizeof(float) * (size_t)max_batch, std::min(params_bytes, piece));
}

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
