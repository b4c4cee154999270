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

}  // namespace sl
