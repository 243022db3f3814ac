// Checks of the index rules that the attention kernels share with their host
// launcher (kv_params.h), over every size that the kernels admit.
#include <cstdio>
#include <cstdlib>

#include "kv_params.h"

namespace {

[[noreturn]] void fail(const char *what, unsigned dv, unsigned splits, unsigned thread) {
    std::fprintf(stderr, "%s: dv %u, %u splits, thread %u\n", what, dv, splits, thread);
    std::exit(1);
}

// The combine kernel's threads: the shares that a merging thread reads lie
// inside the workgroup's array and were written, and every (query, head) of
// the workgroup has `per` whole sets, the first of which merges.
void combine_places() {
    for (unsigned dv = 1; dv <= 1024; ++dv)
        for (unsigned splits = 2; splits <= 600; ++splits) {
            unsigned merging = 0;
            for (unsigned t = 0; t < SGLKV_ATTN_COMBINE_THREADS; ++t) {
                const sglkv_combine_place c = sglkv_combine_place_of(t, dv, splits);
                if (c.per == 0 || c.items == 0) fail("no set", dv, splits, t);
                if (!c.merges) continue;
                if (t + (c.per - 1) * c.lanes >= SGLKV_ATTN_COMBINE_THREADS)
                    fail("a share past the workgroup is read", dv, splits, t);
                for (unsigned k = 1; k < c.per; ++k) {
                    const sglkv_combine_place o = sglkv_combine_place_of(t + k * c.lanes, dv, splits);
                    if (o.own != c.own || o.sub != k) fail("another (query, head)'s share is read", dv, splits, t);
                }
                if (c.own >= c.items) fail("a set with no (query, head) merges", dv, splits, t);
                ++merging;
            }
            const sglkv_combine_place c = sglkv_combine_place_of(0, dv, splits);
            if (merging != c.items * c.lanes) fail("(query, head)s without a merging set", dv, splits, merging);
        }
}

}  // namespace

int main() {
    combine_places();
    std::puts("attention rules ok");
    return 0;
}
