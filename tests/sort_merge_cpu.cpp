// The merges of the sort in runs (sort_merge.h) on the CPU: every step is
// called for the threads of a workgroup in turn.  Runs are sorted by the
// standard library.
#define __HIP_PLATFORM_AMD__
#include "sort_merge.h"

#include <algorithm>
#include <memory>
#include <numeric>
#include <utility>
#include <vector>

using namespace gpunb;

namespace {

// One merge of runs of L, as k_sort_merge does it; c0: the clusters' starts
// and the end of the last.  Returns the records put outside [0, n), or where
// another one is, and merges of more runs than there is room for.
template <class Key>
int merge(const std::vector<Key> &key, const std::vector<int> &val,
          std::vector<Key> &key_out, std::vector<int> &val_out, int L, bool last,
          const int *c0) {
    const int n = (int)key.size();
    int bad = 0;
    key_out.assign(n, 0);
    val_out.assign(n, -1);
    auto lds = std::make_unique<MergeLds<Key>>();
    for (int p0 = 0; p0 < n; p0 += 64) {
        const int p1 = std::min(p0 + 63, n - 1), own = p0 / L;
        const Key a = key[p0], z = key[p1];
        int r0, r1;
        if (last) {
            r0 = (c0 ? c0[(unsigned long long)a >> 32] : 0) / L;
            r1 = ((c0 ? c0[((unsigned long long)z >> 32) + 1] : n) - 1) / L;
        } else {
            r0 = own & ~(kSortWay - 1);
            r1 = std::min(r0 + kSortWay - 1, (n - 1) / L);
        }
        if (r1 - r0 >= kSortWay) ++bad;
        constexpr int T = 64 * kParts;
        auto at = [&](int t) { return std::min(p0 + (t & 63), p1); };
        for (int t = 0; t < T; ++t)
            merge_windows(*lds, t, key.data(), n, (long long)L, own, r0, r1, a, z);
        for (int t = 0; t < T; ++t) merge_offsets(*lds, t);
        for (int t = 0; t < T; ++t) merge_load(*lds, t, key.data(), (long long)L, r0);
        for (int t = 0; t < T; ++t)
            merge_ranks(*lds, t, key.data(), (long long)L, own, r0, key[at(t)]);
        for (int t = 0; p0 + t <= p1; ++t) {
            const int d = merge_place(*lds, t, (long long)L, own, r0, p0 + t);
            if (d < 0 || d >= n || val_out[d] >= 0) {
                ++bad;
                continue;
            }
            key_out[d] = key[p0 + t];
            val_out[d] = val[p0 + t];
        }
    }
    return bad;
}

template <class Key>
int sort(int n, const Key *k, int n_max, bool one, const int *c0, int *order) {
    std::vector<Key> key(n), key2;
    std::vector<int> val(n), val2;
    std::iota(val.begin(), val.end(), 0);
    for (int b = 0; b < n; b += kSortRun)
        std::stable_sort(val.begin() + b, val.begin() + std::min(n, b + kSortRun),
                         [&](int x, int y) { return k[x] < k[y]; });
    for (int i = 0; i < n; ++i) key[i] = k[val[i]];
    int bad = 0;
    long long L = kSortRun;
    for (int m = sort_merges(n, n_max, one); m > 0; --m, L *= kSortWay) {
        bad += merge(key, val, key2, val2, (int)L, false, c0);
        std::swap(key, key2);
        std::swap(val, val2);
    }
    bad += merge(key, val, key2, val2, (int)L, true, c0);
    std::copy(val2.begin(), val2.end(), order);
    return bad;
}

}  // namespace

extern "C" {

int merges_before_last(int n, int n_max, int one) {
    return sort_merges(n, n_max, one != 0);
}
int sort_one(int n, const unsigned *key, int *order) {
    return sort(n, key, n, true, nullptr, order);
}
int sort_clusters(int n, const unsigned long long *key, int n_max, const int *c0,
                  int *order) {
    return sort(n, key, n_max, false, c0, order);
}

}  // extern "C"
