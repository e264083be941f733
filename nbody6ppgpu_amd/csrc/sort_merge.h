// sort_merge.h -- the steps of a merge of the sort in runs (jprep.hip), free of
// launches: each is called by the threads t of a workgroup, a barrier between
// one and the next, or by a loop over t on the CPU.
#pragma once

#include <hip/hip_runtime.h>

namespace gpunb {

constexpr int kSortRun = 1024;   // records of a first run, one per thread
constexpr int kSortWay = 32;     // runs of one merge

// Merges of kSortWay runs before the last merge, for n records, a cluster
// holding at most n_max of them.  The last merge takes the runs of whole
// clusters.  64 records of a run can be of several: the first's may begin, the
// last's end, span - 1 runs away, so a cluster spans at most half of kSortWay;
// a single one all.
inline int sort_merges(int n, int n_max, bool one) {
    auto final_at = [&](long long L) {
        return one ? (n + L - 1) / L <= kSortWay : (n_max - 1) / L + 2 <= kSortWay / 2;
    };
    int merges = 0;
    for (long long L = kSortRun; !final_at(L); L *= kSortWay) ++merges;
    return merges;
}

// Records among a[0, m) (ascending) before one of key k: the smaller keys,
// and the equal ones where eq.  8 pieces a step: their ends' loads overlap,
// a halving search would wait for each (1024 records: 4 waits, not 10).
template <class Key>
__host__ __device__ inline int count_before(const Key *a, int m, Key k, bool eq) {
    int lo = 0, len = m;             // the count is in [lo, lo + len]
    while (len > 0) {
        const int st = (len + 7) >> 3;
        int c = 0;
#pragma unroll
        for (int u = 1; u < 8; ++u) {
            const bool in = u * st <= len;
            const Key o = a[lo + (in ? u * st : st) - 1];
            c += (in && (eq ? o <= k : o < k)) ? 1 : 0;
        }
        const bool closed = c < 7 && (c + 1) * st <= len;   // probe c + 1 is not before
        lo += c * st;
        len = closed ? st - 1 : len - c * st;
    }
    return lo;
}

// A workgroup places 64 consecutive records of a run of L among the runs
// r0..r1: the records of every other run that lie between the first and the
// last of them are counted for each by search in LDS, those before the first
// are common.  kSortWay / kParts runs a wavefront, so that its loads are in
// flight together.
constexpr int kParts = 4;
constexpr int kPartWay = kSortWay / kParts;
template <class Key>
struct MergeLds {
    static constexpr int kWin = 16384 / (int)sizeof(Key);
    Key win[kWin + 1];               // one more: read for an empty window
    int cnt[2 * kSortWay];           // records before the first, the last
    int off[kSortWay + 1];           // windows' starts in win, their total
    int common;
    int sum[kParts][64];
};
// Steps of the threads t, a barrier between each.
template <class Key>
__host__ __device__ inline void merge_windows(MergeLds<Key> &S, int t,
                                              const Key *key, int n, long long L,
                                              int own, int r0, int r1, Key first,
                                              Key last) {
    if (t >= 2 * kSortWay) return;
    const int r = r0 + (t >> 1);
    int c = 0;
    if (r <= r1 && r != own) {
        const long long a = r * L;
        c = count_before(key + a, (int)(n - a < L ? n - a : L),
                         (t & 1) ? last : first, r < own);
    }
    S.cnt[t] = c;
}
template <class Key>
__host__ __device__ inline void merge_offsets(MergeLds<Key> &S, int t) {
    if (t > kSortWay) return;
    int sum = 0, common = 0;
#pragma unroll 8
    for (int q = 0; q < kSortWay; ++q) {
        const int lo = S.cnt[2 * q], hi = S.cnt[2 * q + 1];
        sum += q < t ? hi - lo : 0;
        common += lo;
    }
    S.off[t] = sum;
    if (t == 0) S.common = common;
}
template <class Key>
__host__ __device__ inline void merge_load(MergeLds<Key> &S, int t,
                                           const Key *key, long long L, int r0) {
    if (S.off[kSortWay] > MergeLds<Key>::kWin) return;   // searched in place
    const int lane = t & 63, q0 = (t >> 6) * kPartWay;
    Key v[kPartWay][2];
    int w[kPartWay];
#pragma unroll
    for (int u = 0; u < kPartWay; ++u) {
        const int q = q0 + u;
        const Key *a = key + (r0 + q) * L + S.cnt[2 * q];
        w[u] = S.off[q + 1] - S.off[q];
        if (lane < w[u]) v[u][0] = a[lane];
        if (lane + 64 < w[u]) v[u][1] = a[lane + 64];
    }
#pragma unroll
    for (int u = 0; u < kPartWay; ++u) {
        const int q = q0 + u;
        if (lane < w[u]) S.win[S.off[q] + lane] = v[u][0];
        if (lane + 64 < w[u]) S.win[S.off[q] + lane + 64] = v[u][1];
        for (int e = lane + 128; e < w[u]; e += 64)
            S.win[S.off[q] + e] = key[(r0 + q) * L + S.cnt[2 * q] + e];
    }
}
// Records of part `part` in the windows before one of key k; at(q, e, w) is
// the e-th of window q of w, anything past it.
template <class Key, class At>
__host__ __device__ inline int merge_count(const MergeLds<Key> &S, int part, int own,
                                           int r0, Key k, At at) {
    int pos[kPartWay], w[kPartWay], wmax = 0;
    const int q0 = part * kPartWay;
#pragma unroll
    for (int u = 0; u < kPartWay; ++u) {
        pos[u] = 0;
        w[u] = S.off[q0 + u + 1] - S.off[q0 + u];
        wmax = w[u] > wmax ? w[u] : wmax;
    }
    if (wmax == 0) return 0;
    for (int h = 1 << (31 - __builtin_clz(wmax)); h >= 1; h >>= 1)
#pragma unroll
        for (int u = 0; u < kPartWay; ++u) {
            const int e = pos[u] + h - 1;
            const Key o = at(q0 + u, e, w[u]);
            const bool before = r0 + q0 + u < own ? o <= k : o < k;
            pos[u] += e < w[u] && before ? h : 0;
        }
    int sum = 0;
#pragma unroll
    for (int u = 0; u < kPartWay; ++u) sum += pos[u];
    return sum;
}
template <class Key>
__host__ __device__ inline void merge_ranks(MergeLds<Key> &S, int t, const Key *key,
                                            long long L, int own, int r0, Key k) {
    const int part = t >> 6;
    int c;
    if (S.off[kSortWay] <= MergeLds<Key>::kWin)
        c = merge_count(S, part, own, r0, k,
                        [&](int q, int e, int w) {
                            return S.win[S.off[q] + (e < w ? e : 0)];
                        });
    else
        c = merge_count(S, part, own, r0, k, [&](int q, int e, int w) {
            return e < w ? key[(r0 + q) * L + S.cnt[2 * q] + e] : (Key)0;
        });
    S.sum[part][t & 63] = c;
}
// Place of the group's record `lane`, at position p.
template <class Key>
__host__ __device__ inline int merge_place(const MergeLds<Key> &S, int lane,
                                           long long L, int own, int r0, int p) {
    int d = (int)(r0 * L + (p - own * L)) + S.common;
#pragma unroll
    for (int part = 0; part < kParts; ++part) d += S.sum[part][lane];
    return d;
}

}  // namespace gpunb
