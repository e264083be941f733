// jprep.hip -- the sorted j view of the regular-force engine.
//
// After every send / predict the j set is reordered along a Hilbert curve, so
// that 64 consecutive sorted j form a spatially compact tile, and each j is
// stored as an FP32 offset from its tile's FP64 centre (JRec32).  The pair
// loop then forms x_j - x_i as (C_t - x_i) + o_j: the first term once per
// (i, tile) in FP64 and rounded, the second one FP32 add per pair, instead of
// an FP64 subtraction and a conversion per pair component.
//
// Steps (all on the library stream, deterministic):
//   k_jstat1   per block of kStatChunk j: bounding box and mass sum, reduced
//              in a fixed order
//   k_jstat2   per cluster: the blocks' partials in block order -> JClus
//              (bounding box, mean mass)
//   sort       by key (cluster << 32 | heavy << 30 | 30-bit Hilbert index of
//              the position in the cluster's box; padding records sort last),
//              stable, so equal codes keep their index order: k_sort_runs,
//              then k_sort_merge once or more
//   k_jtile    one wavefront per tile: sorted FP64 records, sorted -> original
//              index map, tile centres and offset bounds, FP32 records
#include "gpunb_internal.h"
#include "sort_merge.h"

#include <algorithm>
#include <cfloat>
#include <cmath>

namespace gpunb {
namespace {

__device__ inline double wmin(double v) {
    for (int o = 32; o >= 1; o >>= 1) v = fmin(v, __shfl_xor(v, o));
    return v;
}
__device__ inline double wmax(double v) {
    for (int o = 32; o >= 1; o >>= 1) v = fmax(v, __shfl_xor(v, o));
    return v;
}
// The same within each kVTile-lane segment of the wavefront.
__device__ inline double smin(double v) {
    for (int o = kVTile / 2; o >= 1; o >>= 1) v = fmin(v, __shfl_xor(v, o));
    return v;
}
__device__ inline double smax(double v) {
    for (int o = kVTile / 2; o >= 1; o >>= 1) v = fmax(v, __shfl_xor(v, o));
    return v;
}

// FP32 value >= v (v finite, >= 0).
__device__ inline float up32(double v) {
    float f = (float)v;
    if ((double)f < v) f = nextafterf(f, INFINITY);
    return f;
}

// Cluster owning position g of the concatenated ranges (last c with
// pc[c].j0 <= g).
__device__ inline int clus_of(const PrepClus *__restrict__ pc, int ncl, int g) {
    int lo = 0, hi = ncl - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (pc[mid].j0 <= g) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}
__device__ inline int clus_of_blk(const PrepClus *__restrict__ pc, int ncl,
                                  int b) {
    int lo = 0, hi = ncl - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (pc[mid].blk0 <= b) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// 10 bits spread to every third position.
__device__ inline unsigned spread3(unsigned v) {
    v &= 0x3ffu;
    v = (v | (v << 16)) & 0x030000ffu;
    v = (v | (v << 8)) & 0x0300f00fu;
    v = (v | (v << 4)) & 0x030c30c3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

__device__ inline unsigned cell10(double x, double lo, double scale) {
    const double q = (x - lo) * scale;
    if (!(q > 0.0)) return 0u;           // also NaN
    if (q >= 1023.0) return 1023u;
    return (unsigned)q;
}

// Index of cell (x, y, z) (10 bits each) along a 3-D Hilbert curve of the
// 1024^3 grid, 30 bits: J. Skilling, "Programming the Hilbert curve", AIP
// Conf. Proc. 707 (2004) 381 -- the axes are turned into the curve's
// "transpose" form (undo the excess work of each level, then Gray-encode),
// whose bits interleaved from the top are the index.  Consecutive indices are
// adjacent cells, so 64 consecutive bodies form a more compact tile than a
// Morton run, which jumps at every power-of-two cell boundary (King N = 131072:
// median tile extent 1.71 against 2.00 neighbour radii).
__device__ inline unsigned hilbert30(unsigned x, unsigned y, unsigned z) {
    unsigned X[3] = {x, y, z};
    for (unsigned Q = 1u << 9; Q > 1u; Q >>= 1) {
        const unsigned P = Q - 1u;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            if (X[i] & Q) {
                X[0] ^= P;
            } else {
                const unsigned t = (X[0] ^ X[i]) & P;
                X[0] ^= t;
                X[i] ^= t;
            }
        }
    }
    X[1] ^= X[0];
    X[2] ^= X[1];
    unsigned t = 0u;
    for (unsigned Q = 1u << 9; Q > 1u; Q >>= 1)
        if (X[2] & Q) t ^= Q - 1u;
    X[0] ^= t;
    X[1] ^= t;
    X[2] ^= t;
    return (spread3(X[0]) << 2) | (spread3(X[1]) << 1) | spread3(X[2]);
}

// Curve key of a position in the cube of a cluster's bounding box.
__device__ inline unsigned cell_key(double x, double y, double z,
                                    const JClus &J) {
    const double ext = fmax(fmax(J.hi[0] - J.lo[0], J.hi[1] - J.lo[1]),
                            J.hi[2] - J.lo[2]);
    const double scale = ext > 0.0 ? 1024.0 / ext : 0.0;
    return hilbert30(cell10(x, J.lo[0], scale), cell10(y, J.lo[1], scale),
                     cell10(z, J.lo[2], scale));
}

// Fixed-order tree reduction of 8 doubles over a 256-thread workgroup
// (components 0-2 min, 3-5 max, 6-7 sum).
__device__ inline void block_reduce8(double v[8], double (*sh)[8]) {
    const int t = threadIdx.x;
#pragma unroll
    for (int k = 0; k < 8; ++k) sh[t][k] = v[k];
    __syncthreads();
    for (int s = 128; s >= 1; s >>= 1) {
        if (t < s) {
#pragma unroll
            for (int k = 0; k < 3; ++k) sh[t][k] = fmin(sh[t][k], sh[t + s][k]);
#pragma unroll
            for (int k = 3; k < 6; ++k) sh[t][k] = fmax(sh[t][k], sh[t + s][k]);
            sh[t][6] += sh[t + s][6];
            sh[t][7] += sh[t + s][7];
        }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = sh[0][k];
}

}  // namespace

__global__ __launch_bounds__(256) void k_jstat1(const JRec *__restrict__ jp,
                                                const PrepClus *__restrict__ pc,
                                                int ncl,
                                                double *__restrict__ part) {
    __shared__ double sh[256][8];
    const int b = blockIdx.x;
    const PrepClus P = pc[clus_of_blk(pc, ncl, b)];
    const int beg = P.j0 + (b - P.blk0) * kStatChunk;
    const int end = min(beg + kStatChunk, P.j0 + P.nj);
    double v[8] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY,
                   -INFINITY, 0.0, 0.0};
    for (int j = beg + (int)threadIdx.x; j < end; j += 256) {
        const JRec &r = jp[j];
        v[0] = fmin(v[0], r.x);
        v[1] = fmin(v[1], r.y);
        v[2] = fmin(v[2], r.z);
        v[3] = fmax(v[3], r.x);
        v[4] = fmax(v[4], r.y);
        v[5] = fmax(v[5], r.z);
        v[6] += r.m;
    }
    block_reduce8(v, sh);
    if (threadIdx.x < 8) part[8 * (size_t)b + threadIdx.x] = v[threadIdx.x];
}

__global__ __launch_bounds__(256) void k_jstat2(const PrepClus *__restrict__ pc,
                                                int ncl, int nblk,
                                                const double *__restrict__ part,
                                                JClus *__restrict__ jcl) {
    __shared__ double sh[256][8];
    const int c = blockIdx.x;
    const int b0 = pc[c].blk0;
    const int b1 = (c + 1 < ncl) ? pc[c + 1].blk0 : nblk;
    double v[8] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY,
                   -INFINITY, 0.0, 0.0};
    for (int b = b0 + (int)threadIdx.x; b < b1; b += 256) {
        const double *p = part + 8 * (size_t)b;
#pragma unroll
        for (int k = 0; k < 3; ++k) v[k] = fmin(v[k], p[k]);
#pragma unroll
        for (int k = 3; k < 6; ++k) v[k] = fmax(v[k], p[k]);
        v[6] += p[6];
    }
    block_reduce8(v, sh);
    if (threadIdx.x == 0) {
        JClus J;
        const int nj = pc[c].nj;
        for (int k = 0; k < 3; ++k) {
            J.lo[k] = nj > 0 ? v[k] : 0.0;
            J.hi[k] = nj > 0 ? v[3 + k] : 0.0;
        }
        J.mbar = nj > 0 ? v[6] / nj : 0.0;
        J.pad = 0.0;
        jcl[c] = J;
    }
}

// Key code of record g of cluster c, and of an i in the box of J.
__device__ inline unsigned j_code(const JRec *__restrict__ jp, const PrepClus &P,
                                  const JClus &J, int g) {
    if (g - P.j0 >= P.nj) return 0xffffffffu;       // padding sorts last
    const JRec &r = jp[g];
    unsigned code = cell_key(r.x, r.y, r.z, J);
    // Heavy bodies (m > kHeavy <m>) sort after the light ones, in tiles of
    // their own: their band weight w_j would otherwise widen the near region
    // of every tile that holds one.
    if (r.m > (double)kHeavy * J.mbar) code |= 1u << 30;
    return code;
}
__device__ inline unsigned i_code(const double *__restrict__ xi, const JClus &J,
                                  int g) {
    return cell_key(xi[3 * (size_t)g + 0], xi[3 * (size_t)g + 1],
                    xi[3 * (size_t)g + 2], J);
}
// Cluster of global i g: the last c with cl_i0[c] <= g (clusters hold
// consecutive i ranges in cluster order, empty ones repeat the next start).
__device__ inline int iclus_of(const int *__restrict__ cl_i0, int ncl, int g) {
    int lo = 0, hi = ncl - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (cl_i0[mid] <= g) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// ---------------------------------------------------------------------------
// Stable sort.  k_sort_runs sorts runs of kSortRun consecutive records by
// (cluster, code) in LDS, forming the keys itself; k_sort_merge merges up to
// kSortWay runs in one launch, and the last merge writes the result (for i:
// gathers the data) in place of another launch.
//
// Bound: launches, load latency and cold instructions, not bandwidth (a sort
// of N = 16411 moves 0.4 MB).  The library's radix sort is at these sizes a
// block sort and a launch per doubling, 8 launches and 41 us for N = 16411
// besides the key and gather launches; here 12.2 + 18.0 us with the keys in
// them (131072: 45 us before, 12.8 + 28.6 + 25.6 us).  Whole step, j and i
// sorts: N = 9000 435 -> 423 us, 16411 703 -> 688 us, 32000 1480 -> 1450 us,
// 131072 13.63 -> 13.66 ms (within its spread).  Rolled loops: unrolled ones
// are 11 KB of code that every launch fetches for one pass, 26.5 us for the
// merge and 703 -> 707 us.
// ---------------------------------------------------------------------------

struct JSort32 {      // j records of one cluster
    using Key = unsigned;
    const JRec *jp;
    const PrepClus *pc;
    const JClus *jcl;
    int *out;
    __device__ Key key(int g) const { return j_code(jp, pc[0], jcl[0], g); }
    __device__ void range(Key, int n, int &b, int &e) const { b = 0, e = n; }
    __device__ void put(int p, int g) const { out[p] = g; }
};
struct JSort64 {      // j records of an ensemble
    using Key = unsigned long long;
    const JRec *jp;
    const PrepClus *pc;
    const JClus *jcl;
    int *out;
    int ncl;
    __device__ Key key(int g) const {
        const int c = clus_of(pc, ncl, g);
        return ((Key)c << 32) | j_code(jp, pc[c], jcl[c], g);
    }
    __device__ void range(Key k, int, int &b, int &e) const {
        const PrepClus &P = pc[k >> 32];
        b = P.j0;
        e = P.j0 + P.ntile * kTile;
    }
    __device__ void put(int p, int g) const { out[p] = g; }
};
// Hilbert order of the i of a call in the box of their cluster's j set, so
// that the 64 i of a pass-1 wavefront are spatially close: far tiles then skip
// the screen for the whole wave, and the near band's FP64 pairs gather in
// fewer tiles.  The i data are gathered into that order.
struct IGather {
    const double *xi, *vi, *h2, *dtr;
    double *xs, *vs, *hs, *ds;
    int *perm;
    __device__ void put(int p, int i) const {
        perm[p] = i;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            xs[3 * (size_t)p + c] = xi[3 * (size_t)i + c];
            vs[3 * (size_t)p + c] = vi[3 * (size_t)i + c];
        }
        hs[p] = h2[i];
        ds[p] = dtr[i];
    }
};
struct ISort32 : IGather {
    using Key = unsigned;
    const JClus *jcl;
    __device__ Key key(int g) const { return i_code(xi, jcl[0], g); }
    __device__ void range(Key, int n, int &b, int &e) const { b = 0, e = n; }
};
struct ISort64 : IGather {
    using Key = unsigned long long;
    const JClus *jcl;
    const int *cl_i0;
    int ncl;
    __device__ Key key(int g) const {
        const int c = iclus_of(cl_i0, ncl, g);
        return ((Key)c << 32) | i_code(xi, jcl[c], g);
    }
    __device__ void range(Key k, int, int &b, int &e) const {
        b = cl_i0[k >> 32];
        e = cl_i0[(k >> 32) + 1];
    }
};

// One record per thread; each level a record finds its place in the pair of
// sorted pieces of w by binary search in the other piece (equal keys: the
// first piece's before the second's).
template <class S>
__global__ __launch_bounds__(kSortRun) void k_sort_runs(S s, int n,
                                                        typename S::Key *__restrict__ key,
                                                        int *__restrict__ val) {
    using Key = typename S::Key;
    __shared__ Key lk[2][kSortRun];
    __shared__ unsigned short lv[2][kSortRun];
    const int t = threadIdx.x;
    const int g = blockIdx.x * kSortRun + t;
    lk[0][t] = g < n ? s.key(g) : ~(Key)0;     // past the end: sorts last
    lv[0][t] = (unsigned short)t;
    __syncthreads();
#pragma unroll 1
    for (int w = 1, cur = 0; w < kSortRun; w <<= 1, cur ^= 1) {
        const Key k = lk[cur][t];
        const bool second = (t & w) != 0;
        const int pair = t & ~(2 * w - 1);
        const int other = pair + (second ? 0 : w);
        int pos = 0;                 // of 0..w - 1; the last record below
#pragma unroll 1
        for (int h = w >> 1; h >= 1; h >>= 1) {
            const Key o = lk[cur][other + pos + h - 1];
            pos += (second ? o <= k : o < k) ? h : 0;
        }
        const Key o = lk[cur][other + pos];
        pos += (second ? o <= k : o < k) ? 1 : 0;
        const int d = pair + (t & (w - 1)) + pos;
        lk[cur ^ 1][d] = k;
        lv[cur ^ 1][d] = lv[cur][t];
        __syncthreads();
    }
    constexpr int last = __builtin_ctz(kSortRun) & 1;
    if (g < n) {
        key[g] = lk[last][t];
        val[g] = blockIdx.x * kSortRun + lv[last][t];
    }
}

// One merge of runs of L, a workgroup per 64 records.  kLast: runs of the
// records' whole clusters, at most kSortWay, the result put by S; else
// kSortWay runs at a time.
template <class S, bool kLast>
__global__ __launch_bounds__(64 * kParts) void k_sort_merge(S s, int n, int L,
                                                   const typename S::Key *__restrict__ key,
                                                   const int *__restrict__ val,
                                                   typename S::Key *__restrict__ key_out,
                                                   int *__restrict__ val_out) {
    using Key = typename S::Key;
    __shared__ MergeLds<Key> lds;
    const int t = threadIdx.x, lane = t & 63;
    const int p0 = blockIdx.x * 64;
    const int p1 = min(p0 + 63, n - 1);
    const int p = min(p0 + lane, p1);
    const int own = p0 / L;
    const Key first = key[p0], last = key[p1], k = key[p];
    const int v = val[p];
    int r0, r1;
    if constexpr (kLast) {
        int beg, end, x;
        s.range(first, n, beg, x);
        s.range(last, n, x, end);
        r0 = beg / L;
        r1 = (end - 1) / L;
    } else {
        r0 = own & ~(kSortWay - 1);
        r1 = min(r0 + kSortWay - 1, (n - 1) / L);
    }
    merge_windows(lds, t, key, n, (long long)L, own, r0, r1, first, last);
    __syncthreads();
    merge_offsets(lds, t);
    __syncthreads();
    merge_load(lds, t, key, (long long)L, r0);
    __syncthreads();
    merge_ranks(lds, t, key, (long long)L, own, r0, k);
    __syncthreads();
    if (t >= 64 || p0 + t > p1) return;
    const int d = merge_place(lds, lane, (long long)L, own, r0, p);
    if constexpr (kLast) {
        s.put(d, v);
    } else {
        key_out[d] = k;
        val_out[d] = v;
    }
}

// Sort of n records, a cluster holding at most n_max of them, in the buffers
// A and B; s.put may write B's values.
template <class S>
static hipError_t sort_records(hipStream_t st, const S &s, int n, int n_max,
                               bool one, typename S::Key *key_a, int *val_a,
                               typename S::Key *key_b, int *val_b) {
    int merges = sort_merges(n, n_max, one);
    if (merges & 1) {             // the last merge reads A
        std::swap(key_a, key_b);
        std::swap(val_a, val_b);
    }
    hipLaunchKernelGGL((k_sort_runs<S>), dim3((n + kSortRun - 1) / kSortRun),
                       dim3(kSortRun), 0, st, s, n, key_a, val_a);
    const dim3 grid((n + 63) / 64);
    long long L = kSortRun;
    for (; merges > 0; --merges, L *= kSortWay) {
        hipLaunchKernelGGL((k_sort_merge<S, false>), grid, dim3(64 * kParts), 0, st, s, n,
                           (int)L, key_a, val_a, key_b, val_b);
        std::swap(key_a, key_b);
        std::swap(val_a, val_b);
    }
    hipLaunchKernelGGL((k_sort_merge<S, true>), grid, dim3(64 * kParts), 0, st, s, n,
                       (int)L, key_a, val_a, key_b, val_b);
    return hipGetLastError();
}

__global__ __launch_bounds__(64) void k_jtile(
    const JRec *__restrict__ jp, const PrepClus *__restrict__ pc, int ncl,
    const JClus *__restrict__ jcl, const int *__restrict__ sorted,
    JRec *__restrict__ jps, JRec32 *__restrict__ j32,
    JTile *__restrict__ tiles, int *__restrict__ jidx) {
    const int t = blockIdx.x;
    const int lane = threadIdx.x;
    const int p = t * kTile + lane;
    const int c = clus_of(pc, ncl, t * kTile);
    const PrepClus P = pc[c];
    const int g = sorted[p];
    const int local = g - P.j0;
    const bool real = local < P.nj;
    const JRec r = jp[g];
    jps[p] = r;
    jidx[p] = local;

    // The wavefront's lanes hold kTile / kVTile view tiles, one per
    // kVTile-lane segment: every reduction below stays within a segment.
    double v[6] = {r.x, r.y, r.z, r.vx, r.vy, r.vz};
    double cen[6];
    const unsigned long long seg_mask =
        kVTile >= 64 ? ~0ull : ((1ull << kVTile) - 1ull);
    const bool any =
        ((__ballot(real) >> (lane & ~(kVTile - 1))) & seg_mask) != 0;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const double lo = smin(real ? v[k] : INFINITY);
        const double hi = smax(real ? v[k] : -INFINITY);
        cen[k] = any ? 0.5 * lo + 0.5 * hi : 0.0;
    }
    JRec32 q;
    double e = 0.0, ev = 0.0, w = 1.0;
    if (real) {
        q.ox = (float)(r.x - cen[0]);
        q.oy = (float)(r.y - cen[1]);
        q.oz = (float)(r.z - cen[2]);
        q.ovx = (float)(r.vx - cen[3]);
        q.ovy = (float)(r.vy - cen[4]);
        q.ovz = (float)(r.vz - cen[5]);
        q.m = r.m32;
        const double ox = q.ox, oy = q.oy, oz = q.oz;
        const double ux = q.ovx, uy = q.ovy, uz = q.ovz;
        e = sqrt(ox * ox + oy * oy + oz * oz) * (1.0 + 1e-12);
        ev = sqrt(ux * ux + uy * uy + uz * uz) * (1.0 + 1e-12);
        const double mbar = jcl[c].mbar;
        if (mbar > 0.0 && r.m > mbar) {
            const double x = r.m / mbar;
            w = fmax(fmax(1.0, cbrt(x * x)), 1.4 * x / (double)kBand);
            w *= 1.0 + 1e-12;
        }
        q.w = up32(w);
    } else {
        // Padding: far away and massless, never screened.
        q.ox = q.oy = q.oz = 1.0e18f;
        q.ovx = q.ovy = q.ovz = 0.0f;
        q.m = 0.0f;
        q.w = 1.0f;
    }
    j32[p] = q;
    e = smax(e);
    ev = smax(ev);
    w = smax(real ? (double)q.w : 1.0);
    if ((lane & (kVTile - 1)) == 0) {
        JTile T;
        T.cx = cen[0];
        T.cy = cen[1];
        T.cz = cen[2];
        T.cu = cen[3];
        T.cv = cen[4];
        T.cw = cen[5];
        T.e = up32(e);
        T.ev = up32(ev);
        T.wmax = (float)w;
        T.eb = up32((double)kTileBand * (double)kTileBand * (double)T.e *
                    (double)T.e * (1.0 + 1e-12));
        tiles[t * (kTile / kVTile) + lane / kVTile] = T;
    }
}

__global__ void k_set_prepclus(PrepClus *pc, PrepClus v) { *pc = v; }

// Padding FP32 records and empty tiles over a whole allocation.
__global__ __launch_bounds__(256) void k_park_view(JRec32 *__restrict__ j32,
                                                   int n, JTile *__restrict__ tiles,
                                                   int ntile) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) {
        JRec32 q;
        q.ox = q.oy = q.oz = 1.0e18f;
        q.ovx = q.ovy = q.ovz = 0.0f;
        q.m = 0.0f;
        q.w = 1.0f;
        j32[k] = q;
    }
    if (k < ntile) {
        JTile T;
        T.cx = T.cy = T.cz = T.cu = T.cv = T.cw = 0.0;
        T.e = T.ev = 0.0f;
        T.wmax = 1.0f;
        T.eb = 0.0f;
        tiles[k] = T;
    }
}

hipError_t launch_isort_ens(hipStream_t st, const JClus *jcl, const int *cl_i0,
                            int ncl, const double *xi, const double *vi,
                            const double *h2, const double *dtr, int ni,
                            int ni_max, const ISortBufs &B) {
    if (ni <= 0) return hipSuccess;
    ISort64 s;
    static_cast<IGather &>(s) = {xi, vi, h2, dtr, B.xs, B.vs, B.hs, B.ds, B.perm};
    s.jcl = jcl;
    s.cl_i0 = cl_i0;
    s.ncl = ncl;
    return sort_records(st, s, ni, ni_max, ncl == 1, B.key64_in, B.val_in,
                        B.key64_out, B.perm);
}

hipError_t launch_isort(hipStream_t st, const JClus *jcl, const double *xi,
                        const double *vi, const double *h2, const double *dtr,
                        int ni, const ISortBufs &B) {
    if (ni <= 0) return hipSuccess;
    ISort32 s;
    static_cast<IGather &>(s) = {xi, vi, h2, dtr, B.xs, B.vs, B.hs, B.ds, B.perm};
    s.jcl = jcl;
    return sort_records(st, s, ni, ni, true, B.key_in, B.val_in, B.key_out, B.perm);
}

void launch_set_prepclus(hipStream_t st, PrepClus *pc, const PrepClus &v) {
    hipLaunchKernelGGL(k_set_prepclus, dim3(1), dim3(1), 0, st, pc, v);
}

void launch_park_view(hipStream_t st, JRec32 *j32, int n, JTile *tiles,
                      int ntile) {
    const int m = std::max(n, ntile);
    if (m <= 0) return;
    hipLaunchKernelGGL(k_park_view, dim3((m + 255) / 256), dim3(256), 0, st,
                       j32, n, tiles, ntile);
}

hipError_t launch_jprep(hipStream_t st, const JView &V, const PrepClus *pc,
                        int ncl, int nblk, int ntile_all, int ntile_max,
                        const PrepBufs &B) {
    if (ntile_all <= 0) return hipSuccess;
    const int n_all = ntile_all * kTile;
    hipLaunchKernelGGL(k_jstat1, dim3(nblk), dim3(256), 0, st, V.jp, pc, ncl,
                       B.part);
    hipLaunchKernelGGL(k_jstat2, dim3(ncl), dim3(256), 0, st, pc, ncl, nblk,
                       B.part, V.jcl);
    hipError_t rc;
    if (ncl == 1) {
        const JSort32 k = {V.jp, pc, V.jcl, B.val_out};
        rc = sort_records(st, k, n_all, n_all, true, (unsigned *)B.key_in, B.val_in,
                          (unsigned *)B.key_out, B.val_out);
    } else {
        const JSort64 k = {V.jp, pc, V.jcl, B.val_out, ncl};
        rc = sort_records(st, k, n_all, ntile_max * kTile, false, B.key_in, B.val_in,
                          B.key_out, B.val_out);
    }
    if (rc != hipSuccess) return rc;
    hipLaunchKernelGGL(k_jtile, dim3(ntile_all), dim3(64), 0, st, V.jp, pc, ncl,
                       V.jcl, B.val_out, V.jps, V.j32, V.tiles, V.jidx);
    return hipGetLastError();
}

}  // namespace gpunb
