// irr.hip -- irregular (neighbour) force on the device: a drop-in for the
// reference's irr_simd library (irr.avx.cpp:565-603, the Fortran interface
// irr_simd_open_/close_/profile_/set_jp_/set_list_/firr_vec_), plus batched
// entry points for callers that hold many particles at once.
//
// State in HBM: one 128-byte predictor record per particle (x0, v0, f = a/2,
// fd = jerk/6, m, t0 in FP64) and a neighbour table of nmax rows of lmax ints
// (count, then 0-based indices).  set_jp / set_list stage their data on the
// host and the next firr_vec scatters it with a kernel, so per-particle
// Fortran calls cost no device round trip.  A batched call
// (gpunb_irr_set_jp, gpunb_irr_set_lists) copies the caller's arrays as they
// are into one pinned block; the scatter kernel forms the records and rows
// from it, from a device copy whose upload starts in the batched call when
// the block is large, else from the pinned block itself.
//
// k_irr_force: one wavefront per active particle.  Every lane predicts its
// list members with the FP64 polynomial of xbpredall.f:18-26 (the same
// association as the oracle, no contraction), evaluates the pair in FP64 and
// accumulates in FP64; the wave then reduces in a fixed order.  When a call
// has more than three pairs per slot, k_irr_predict first predicts every
// slot once with the same function, and the members are read predicted.  The nearest
// member is the smallest r^2, ties to the smaller index (the reference's
// packed (r^2, index) minimum, irr.avx.cpp:317-320), returned 1-based, 0 for
// an empty list.  The reference evaluates the pairs in FP32 on double-single
// positions; FP64 costs little here (a few tens of pairs per particle).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <ctime>
#include <mutex>
#include <stdexcept>
#include <string>
#include <thread>
#include <vector>

#include "gpunb.h"
#include "gpunb_internal.h"

namespace gpunb_irr {

struct alignas(128) IRec {
    double x[3], v[3], f[3], fd[3];
    double m, t0;
    double pad[2];
};
static_assert(sizeof(IRec) == 128, "IRec must be 128 bytes");

#define ICHK(e)                                                               \
    do {                                                                      \
        hipError_t r_ = (e);                                                  \
        if (r_ != hipSuccess)                                                 \
            throw std::runtime_error(std::string(#e) + ": " +                 \
                                     hipGetErrorString(r_));                  \
    } while (0)

#define IREQ(c, msg)                                                          \
    do {                                                                      \
        if (!(c)) throw std::runtime_error(msg);                              \
    } while (0)

// Predicted position and velocity at t (xbpredall.f:18-26 association).
__device__ inline void predict(const IRec &r, double t, double *x, double *v) {
    const double s = t - r.t0;
    const double s1 = 1.5 * s;
    const double s2 = 2.0 * s;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        x[k] = ((r.fd[k] * s + r.f[k]) * s + r.v[k]) * s + r.x[k];
        v[k] = (r.fd[k] * s1 + r.f[k]) * s2 + r.v[k];
    }
}

constexpr int kWavesPerBlock = 4;
// Results of calls of at least kChunkMin bodies go to the host in kOutChunks
// parts, so the host moves one part into the caller's arrays while the next
// one crosses the host link.
constexpr int kOutChunks = 4;
constexpr int kChunkMin = 4 * 8192;
// Calls of up to kDirectMax bodies write their results to the mapped pinned
// buffers from the force kernel itself.
constexpr int kDirectMax = 2048;
// Pairs of a call from which members are read from records predicted once
// (N = 131072, 7.3M pairs: 0.150 against 0.176 ms of kernels; 1.9M pairs:
// 564 against 553 us a call, the extra launch costing what it saves).
constexpr long long kPreMin = 3000000;
// Batched calls of at least kBlockMin bodies are staged as blocks, at most
// kMaxBlocks of them at a time; a block of at least kUploadMin bytes is
// uploaded by the copy engine while the host goes on, a smaller one read from
// the host by the scatter kernel (8192 bodies, a call: 193 us with the line at
// 1 MiB, 181 at 512 KiB, 179 at 256 KiB and below).  Batches past the eighth
// are merged, as single calls are, into a block of each kind more; as many are
// kept at rest, or every such call would allocate them again (1000 bodies in
// batches of 100: 190 us a call with eight kept, 97 so).
constexpr int kBlockMin = 64;
constexpr size_t kMaxBlocks = 8;
constexpr size_t kMaxIdle = kMaxBlocks + 2;
constexpr size_t kUploadMin = 256 << 10;

// A particle predicted to the call's time: position, velocity, mass.
struct alignas(64) PRec {
    double x[3], v[3], m, pad;
};
static_assert(sizeof(PRec) == 64, "PRec must be 64 bytes");

// Every slot predicted once (the same function and operation order as the
// per-member prediction of k_irr_force<false>, so the values are the same).
__global__ __launch_bounds__(256) void k_irr_predict(int n, double t,
                                                     const IRec *__restrict__ jp,
                                                     PRec *__restrict__ pj) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const IRec &r = jp[k];
    PRec o;
    predict(r, t, o.x, o.v);
    o.m = r.m;
    o.pad = 0.0;
    pj[k] = o;
}

// PRE: members read from the predicted records pj (64 B each) instead of
// being predicted from jp (128 B each) member by member.
template <bool PRE>
__global__ __launch_bounds__(64 * kWavesPerBlock) void k_irr_force(
    int ni, const int *__restrict__ idx, double t, const IRec *__restrict__ jp,
    const PRec *__restrict__ pj, const int *__restrict__ list, int lstride,
    double *__restrict__ acc, double *__restrict__ jrk,
    int *__restrict__ nnbid) {
    const int lane = threadIdx.x & 63;
    const int q = blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    if (q >= ni) return;                  // uniform per wavefront
    const int i = idx[q];
    double xi[3], vi[3];
    if (PRE) {
        const PRec &p = pj[i];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            xi[c] = p.x[c];
            vi[c] = p.v[c];
        }
    } else {
        predict(jp[i], t, xi, vi);
    }
    const int *row = list + (size_t)i * lstride;
    const int nnb = row[0];
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, j0 = 0.0, j1 = 0.0, j2 = 0.0;
    double best = INFINITY;
    int bestj = INT_MAX;
    for (int k = lane; k < nnb; k += 64) {
        const int j = row[1 + k];
        double xj[3], vj[3], mj;
        if (PRE) {
            const PRec &p = pj[j];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                xj[c] = p.x[c];
                vj[c] = p.v[c];
            }
            mj = p.m;
        } else {
            predict(jp[j], t, xj, vj);
            mj = jp[j].m;
        }
        const double dx = xj[0] - xi[0], dy = xj[1] - xi[1], dz = xj[2] - xi[2];
        const double dvx = vj[0] - vi[0], dvy = vj[1] - vi[1], dvz = vj[2] - vi[2];
        double r2 = dx * dx;
        r2 = r2 + dy * dy;
        r2 = r2 + dz * dz;
        if (r2 < best || (r2 == best && j < bestj)) {
            best = r2;
            bestj = j;
        }
        if (r2 == 0.0) continue;
        const double rinv = 1.0 / sqrt(r2);
        const double rinv2 = rinv * rinv;
        const double mr3 = mj * rinv2 * rinv;
        double rv = dx * dvx;
        rv = rv + dy * dvy;
        rv = rv + dz * dvz;
        const double alpha = -3.0 * rv * rinv2;
        a0 += mr3 * dx;
        a1 += mr3 * dy;
        a2 += mr3 * dz;
        j0 += mr3 * (dvx + alpha * dx);
        j1 += mr3 * (dvy + alpha * dy);
        j2 += mr3 * (dvz + alpha * dz);
    }
    for (int o = 32; o >= 1; o >>= 1) {
        a0 += __shfl_xor(a0, o);
        a1 += __shfl_xor(a1, o);
        a2 += __shfl_xor(a2, o);
        j0 += __shfl_xor(j0, o);
        j1 += __shfl_xor(j1, o);
        j2 += __shfl_xor(j2, o);
        const double ob = __shfl_xor(best, o);
        const int oj = __shfl_xor(bestj, o);
        if (ob < best || (ob == best && oj < bestj)) {
            best = ob;
            bestj = oj;
        }
    }
    // Every lane holds the sums: one store per vector.
    if (lane < 3) {
        acc[3 * (size_t)q + lane] = lane == 0 ? a0 : lane == 1 ? a1 : a2;
        jrk[3 * (size_t)q + lane] = lane == 0 ? j0 : lane == 1 ? j1 : j2;
    }
    if (lane == 0) nnbid[q] = bestj == INT_MAX ? 0 : bestj + 1;
}

// Staged data -> its slots, and the active indices of the call to the device,
// in one launch: workgroups [0, bj) take 256 records each, [bj, bj + bl) four
// list rows each (one wavefront per row), the rest 256 indices each.
//   records: arrays x, v, f, fd [n][3], m, t0 [n] one after another (soa) and
//            the slots; the caller's arrays as they are.
//   rows:    hdr[3r] = slot, hdr[3r+1] = offset of the row in flat,
//            hdr[3r+2] = count; flat: 0-based members.
struct StageArgs {
    int nj, nr, ni;
    unsigned bj, bl;
    const double *soa;
    const int *slot;
    IRec *jp;
    const int *hdr, *flat;
    int *list;
    int lstride;
    const int *idx_src;
    int *idx;
};

__global__ __launch_bounds__(256) void k_irr_stage(StageArgs s) {
    const unsigned b = blockIdx.x;
    if (b < s.bj) {
        const int k = b * 256 + threadIdx.x;
        if (k >= s.nj) return;
        const size_t n = (size_t)s.nj;
        IRec r;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            r.x[c] = s.soa[3 * (size_t)k + c];
            r.v[c] = s.soa[3 * (n + k) + c];
            r.f[c] = s.soa[3 * (2 * n + k) + c];
            r.fd[c] = s.soa[3 * (3 * n + k) + c];
        }
        r.m = s.soa[12 * n + k];
        r.t0 = s.soa[13 * n + k];
        r.pad[0] = r.pad[1] = 0.0;
        s.jp[s.slot[k]] = r;
    } else if (b < s.bj + s.bl) {
        const int lane = threadIdx.x & 63;
        const int r = (int)(b - s.bj) * 4 + (int)(threadIdx.x >> 6);
        if (r >= s.nr) return;
        const int slot = s.hdr[3 * r], off = s.hdr[3 * r + 1],
                  cnt = s.hdr[3 * r + 2];
        int *row = s.list + (size_t)slot * s.lstride;
        if (lane == 0) row[0] = cnt;
        for (int k = lane; k < cnt; k += 64) row[1 + k] = s.flat[off + k];
    } else {
        const int q = (int)(b - s.bj - s.bl) * 256 + threadIdx.x;
        if (q < s.ni) s.idx[q] = s.idx_src[q];
    }
}

// Device -> mapped pinned host copy of three ranges of n16[b] 16-byte units,
// blockIdx.y selecting the range: one part of a call's acceleration, jerk and
// nearest-neighbour results.
struct Ranges {
    const uint4 *src[3];
    uint4 *dst[3];
    size_t n16[3];
};

__global__ __launch_bounds__(256) void k_irr_to_host(Ranges r) {
    const int b = blockIdx.y;
    const uint4 *__restrict__ src = r.src[b];
    uint4 *__restrict__ dst = r.dst[b];
    const size_t n16 = r.n16[b];
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < n16;
         k += stride)
        dst[k] = src[k];
}

// Grow-only device / pinned host buffers.
template <class T>
struct DBuf {
    T *p = nullptr;
    size_t cap = 0;
    void ensure(size_t n) {
        if (n <= cap) return;
        release();
        ICHK(hipMalloc((void **)&p, std::max<size_t>(n, 1) * sizeof(T)));
        cap = n;
    }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        cap = 0;
    }
};

template <class T>
struct HBuf {
    T *p = nullptr;
    size_t cap = 0;
    void ensure(size_t n) {
        if (n <= cap) return;
        release();
        ICHK(hipHostMalloc((void **)&p, std::max<size_t>(n, 1) * sizeof(T)));
        cap = n;
    }
    void release() {
        if (p) (void)hipHostFree(p);
        p = nullptr;
        cap = 0;
    }
};

// The data of one batched call (or of the merged per-particle calls), pinned:
// records as the arrays and slots of k_irr_stage, rows as its headers and
// members.
struct Block {
    bool rows = false;
    int n = 0;
    size_t nflat = 0;
    HBuf<char> h;
    DBuf<char> d;
    const char *src = nullptr;   // where the device reads it
    size_t ints_at() const { return rows ? 0 : (size_t)n * 14 * sizeof(double); }
    size_t bytes() const {
        return ints_at() + (rows ? 3 * (size_t)n + nflat : (size_t)n) * sizeof(int);
    }
    double *soa() { return (double *)h.p; }
    int *ints() { return (int *)(h.p + ints_at()); }
    void release() {
        h.release();
        d.release();
    }
};

struct State {
    bool open = false;
    int nmax = 0, lstride = 0;
    int dev = 0;
    hipStream_t st = nullptr;
    DBuf<IRec> jp;
    DBuf<PRec> pj;                            // slots predicted to a call's t
    DBuf<int> list;
    // staging (host), latest data per slot wins
    std::vector<IRec> jp_rec;
    std::vector<int> jp_addr, jp_slot;        // jp_slot[a] = staged index or -1
    std::vector<int> ls_hdr, ls_flat, ls_slot;
    std::vector<int> nnb;                     // host mirror of the counts
    std::vector<int> seen;                    // slot marks of a batched call
    int seen_mark = 0;
    // Blocks staged, in call order (older than anything staged per particle),
    // and blocks at rest, kept for the next calls.
    std::vector<Block *> blocks, idle;
    HBuf<int> h_idx;
    DBuf<int> d_idx;
    // results of a call: acc[ni_pad][3], jerk[ni_pad][3] (d_out, h_out) and
    // the nearest neighbours[ni_pad] (d_nn, h_nn), ni_pad = ni rounded up to
    // 64, so every part of them starts on a 16-byte boundary
    DBuf<double> d_out;
    DBuf<int> d_nn;
    HBuf<double> h_out;
    HBuf<int> h_nn;
    // profile
    long long ncall = 0, nsteps = 0, ninter = 0;
    double t_force = 0.0;
    // k_irr_force of the last call, timed on the stream
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    double last_kernel_ms = 0.0;
    hipEvent_t part[kOutChunks] = {};        // after the copy of part c
};
State I;

// Staging.  The reference's host calls set_jp / set_list for every particle
// inside an OpenMP parallel loop (intgrt.F:200-205), so they must be safe to
// call concurrently: each thread appends to its own buffer, and the next
// firr_vec (called from one thread, with no staging running) merges all
// buffers, keeping the last value staged for each particle.  Batched calls
// stage blocks, under the lock; one that follows per-particle calls which no
// firr_vec has merged yet goes the per-particle way, so blocks are always the
// older data.
struct Stage {
    std::vector<IRec> rec;
    std::vector<int> rec_addr;   // 0-based slot per record
    std::vector<int> hdr;        // (slot, offset in flat, count) per row
    std::vector<int> flat;       // members, 0-based
    std::atomic<bool> used{false};
    void clear() {
        rec.clear();
        rec_addr.clear();
        hdr.clear();
        flat.clear();
        used.store(false, std::memory_order_relaxed);
    }
};
std::mutex g_stage_mu;
std::vector<Stage *> g_stages;   // kept for the life of the process
thread_local Stage *t_stage = nullptr;

Stage &my_stage() {
    if (!t_stage) {
        Stage *st = new Stage;
        std::lock_guard<std::mutex> g(g_stage_mu);
        g_stages.push_back(st);
        t_stage = st;
    }
    return *t_stage;
}

void stage_jp(int a, const double *x, const double *v, const double *f,
              const double *fd, double m, double t0) {
    IREQ(a >= 1 && a <= I.nmax, "address out of range [1, nmax]");
    IRec r{};
    for (int k = 0; k < 3; ++k) {
        r.x[k] = x[k];
        r.v[k] = v[k];
        r.f[k] = f[k];
        r.fd[k] = fd[k];
    }
    r.m = m;
    r.t0 = t0;
    Stage &st = my_stage();
    st.used.store(true, std::memory_order_release);
    st.rec.push_back(r);
    st.rec_addr.push_back(a - 1);
}

// nb: 1-based member indices.
void stage_list(int a, int cnt, const int *nb) {
    IREQ(a >= 1 && a <= I.nmax, "address out of range [1, nmax]");
    IREQ(cnt >= 0 && cnt <= I.lstride - 1, "list longer than lmax - 1");
    for (int k = 0; k < cnt; ++k)
        IREQ(nb[k] >= 1 && nb[k] <= I.nmax, "list member out of range [1, nmax]");
    Stage &st = my_stage();
    st.used.store(true, std::memory_order_release);
    st.hdr.push_back(a - 1);
    st.hdr.push_back((int)st.flat.size());
    st.hdr.push_back(cnt);
    for (int k = 0; k < cnt; ++k) st.flat.push_back(nb[k] - 1);
}

// All threads' staged data into I.jp_rec / jp_addr / ls_hdr / ls_flat, the
// last value per particle winning (a superseded row keeps slot -1).
void merge_stages() {
    std::lock_guard<std::mutex> g(g_stage_mu);
    for (Stage *st : g_stages) {
        for (size_t k = 0; k < st->rec.size(); ++k) {
            const int s = st->rec_addr[k];
            if (I.jp_slot[s] >= 0) {
                I.jp_rec[I.jp_slot[s]] = st->rec[k];
            } else {
                I.jp_slot[s] = (int)I.jp_rec.size();
                I.jp_rec.push_back(st->rec[k]);
                I.jp_addr.push_back(s);
            }
        }
        for (size_t r = 0; r < st->hdr.size(); r += 3) {
            const int s = st->hdr[r], off = st->hdr[r + 1], cnt = st->hdr[r + 2];
            if (I.ls_slot[s] >= 0) I.ls_hdr[3 * I.ls_slot[s]] = -1;
            I.ls_slot[s] = (int)(I.ls_hdr.size() / 3);
            I.ls_hdr.push_back(s);
            I.ls_hdr.push_back((int)I.ls_flat.size());
            I.ls_hdr.push_back(cnt);
            I.ls_flat.insert(I.ls_flat.end(), st->flat.begin() + off,
                             st->flat.begin() + off + cnt);
            I.nnb[s] = cnt;
        }
        st->clear();
    }
}

void clear_stages() {
    std::lock_guard<std::mutex> g(g_stage_mu);
    for (Stage *st : g_stages) st->clear();
    for (Block *b : I.blocks) I.idle.push_back(b);
    I.blocks.clear();
}

// Copies of more than kSplitMin bytes are split over four threads: one core
// moves them at a fraction of the memory's rate, but starting the threads
// takes about 30 us (8192 bodies, a call: 192 us unsplit, 239 split; 131072
// bodies staged and evaluated: 10.3 ms with a record and row at a time through
// the per-particle buffers, 1.7 ms so).
constexpr size_t kSplitMin = 2 << 20;
template <class F>
void split(size_t n, size_t bytes, F f) {
    constexpr int T = 4;
    std::thread th[T - 1];
    size_t done = 0;
    int started = 0;
    if (bytes >= kSplitMin) {
        try {
            for (; started < T - 1; ++started) {
                const size_t lo = done, hi = n * (started + 1) / T;
                th[started] = std::thread([=] { f(lo, hi); });
                done = hi;
            }
        } catch (const std::exception &) {
            // No more threads, or no memory for one: this one does the rest.
        }
    }
    f(done, n);
    for (int k = 0; k < started; ++k) th[k].join();
}

// A block that can hold n records, or n rows of nflat members in all, from the
// idle ones or new.
Block *take_block(bool rows, int n, size_t nflat) {
    Block *b = nullptr;
    if (!I.idle.empty()) {
        // The one whose buffer fits best: the smallest that is large enough,
        // else the largest.
        Block w;
        w.rows = rows;
        w.n = n;
        w.nflat = nflat;
        const size_t need = w.bytes();
        size_t at = 0;
        for (size_t k = 1; k < I.idle.size(); ++k) {
            const size_t c = I.idle[k]->h.cap, a = I.idle[at]->h.cap;
            if (a < need ? c > a : (c >= need && c < a)) at = k;
        }
        b = I.idle[at];
        I.idle.erase(I.idle.begin() + at);
    } else {
        b = new Block;
    }
    b->rows = rows;
    b->n = n;
    b->nflat = nflat;
    b->src = nullptr;
    try {
        b->h.ensure(b->bytes());
    } catch (...) {
        I.idle.push_back(b);
        throw;
    }
    return b;
}

// Start the upload of a large block; small ones are read where they are.
void place_block(Block *b) {
    const size_t n = b->bytes();
    if (n >= kUploadMin) {
        int cur = 0;
        ICHK(hipGetDevice(&cur));
        if (cur != I.dev) ICHK(hipSetDevice(I.dev));
        hipError_t rc = hipSuccess;
        try {
            b->d.ensure(n);
            rc = hipMemcpyAsync(b->d.p, b->h.p, n, hipMemcpyHostToDevice, I.st);
        } catch (...) {
            if (cur != I.dev) (void)hipSetDevice(cur);
            throw;
        }
        if (cur != I.dev) ICHK(hipSetDevice(cur));
        ICHK(rc);
        b->src = b->d.p;
    } else {
        void *p = nullptr;
        ICHK(hipHostGetDevicePointer(&p, b->h.p, 0));
        b->src = (const char *)p;
    }
}

// Stage a block that fill fills.  After an error nothing of it is staged: it is
// at rest, and what it was to hold stays where the caller has it.
template <class F>
void stage_block(bool rows, int n, size_t nflat, F fill) {
    I.blocks.reserve(I.blocks.size() + 1);
    Block *b = take_block(rows, n, nflat);
    try {
        fill(b);
        place_block(b);
    } catch (...) {
        I.idle.push_back(b);
        throw;
    }
    I.blocks.push_back(b);
}

// Whether a batched call of n bodies is staged as a block (lock held).
bool block_ok(int n) {
    if (n < kBlockMin || I.blocks.size() >= kMaxBlocks) return false;
    if (!I.jp_rec.empty() || !I.ls_hdr.empty()) return false;
    for (Stage *st : g_stages)
        if (st->used.load(std::memory_order_acquire)) return false;
    return true;
}

// Addresses of a batched call in range (an error otherwise) and each listed
// once (false otherwise: the per-particle way keeps the last).
bool addresses_once(int n, const int *addr) {
    bool ascending = true, range = true;
    for (int q = 0; q < n; ++q) {
        range = range && addr[q] >= 1 && addr[q] <= I.nmax;
        ascending = ascending && (q == 0 || addr[q] > addr[q - 1]);
    }
    IREQ(range, "address out of range [1, nmax]");
    if (ascending) return true;
    if (++I.seen_mark == INT_MAX) {
        std::fill(I.seen.begin(), I.seen.end(), 0);
        I.seen_mark = 1;
    }
    for (int q = 0; q < n; ++q) {
        int &m = I.seen[addr[q] - 1];
        if (m == I.seen_mark) return false;
        m = I.seen_mark;
    }
    return true;
}

bool block_jp(int n, const int *addr, const double *x, const double *v,
              const double *f, const double *fd, const double *m,
              const double *t0) {
    std::lock_guard<std::mutex> g(g_stage_mu);
    if (!block_ok(n) || !addresses_once(n, addr)) return false;
    stage_block(false, n, 0, [&](Block *b) {
        double *h = b->soa();
        int *slot = b->ints();
        const size_t N = (size_t)n;
        split(N, b->bytes(), [=](size_t lo, size_t hi) {
            const double *v3[4] = {x, v, f, fd};
            for (int c = 0; c < 4; ++c)
                memcpy(h + 3 * (c * N + lo), v3[c] + 3 * lo,
                       3 * (hi - lo) * sizeof(double));
            memcpy(h + 12 * N + lo, m + lo, (hi - lo) * sizeof(double));
            memcpy(h + 13 * N + lo, t0 + lo, (hi - lo) * sizeof(double));
            for (size_t q = lo; q < hi; ++q) slot[q] = addr[q] - 1;
        });
    });
    return true;
}

bool block_lists(int n, const int *addr, const int *nnb, const int *members) {
    std::lock_guard<std::mutex> g(g_stage_mu);
    if (!block_ok(n)) return false;
    size_t nf = 0;
    for (int q = 0; q < n; ++q) {
        IREQ(nnb[q] >= 0 && nnb[q] <= I.lstride - 1, "list longer than lmax - 1");
        nf += (size_t)nnb[q];
    }
    if (nf > (size_t)INT_MAX || !addresses_once(n, addr)) return false;
    stage_block(true, n, nf, [&](Block *b) {
        int *hdr = b->ints(), *flat = hdr + 3 * (size_t)n;
        int off = 0;
        for (int q = 0; q < n; ++q) {
            hdr[3 * (size_t)q] = addr[q] - 1;
            hdr[3 * (size_t)q + 1] = off;
            hdr[3 * (size_t)q + 2] = nnb[q];
            off += nnb[q];
        }
        std::atomic<bool> bad{false};
        std::atomic<bool> *pbad = &bad;
        const unsigned nmax = (unsigned)I.nmax;
        split(nf, nf * sizeof(int), [=](size_t lo, size_t hi) {
            unsigned out = 0;
            for (size_t k = lo; k < hi; ++k) {
                const int j = members[k] - 1;
                out |= (unsigned)j >= nmax;
                flat[k] = j;
            }
            if (out) pbad->store(true, std::memory_order_relaxed);
        });
        IREQ(!bad.load(), "list member out of range [1, nmax]");
    });
    for (int q = 0; q < n; ++q) I.nnb[addr[q] - 1] = nnb[q];
    return true;
}

// What the per-particle calls staged, as blocks.
void block_merged() {
    const size_t nj = I.jp_rec.size();
    if (nj) {
        stage_block(false, (int)nj, 0, [&](Block *b) {
            double *h = b->soa();
            for (size_t k = 0; k < nj; ++k) {
                const IRec &r = I.jp_rec[k];
                for (int c = 0; c < 3; ++c) {
                    h[3 * k + c] = r.x[c];
                    h[3 * (nj + k) + c] = r.v[c];
                    h[3 * (2 * nj + k) + c] = r.f[c];
                    h[3 * (3 * nj + k) + c] = r.fd[c];
                }
                h[12 * nj + k] = r.m;
                h[13 * nj + k] = r.t0;
            }
            memcpy(b->ints(), I.jp_addr.data(), nj * sizeof(int));
        });
        for (int s : I.jp_addr) I.jp_slot[s] = -1;
        I.jp_rec.clear();
        I.jp_addr.clear();
    }
    size_t nr = 0;
    for (size_t r = 0; r < I.ls_hdr.size(); r += 3) nr += I.ls_hdr[r] >= 0;
    if (nr) {
        stage_block(true, (int)nr, I.ls_flat.size(), [&](Block *b) {
            int *hdr = b->ints();
            for (size_t r = 0; r < I.ls_hdr.size(); r += 3)
                if (I.ls_hdr[r] >= 0) {
                    memcpy(hdr, I.ls_hdr.data() + r, 3 * sizeof(int));
                    hdr += 3;
                }
            memcpy(hdr, I.ls_flat.data(), I.ls_flat.size() * sizeof(int));
        });
        for (size_t r = 0; r < I.ls_hdr.size(); r += 3)
            if (I.ls_hdr[r] >= 0) I.ls_slot[I.ls_hdr[r]] = -1;
    }
    I.ls_hdr.clear();
    I.ls_flat.clear();
}

double wtime() {
    struct timespec ts;
    clock_gettime(CLOCK_MONOTONIC, &ts);
    return ts.tv_sec + 1e-9 * ts.tv_nsec;
}

bool quiet() {
    const char *q = getenv("GPUNB_QUIET");
    return q && *q && *q != '0';
}

void do_open(int nmax, int lmax, int rank) {
    if (I.open) {
        fprintf(stderr, "irr_simd: it is already open\n");
        return;
    }
    IREQ(nmax > 0, "irr_simd_open: nmax must be > 0");
    IREQ(lmax >= 1, "irr_simd_open: lmax must be >= 1");
    ICHK(hipStreamCreateWithFlags(&I.st, hipStreamNonBlocking));
    ICHK(hipEventCreate(&I.ev0));
    ICHK(hipEventCreate(&I.ev1));
    for (int c = 0; c < kOutChunks; ++c)
        ICHK(hipEventCreateWithFlags(&I.part[c], hipEventDisableTiming));
    I.last_kernel_ms = 0.0;
    ICHK(hipGetDevice(&I.dev));
    I.nmax = nmax;
    I.lstride = lmax;
    I.jp.ensure((size_t)nmax);
    I.list.ensure((size_t)nmax * lmax);
    // Empty lists and a parked predictor state until the caller sets them.
    ICHK(hipMemsetAsync(I.list.p, 0, (size_t)nmax * lmax * sizeof(int), I.st));
    ICHK(hipMemsetAsync(I.jp.p, 0, (size_t)nmax * sizeof(IRec), I.st));
    ICHK(hipStreamSynchronize(I.st));
    I.jp_slot.assign(nmax, -1);
    I.ls_slot.assign(nmax, -1);
    I.nnb.assign(nmax, 0);
    I.seen.assign(nmax, 0);
    I.seen_mark = 0;
    I.jp_rec.clear();
    I.jp_addr.clear();
    I.ls_hdr.clear();
    I.ls_flat.clear();
    clear_stages();
    I.ncall = I.nsteps = I.ninter = 0;
    I.t_force = 0.0;
    I.open = true;
    if (!quiet())
        fprintf(stderr, "# Opening irr_simd lib. MI355X ver. - rank: %d; nmax: %d, lmax: %d\n",
                rank, nmax, lmax);
}

void do_close(int rank) {
    if (!I.open) {
        fprintf(stderr, "irr_simd: it is already close\n");
        return;
    }
    ICHK(hipStreamSynchronize(I.st));
    I.jp.release();
    I.pj.release();
    I.list.release();
    I.d_idx.release();
    I.d_out.release();
    I.d_nn.release();
    I.h_idx.release();
    clear_stages();
    for (Block *b : I.idle) {
        b->release();
        delete b;
    }
    I.idle.clear();
    I.h_out.release();
    I.h_nn.release();
    (void)hipEventDestroy(I.ev0);
    (void)hipEventDestroy(I.ev1);
    I.ev0 = I.ev1 = nullptr;
    for (int c = 0; c < kOutChunks; ++c) {
        (void)hipEventDestroy(I.part[c]);
        I.part[c] = nullptr;
    }
    (void)hipStreamDestroy(I.st);
    I.st = nullptr;
    I.open = false;
    if (!quiet()) fprintf(stderr, "Closing irr_simd lib. MI355X ver. - rank: %d\n", rank);
}

// Scatter the staged blocks, then (ni > 0) the force of addr[] at t; the host
// waits only for each part of the results (one part below kChunkMin bodies).
void flush_and_force(double t, int ni, const int *addr, double *acc,
                     double *jrk, int *nnbid) {
    I.h_idx.ensure((size_t)ni);
    I.d_idx.ensure((size_t)ni);
    merge_stages();
    long long pairs = 0;
    for (int q = 0; q < ni; ++q) {
        const int a = addr[q];
        IREQ(a >= 1 && a <= I.nmax, "address out of range [1, nmax]");
        I.h_idx.p[q] = a - 1;
        pairs += I.nnb[a - 1];
    }
    block_merged();
    // One launch per pair of a record and a row block, in staging order (a
    // later block overwrites an earlier one's slots); the last one also
    // brings the call's indices.
    StageArgs s = {};
    s.jp = I.jp.p;
    s.list = I.list.p;
    s.lstride = I.lstride;
    auto launch = [&] {
        s.bj = (unsigned)((s.nj + 255) / 256);
        s.bl = (unsigned)((s.nr + 3) / 4);
        const unsigned nb = s.bj + s.bl + (unsigned)((s.ni + 255) / 256);
        if (nb) hipLaunchKernelGGL(k_irr_stage, dim3(nb), dim3(256), 0, I.st, s);
        s.nj = s.nr = 0;
    };
    for (Block *b : I.blocks) {
        if (b->rows ? s.nr : s.nj) launch();
        if (b->rows) {
            s.nr = b->n;
            s.hdr = (const int *)b->src;
            s.flat = s.hdr + 3 * (size_t)b->n;
        } else {
            s.nj = b->n;
            s.soa = (const double *)b->src;
            s.slot = (const int *)(b->src + b->ints_at());
        }
    }
    if (ni > 0) {
        void *hi = nullptr;
        ICHK(hipHostGetDevicePointer(&hi, I.h_idx.p, 0));
        s.ni = ni;
        s.idx_src = (const int *)hi;
        s.idx = I.d_idx.p;
    }
    launch();
    if (ni > 0) {
        const size_t np = ((size_t)ni + 63) & ~(size_t)63;
        I.d_out.ensure(np * 6);
        I.d_nn.ensure(np);
        I.h_out.ensure(np * 6);
        I.h_nn.ensure(np);
        void *ho = nullptr, *hn = nullptr;
        ICHK(hipHostGetDevicePointer(&ho, I.h_out.p, 0));
        ICHK(hipHostGetDevicePointer(&hn, I.h_nn.p, 0));
        const bool direct = ni <= kDirectMax;
        double *out = direct ? (double *)ho : I.d_out.p;
        int *nn = direct ? (int *)hn : I.d_nn.p;
        // Predict every slot once when the call's pairs are many and outnumber
        // the slots threefold: each member then costs a 64-byte read instead of a
        // 128-byte read and its prediction.
        const bool pre = pairs > 3LL * I.nmax && pairs > kPreMin;
        // Event records around the kernels, not hipExtLaunchKernel's: waiting
        // for a call whose launch carries both events takes 15 us longer (20
        // bodies: 24 and 40 us a call, 8192: 217 and 217 us).
        if (pre) I.pj.ensure((size_t)I.nmax);
        ICHK(hipEventRecord(I.ev0, I.st));
        if (pre)
            hipLaunchKernelGGL(k_irr_predict, dim3((unsigned)((I.nmax + 255) / 256)),
                               dim3(256), 0, I.st, I.nmax, t, I.jp.p, I.pj.p);
        const dim3 grid((unsigned)((ni + kWavesPerBlock - 1) / kWavesPerBlock));
        if (pre)
            hipLaunchKernelGGL(k_irr_force<true>, grid, dim3(64 * kWavesPerBlock),
                               0, I.st, ni, I.d_idx.p, t, I.jp.p, I.pj.p, I.list.p,
                               I.lstride, out, out + 3 * np, nn);
        else
            hipLaunchKernelGGL(k_irr_force<false>, grid, dim3(64 * kWavesPerBlock),
                               0, I.st, ni, I.d_idx.p, t, I.jp.p,
                               (const PRec *)nullptr, I.list.p, I.lstride, out,
                               out + 3 * np, nn);
        ICHK(hipEventRecord(I.ev1, I.st));
        // Part c: bodies q0 .. q0 + nq (q0 a multiple of 64), copied by one
        // launch to the mapped h_out / h_nn; a byte count is rounded up to
        // 16, which stays inside the padded arrays.
        const int nchunk = ni >= kChunkMin ? kOutChunks : 1;
        const int per = (int)((((size_t)ni + nchunk - 1) / nchunk + 63) & ~(size_t)63);
        for (int c = 0; c < nchunk && !direct; ++c) {
            const size_t q0 = (size_t)c * per;
            if (q0 >= (size_t)ni) break;
            const size_t nq = std::min<size_t>(ni - q0, per);
            Ranges r;
            r.src[0] = (const uint4 *)(I.d_out.p + 3 * q0);
            r.dst[0] = (uint4 *)((double *)ho + 3 * q0);
            r.src[1] = (const uint4 *)(I.d_out.p + 3 * (np + q0));
            r.dst[1] = (uint4 *)((double *)ho + 3 * (np + q0));
            r.src[2] = (const uint4 *)(I.d_nn.p + q0);
            r.dst[2] = (uint4 *)((int *)hn + q0);
            r.n16[0] = r.n16[1] = (24 * nq + 15) / 16;
            r.n16[2] = (4 * nq + 15) / 16;
            const unsigned gx = (unsigned)std::min<size_t>(512, (r.n16[0] + 255) / 256);
            hipLaunchKernelGGL(k_irr_to_host, dim3(gx, 3), dim3(256), 0, I.st, r);
            ICHK(hipEventRecord(I.part[c], I.st));
        }
        ICHK(hipGetLastError());
        // Each part into the caller's arrays once its copy is done (the
        // uploads, the force and every earlier copy were before it on I.st).
        for (int c = 0; c < nchunk; ++c) {
            const size_t q0 = (size_t)c * per;
            if (q0 >= (size_t)ni) break;
            const size_t nq = std::min<size_t>(ni - q0, per);
            if (direct)
                ICHK(hipStreamSynchronize(I.st));
            else
                ICHK(hipEventSynchronize(I.part[c]));
            memcpy(acc + 3 * q0, I.h_out.p + 3 * q0, 3 * nq * sizeof(double));
            memcpy(jrk + 3 * q0, I.h_out.p + 3 * (np + q0), 3 * nq * sizeof(double));
            if (nnbid) memcpy(nnbid + q0, I.h_nn.p + q0, nq * sizeof(int));
        }
        float ms = 0.0f;
        ICHK(hipEventElapsedTime(&ms, I.ev0, I.ev1));
        I.last_kernel_ms = ms;
        I.ncall++;
        I.nsteps += ni;
        I.ninter += pairs;
    } else {
        ICHK(hipGetLastError());
        // The pinned blocks are reused by the next calls.
        if (!I.blocks.empty()) ICHK(hipStreamSynchronize(I.st));
    }
    std::lock_guard<std::mutex> g(g_stage_mu);
    for (Block *b : I.blocks) I.idle.push_back(b);
    I.blocks.clear();
    while (I.idle.size() > kMaxIdle) {
        I.idle.back()->release();
        delete I.idle.back();
        I.idle.pop_back();
    }
}

void firr(double t, int ni, const int *addr, double *acc, double *jrk,
          int *nnbid) {
    IREQ(I.open, "irr_simd is not open");
    IREQ(ni >= 0, "ni must be >= 0");
    const double w0 = wtime();
    flush_and_force(t, ni, addr, acc, jrk, nnbid);
    I.t_force += wtime() - w0;
}

void profile(int rank) {
    if (!I.open || quiet()) return;
    const double gf = I.t_force > 0 ? 60.0 * (double)I.ninter * 1e-9 / I.t_force : 0.0;
    fprintf(stderr,
            "[R.%d MI355X Irr.F ] Ncall: %lld <NI>: %lld <NB>: %f grav: %f s, %f Gflops, %f usec\n",
            rank, I.ncall, I.ncall ? I.nsteps / I.ncall : 0,
            I.nsteps ? (double)I.ninter / I.nsteps : 0.0, I.t_force, gf,
            I.ncall ? 1e6 * I.t_force / I.ncall : 0.0);
    I.ncall = I.nsteps = I.ninter = 0;
    I.t_force = 0.0;
}

}  // namespace gpunb_irr

using namespace gpunb_irr;

#define IRR_EXPORT __attribute__((visibility("default")))

extern "C" {

IRR_EXPORT void irr_simd_open_(int *nmax, int *lmax, int *rank) {
    gpunb::run_guarded("irr_simd_open_", [&] { do_open(*nmax, *lmax, *rank); });
}

IRR_EXPORT void irr_simd_close_(int *rank) {
    gpunb::run_guarded("irr_simd_close_", [&] { do_close(*rank); });
}

IRR_EXPORT void irr_simd_profile_(int *rank) {
    gpunb::run_guarded("irr_simd_profile_", [&] { profile(*rank); });
}

IRR_EXPORT void irr_simd_set_jp_(int *addr, double pos[3], double vel[3],
                                 double acc2[3], double jrk6[3], double *mass,
                                 double *time) {
    gpunb::run_guarded("irr_simd_set_jp_", [&] {
        IREQ(I.open, "irr_simd is not open");
        stage_jp(*addr, pos, vel, acc2, jrk6, *mass, *time);
    });
}

IRR_EXPORT void irr_simd_set_list_(int *addr, int *nblist) {
    gpunb::run_guarded("irr_simd_set_list_", [&] {
        IREQ(I.open, "irr_simd is not open");
        stage_list(*addr, nblist[0], nblist + 1);
    });
}

IRR_EXPORT void irr_simd_firr_vec_(double *ti, int *ni, int addr[],
                                   double acc[][3], double jrk[][3],
                                   int nnbid[]) {
    gpunb::run_guarded("irr_simd_firr_vec_", [&] {
        firr(*ti, *ni, addr, &acc[0][0], &jrk[0][0], nnbid);
    });
}

IRR_EXPORT int gpunb_irr_set_jp(int n, const int *addr, const double *x,
                                const double *v, const double *f,
                                const double *fd, const double *m,
                                const double *t0) {
    return gpunb::run_guarded("gpunb_irr_set_jp", [&] {
        IREQ(I.open, "irr_simd is not open");
        if (block_jp(n, addr, x, v, f, fd, m, t0)) return;
        for (int q = 0; q < n; ++q)
            stage_jp(addr[q], x + 3 * (size_t)q, v + 3 * (size_t)q,
                     f + 3 * (size_t)q, fd + 3 * (size_t)q, m[q], t0[q]);
    });
}

IRR_EXPORT double gpunb_irr_kernel_ms(void) { return I.last_kernel_ms; }

IRR_EXPORT int gpunb_irr_set_lists(int n, const int *addr, const int *nnb,
                                   const int *members) {
    return gpunb::run_guarded("gpunb_irr_set_lists", [&] {
        IREQ(I.open, "irr_simd is not open");
        if (block_lists(n, addr, nnb, members)) return;
        size_t off = 0;
        for (int q = 0; q < n; ++q) {
            stage_list(addr[q], nnb[q], members + off);
            off += (size_t)nnb[q];
        }
    });
}

}  // extern "C"
