// pot.hip -- the O(N^2) potential of gpupot_ and of the energy sum
// (gpupot.gpu.cu:32-57): phi_i = sum over j with r2 > 0 of m_j / r_ij.
//
// Arithmetic of every pair: FP64 differences rounded to FP32, FP32 r2, 1/r
// and product; a tile's 64 terms are added in FP32 in j order and the tile
// sums in FP64.
//
// Kernels
//   k_pack_p     FP64 (m, x) -> 32-byte records, FP32 masses; NaN check.
//   k_pot_pass1  potential of a range of i against slices of all j.
//   k_pot_sym    potential of all bodies: each 1/r is formed once for the
//                pair and used for both bodies.
//   k_pot_pass2, k_pot_rows   FP64 sums of the partials.
#include "gpunb_internal.h"

#include <algorithm>
#include <cmath>

namespace gpunb {

namespace {

// A record as one eight-register load (member by member, it would be three).
typedef int v8i __attribute__((ext_vector_type(8)));
__device__ __forceinline__ double rec_f64(const v8i &r, int k) {
    return __hiloint2double(r[2 * k + 1], r[2 * k]);
}

// 1/r of record J and a body at (x0, y0, z0).  A pair at zero distance gives
// +inf; with CHECK it gives 0, which leaves it out of the sums.
template <bool CHECK>
__device__ __forceinline__ float pair_rinv(const v8i &J, double x0, double y0,
                                           double z0) {
    const float fx = (float)(rec_f64(J, 0) - x0);
    const float fy = (float)(rec_f64(J, 1) - y0);
    const float fz = (float)(rec_f64(J, 2) - z0);
    const float r2 = fmaf(fz, fz, fmaf(fy, fy, fx * fx));
    const float r = __builtin_amdgcn_rsqf(r2);
    return !CHECK || r2 > 0.0f ? r : 0.0f;
}

// a + the terms of the NJ records p[0, NJ), in order.  With KEEP, 1/r of
// record j goes to keep[kPotStride * j].  The next group of records loads
// while the current one is evaluated, in two buffers used in turn (the
// scheduling barriers keep the loads ahead of it); the record array carries a
// spare tile past its end, so the last look-ahead stays in bounds.
constexpr int kPotStride = 68;   // floats per LDS row: 64 i, 16-byte aligned
template <bool CHECK, bool KEEP, int NJ>
__device__ __forceinline__ float pot_run(const PRec *__restrict__ p, double x0,
                                         double y0, double z0, float a,
                                         float *keep) {
    constexpr int G = 2;
    static_assert(NJ % (2 * G) == 0, "whole groups in both buffers");
    const v8i *__restrict__ rec = reinterpret_cast<const v8i *>(p);
    v8i Pa[G], Pb[G];
    auto group = [&](const v8i(&J)[G], int j) {
        float r[G];
#pragma unroll
        for (int k = 0; k < G; ++k) r[k] = pair_rinv<CHECK>(J[k], x0, y0, z0);
#pragma unroll
        for (int k = 0; k < G; ++k) {
            a += __int_as_float(J[k][6]) * r[k];
            if (KEEP) keep[kPotStride * (j + k)] = r[k];
        }
    };
#pragma unroll
    for (int k = 0; k < G; ++k) {
        Pa[k] = rec[k];
        asm volatile("" : "+s"(Pa[k]));
    }
#pragma unroll 1
    for (int j = 0; j < NJ; j += 2 * G) {
#pragma unroll
        for (int k = 0; k < G; ++k) Pb[k] = rec[j + G + k];
        __builtin_amdgcn_sched_barrier(0);
        group(Pa, j);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < G; ++k) Pa[k] = rec[j + 2 * G + k];
        __builtin_amdgcn_sched_barrier(0);
        group(Pb, j + G);
        __builtin_amdgcn_sched_barrier(0);
    }
    return a;
}

// As pot_run, on records of which hardly any is at zero distance: without
// the check first, again with it when a sum is not finite (zero distance:
// m * inf, or NaN for m = 0).  The check would be 9 of 51 issue cycles a pair.
// own: the bodies are among the records, so only the run with the check.
template <bool KEEP, int NJ>
__device__ __forceinline__ float pot_run_rare(const PRec *__restrict__ p,
                                              double x0, double y0, double z0,
                                              float a, float *keep, bool own) {
    if (!own) {
        const float b = pot_run<false, KEEP, NJ>(p, x0, y0, z0, a, keep);
        if (__ballot(!(fabsf(b) < INFINITY)) == 0) return b;
    }
    return pot_run<true, KEEP, NJ>(p, x0, y0, z0, a, keep);
}

}  // namespace

__global__ __launch_bounds__(256) void k_pack_p(const double *__restrict__ m,
                                                const double *__restrict__ x,
                                                int n, int n_pad,
                                                PRec *__restrict__ p,
                                                float *__restrict__ pm,
                                                unsigned *__restrict__ err) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n_pad) return;
    PRec r;
    r.x = r.y = r.z = kPadPos;
    r.m32 = 0.0f;
    r.pad = 0.0f;
    if (j < n) {
        r.x = x[3 * (size_t)j + 0];
        r.y = x[3 * (size_t)j + 1];
        r.z = x[3 * (size_t)j + 2];
        const double mj = m[j];
        r.m32 = (float)mj;
        const double chk = r.x + r.y + r.z + mj;
        if (chk != chk) atomicOr(err, ERR_NAN_J);
    }
    p[j] = r;
    pm[j] = r.m32;
}

__global__ __launch_bounds__(64) void k_pot_pass1(const PRec *__restrict__ p,
                                                  int ntile, int i0, int ni,
                                                  int n_iw, int nslice,
                                                  double *__restrict__ part) {
    const int ntask = n_iw * nslice;
    const int per = (ntask + 7) >> 3;
    const int task = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (task >= ntask) return;
    const int s = task / n_iw;
    const int iw = task - s * n_iw;
    const int q = iw * 64 + threadIdx.x;
    const bool act = q < ni;
    const int tb = (int)(((long long)ntile * s) / nslice);
    const int te = (int)(((long long)ntile * (s + 1)) / nslice);
    double x0 = 0.0, y0 = 0.0, z0 = 0.0;
    if (act) {
        const PRec r = p[i0 + q];
        x0 = r.x;
        y0 = r.y;
        z0 = r.z;
    }
    // The wavefront's own bodies, b0 and the 63 after it, are in one or two
    // tiles.  In a call of few tiles a second run of those is its longest task:
    // 4000 bodies 80 us with it, 73 us so.
    const int b0 = i0 + iw * 64;
    double A = 0.0;
    for (int t = tb; t < te; ++t) {
        const bool own = (t + 1) * kTile > b0 && t * kTile < b0 + 64;
        A += (double)pot_run_rare<false, kTile>(p + t * kTile, x0, y0, z0, 0.0f,
                                                nullptr, own);
    }
    if (act) part[(size_t)q * nslice + s] = A;
}

__global__ __launch_bounds__(256) void k_pot_pass2(const double *__restrict__ part,
                                                   int ni, int nslice,
                                                   double *__restrict__ pot) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= ni) return;
    double s = 0.0;
    for (int k = 0; k < nslice; ++k) s += part[(size_t)q * nslice + k];
    pot[q] = s;
}

// ---------------------------------------------------------------------------
// All bodies: 1/r of a pair is the same bits seen from either body (the
// differences only change sign), so each is formed once.  The bodies are cut
// in blocks of g = K * nsub tiles; a wavefront (workgroup) takes one block
// pair bp <= bq, K tiles I of block bp at a time (one body per lane, in
// registers) against the tiles J of block bq.  Per tile pair, for each half
// of J (32 j): the lanes run the half as k_pot_pass1 does and leave every
// 1/r in LDS (row j, column i); then 32 lanes, one per j, add m_i / r over
// the 64 i of the row, in i order: the sum that k_pot_pass1 forms for body j
// over tile I, bit for bit.  The half keeps the LDS at 8.7 KB, so that four
// wavefronts fit a SIMD; with whole tiles (17.4 KB, two wavefronts) the
// second sum would use all 64 lanes, but the issue rate falls by more.
//
// Partials: row r of part holds, for every body of block b, its sum over
// block r (r = b: tiles at and after its own; row nblock: tiles of its own
// block before its own).
//
// Bound: VALU issue, as k_pot_pass1; of its 51 issue cycles a pair, the 43 of
// the distance and 1/r are paid once for two bodies.  N = 131072, the kernel
// alone: 5.62 ms with a pass over all pairs (3.1e12 pairs/s), 3.4 ms so (2.5e12
// unordered pairs/s), the same bits.
// ---------------------------------------------------------------------------
template <int K>
__global__ __launch_bounds__(64) void k_pot_sym(const PRec *__restrict__ p,
                                                const float *__restrict__ pm,
                                                int ntile, int nblock, int nsub,
                                                double *__restrict__ part) {
    __shared__ __align__(16) float keep[32 * kPotStride];
    const int lane = threadIdx.x;
    const size_t npad = (size_t)ntile * kTile;
    // Block pair of task t = bq (bq + 1) / 2 + bp.
    const long long t = blockIdx.x;
    int bq = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while ((long long)bq * (bq + 1) / 2 > t) --bq;
    while ((long long)(bq + 1) * (bq + 2) / 2 <= t) ++bq;
    bq = __builtin_amdgcn_readfirstlane(bq);
    const int bp = (int)(t - (long long)bq * (bq + 1) / 2);
    const int g = K * nsub;
    const int j0 = bq * g, j1 = min(j0 + g, ntile);
    const int it1 = min((bp + 1) * g, ntile);
    double *drow = part + (size_t)(bp == bq ? nblock : bp) * npad;   // of bq
    double *irow = part + (size_t)bq * npad;                         // of bp
    for (int sub = 0; sub < nsub; ++sub) {
        const int i0 = bp * g + K * sub;
        double xi[K], yi[K], zi[K], A[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            A[k] = 0.0;
            const PRec r = p[(size_t)min(i0 + k, ntile - 1) * kTile + lane];
            xi[k] = r.x;
            yi[k] = r.y;
            zi[k] = r.z;
        }
        for (int J = j0; J < j1; ++J) {
            const PRec *__restrict__ pj = p + (size_t)J * kTile;
            double B = 0.0;
            if (sub > 0) B = drow[(size_t)J * kTile + lane];
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const int I = i0 + k;
                if (I >= it1 || I > J) continue;
                if (I == J) {
                    A[k] += (double)pot_run<true, false, kTile>(
                        pj, xi[k], yi[k], zi[k], 0.0f, nullptr);
                    continue;
                }
                const float *__restrict__ mi = pm + (size_t)I * kTile;
                float a = 0.0f, b = 0.0f;
#pragma unroll 1
                for (int h = 0; h < 2; ++h) {
                    a = pot_run_rare<true, kTile / 2>(pj + 32 * h, xi[k], yi[k],
                                                      zi[k], a, keep + lane, false);
                    __threadfence_block();
                    if ((lane >> 5) == h) {
                        const float4 *row = reinterpret_cast<const float4 *>(
                            keep + kPotStride * (lane & 31));
#pragma unroll 4
                        for (int c = 0; c < kTile / 4; ++c) {
                            const float4 r = row[c];
                            b += mi[4 * c] * r.x;
                            b += mi[4 * c + 1] * r.y;
                            b += mi[4 * c + 2] * r.z;
                            b += mi[4 * c + 3] * r.w;
                        }
                    }
                    __threadfence_block();
                }
                A[k] += (double)a;
                B += (double)b;
            }
            drow[(size_t)J * kTile + lane] = B;
        }
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (i0 + k < it1) irow[(size_t)(i0 + k) * kTile + lane] = A[k];
    }
}

// pot[q] = sum of the nrow partial rows.
__global__ __launch_bounds__(256) void k_pot_rows(const double *__restrict__ part,
                                                  size_t npad, int nrow, int n,
                                                  double *__restrict__ pot) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    constexpr int U = 8;
    double s = 0.0;
    int r = 0;
    for (; r + U <= nrow; r += U) {
        double v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = part[(size_t)(r + u) * npad + q];
#pragma unroll
        for (int u = 0; u < U; ++u) s += v[u];
    }
    for (; r < nrow; ++r) s += part[(size_t)r * npad + q];
    pot[q] = s;
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------

static inline int cdiv(long long a, long long b) { return (int)((a + b - 1) / b); }

void launch_pack_p(hipStream_t st, const double *m, const double *x, int n,
                   int n_pad, PRec *p, float *pm, unsigned *err) {
    if (n_pad <= 0) return;
    hipLaunchKernelGGL(k_pack_p, dim3(cdiv(n_pad, 256)), dim3(256), 0, st, m, x,
                       n, n_pad, p, pm, err);
}

void launch_pot(hipStream_t st, const PRec *p, int ntile, int i0, int ni,
                int nslice, double *part, double *pot) {
    if (ni <= 0) return;
    const int n_iw = cdiv(ni, 64);
    const int ntask = n_iw * nslice;
    const int nblk = 8 * ((ntask + 7) / 8);
    hipLaunchKernelGGL(k_pot_pass1, dim3(nblk), dim3(64), 0, st, p, ntile, i0,
                       ni, n_iw, nslice, part);
    hipLaunchKernelGGL(k_pot_pass2, dim3(cdiv(ni, 256)), dim3(256), 0, st, part,
                       ni, nslice, pot);
}

// Tiles held by a wavefront: few where the block pairs would not fill the
// machine.  Blocks: a launch of G blocks has G (G + 1) / 2 workgroups, about
// 4600 resident at once, and G + 1 partials per body; 512 MiB of partials or
// 256 blocks, whichever is more (N = 131072: 512 blocks 3.59 ms, 256 blocks
// 3.75 ms, the last round of workgroups being nearly empty; N = 16384: 2
// tiles 143 us, 1 tile 145, 4 tiles 178).
PotSym pot_sym_plan(int ntile) {
    PotSym P;
    P.k = ntile >= 1024 ? 4 : ntile >= 128 ? 2 : 1;
    const int rows = std::max(256, (1 << 26) / (kTile * ntile));
    P.nsub = std::max(1, cdiv(ntile, rows * P.k));
    P.nblock = cdiv(ntile, P.k * P.nsub);
    return P;
}

void launch_pot_sym(hipStream_t st, const PRec *p, const float *pm, int n,
                    int ntile, const PotSym &P, double *part, double *pot) {
    if (n <= 0) return;
    const unsigned ntask =
        (unsigned)((long long)P.nblock * (P.nblock + 1) / 2);
    const auto fn = P.k == 4 ? k_pot_sym<4> : P.k == 2 ? k_pot_sym<2> : k_pot_sym<1>;
    hipLaunchKernelGGL(fn, dim3(ntask), dim3(64), 0, st, p, pm, ntile, P.nblock,
                       P.nsub, part);
    hipLaunchKernelGGL(k_pot_rows, dim3(cdiv(n, 256)), dim3(256), 0, st, part,
                       (size_t)ntile * kTile, P.nblock + 1, n, pot);
}

int pot_resident_waves() {
    int dev = 0, nb = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipGetDeviceProperties(&prop, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &nb, (const void *)k_pot_pass1, 64, 0) != hipSuccess)
        return 0;
    return nb * prop.multiProcessorCount;
}

}  // namespace gpunb
