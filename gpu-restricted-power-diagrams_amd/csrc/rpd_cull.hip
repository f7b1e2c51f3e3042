// rpd_cull.hip -- cells whose restriction to the domain is provably empty,
// found before the kNN search.
//
// A domain point x lies in some domain voxel v (a voxel holding triangles or
// whose centre is inside).  For any seed t, |x - t| <= |c_v - t| + r_v with
// c_v the voxel centre and r_v its half diagonal, so the smallest power
// distance U(x) = min_t |x - t|^2 + w_t of x satisfies
//     U(x) - w_min <= M = max_v min_t ((|c_v - t| + r_v)^2 + w_t - w_min).
// Here the min over t runs over the seeds of the kNN-grid cells around c_v
// (any seed gives an upper bound).  A seed s whose voxel lies d >= 2 voxels
// (Chebyshev) from every domain voxel is at least D = (d - 1) vs from every
// domain point.  When D^2 + w_s - w_min > M, every domain point has a strictly
// smaller power distance to another seed: the restricted cell of s has volume
// 0, which is what clipping it would give.  Such seeds skip the kNN search and
// the clip kernels.  Only for the exact power stop (the cell computed is the
// power cell) and without border seeds (walls are not power distances).

#include <hip/hip_runtime.h>

#include <algorithm>

#include "rpd_internal.h"
#include "rpd_wave.h"

namespace rpd {

// margin over the rounding of M and of the seed test (units of the [0,1000] frame)
constexpr double kCoverRel = 1e-9, kCoverAbs = 1e-6;

// Up to kCoverSet requests of one launch: blocks [vb[r], vb[r + 1]) of the
// coverage kernel and tiles [tb[r], tb[r + 1]) of the skip kernel are request
// r's.  In the kernel arguments: nothing is uploaded.
constexpr int kCoverSet = 32;
struct CoverReq {
    const int *counters, *dvox;
    const uint8_t *dist;
    const double *wdev;
    int64_t base, n;
    double vs, wmin;
    int dim, n_dvox, g, apply;
};
struct CoverSet {
    CoverReq r[kCoverSet];
    int vb[kCoverSet + 1], tb[kCoverSet + 1];
    int k;
};

// One thread per domain voxel.  The distance to a seed is rounded up: the
// hardware FP32 square root (1 ulp) of d^2 rounded to FP32 is within 2^-22 of
// the exact one, relative, so scaling it by 1 + 2^-18 bounds it from above
// with room to spare (a d^2 that FP32 flushes to 0 is below 1e-37, far under
// kCoverAbs).  Any upper bound of M is a valid one; this one is looser by
// about 1e-5, relative, and takes a fraction of the VALU of the correctly
// rounded FP64 square root.  (Four lanes per voxel, each over some of the 9
// rows, was slower: the rows do not split evenly.)
//
// What bounds it is FP64 work on many voxels and the latency of a chain of
// loads on few.  A request has at most kCoverBlocks blocks, which go over its
// voxels: from the second round on, a voxel whose minimum so far is not above
// the M found so far cannot raise it, and ends there (its own row of cells
// comes first), which leaves M what it is.  The nine rows' ranges are read at
// once, and a row's seeds four at a time (the last stands in past the end).
// Before (one launch a request, every voxel to its end, one seed at a time) and
// now, with the list of kept cells: 1,000 seeds, sphere in 96^3 70 -> 43 us; 1M
// lattice seeds, cube in 100^3 243 -> 104 us; 16 requests in 96^3 1,422 -> 387.
constexpr int kCoverBlocks = 512;
__global__ __launch_bounds__(256) void coverage_kernel(CoverSet cs, const double4 *__restrict__ stored64,
                                                       unsigned long long *__restrict__ mbits) {
    int q = 0;
    while (q + 1 < cs.k && int(blockIdx.x) >= cs.vb[q + 1]) ++q;
    const CoverReq &rq = cs.r[q];
    double wmin = rq.wmin;
    if (rq.wdev) {
        if (rq.wdev[1] <= RPD_NO_CELL_LIMITS) return;  // walls: no test (every block returns)
        wmin = rq.wdev[0] < INFINITY ? rq.wdev[0] : 0.0;
    }
    const int g = rq.g, dim = rq.dim, n_dvox = rq.n_dvox;
    const double vs = rq.vs;
    __shared__ double red[4];
    // (the values are >= 0, so their bit patterns order as the values)
    unsigned long long *const mp = mbits + q;
    auto m_now = [&]() {
        return __longlong_as_double((long long)__hip_atomic_load(mp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    };
    const int stride = (cs.vb[q + 1] - cs.vb[q]) * 256;
    for (int i0 = (int(blockIdx.x) - cs.vb[q]) * 256; i0 < n_dvox; i0 += stride) {
        const int i = i0 + int(threadIdx.x);
        // at most this, and the voxel's term (below) is at most M so far
        const double enough = m_now() * (1.0 - 4.0 * kCoverRel) - 4.0 * kCoverAbs;
        double best = INFINITY;
        if (i < n_dvox) {
            const int v = rq.dvox[i];
            const double cx = (v % g + 0.5) * vs, cy = ((v / g) % g + 0.5) * vs, cz = (v / (g * g) + 0.5) * vs;
            const double rv = 0.8660254037844387 * vs * (1.0 + 1e-12);  // sqrt(3)/2, rounded up
            auto cc = [&](double c) { return max(0, min(dim - 1, int(c * double(dim) / 1000.0))); };
            const int ci = cc(cx), cj = cc(cy), ck = cc(cz);
            const int x0 = max(0, ci - 1), x1 = min(dim - 1, ci + 1);
            constexpr double kUp = 1.0 + 0x1p-18;
            constexpr int kOrder[9] = {4, 1, 3, 5, 7, 0, 2, 6, 8};  // the own row, its neighbours, the corners
            int lo[9], hi[9];
#pragma unroll
            for (int k = 0; k < 9; ++k) {
                // (a row outside the grid: its own row's range, left empty)
                const int z = ck + kOrder[k] / 3 - 1, y = cj + kOrder[k] % 3 - 1;
                const bool in = z >= 0 && z < dim && y >= 0 && y < dim;
                const int row = in ? (y + z * dim) * dim : (cj + ck * dim) * dim;
                lo[k] = rq.counters[row + x0];
                hi[k] = in ? rq.counters[row + x1 + 1] : lo[k];
            }
#pragma unroll
            for (int k = 0; k < 9; ++k) {
                for (int j = lo[k]; j < hi[k] && best > enough; j += 4) {
                    double4 t[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) t[u] = stored64[min(j + u, hi[k] - 1)];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const double ex = t[u].x - cx, ey = t[u].y - cy, ez = t[u].z - cz;
                        const double d2 = ex * ex + ey * ey + ez * ez;
                        const double dd = double(__builtin_amdgcn_sqrtf(float(d2))) * kUp + rv;
                        best = fmin(best, dd * dd + (t[u].w - wmin));
                    }
                }
            }
            // no seed around this voxel: no bound
            best = best * (1.0 + kCoverRel) + kCoverAbs;
        }
        // block maximum, then at most one atomic per block and round
        const double m = wave_max(i < n_dvox ? best : 0.0);
        if (lane_id() == 0) red[threadIdx.x >> 6] = m;
        __syncthreads();
        if (threadIdx.x == 0) {
            const double bm = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
            if (bm > m_now()) atomicMax(mp, (unsigned long long)__double_as_longlong(bm));
        }
        __syncthreads();  // the next round overwrites red
    }
}

// The seeds' tests and, in the same launch, the ascending list of those kept:
// a tile is 1,024 ids, and the number kept before it comes from the tiles
// before (the library's selection takes three launches and a copy).  The
// outputs of the seeds left out are what every output was filled with before
// the test: written here they went to places all over (1M seeds, torus in
// 128^3, 842,430 of them left out: 64 us, now 29, and 10 more for the fill).
constexpr int kSkipTile = 1024;
__global__ __launch_bounds__(256) void skip_kernel(CoverSet cs, const double4 *__restrict__ stored64,
                                                   const unsigned long long *__restrict__ mbits,
                                                   unsigned long long *__restrict__ state,
                                                   int *__restrict__ ticket, int tile0, int tiles_all,
                                                   int *__restrict__ ids_out, int *__restrict__ cnt,
                                                   int *__restrict__ cnt_host) {
    __shared__ int tile_s, before_s, kept[16];
    const int lane = lane_id(), wv = uni(int(threadIdx.x >> 6));
    if (threadIdx.x == 0) tile_s = atomicAdd(ticket, 1);
    __syncthreads();
    const int tile = uni(tile_s);  // over all launches of this test
    int q = 0;
    while (q + 1 < cs.k && tile - tile0 >= cs.tb[q + 1]) ++q;
    const CoverReq &rq = cs.r[q];
    bool test = rq.apply != 0;
    double wmin = rq.wmin, lim = 0;
    if (test && rq.wdev) {
        test = !(rq.wdev[1] <= RPD_NO_CELL_LIMITS);  // walls: every cell is kept
        wmin = rq.wdev[0] < INFINITY ? rq.wdev[0] : 0.0;
    }
    if (test) lim = __longlong_as_double((long long)mbits[q]) * (1.0 + kCoverRel) + kCoverAbs;
    const int64_t i0 = int64_t(tile - tile0 - cs.tb[q]) * kSkipTile + int64_t(threadIdx.x);
    uint64_t km[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int64_t i = i0 + 256 * u, s = rq.base + i;
        bool skip = false;
        if (test && i < rq.n) {
            const double4 p = stored64[s];
            const int g = rq.g;
            const double vs = rq.vs;
            auto vox = [&](double x) { return int(fmin(fmax(x / vs, 0.0), double(g - 1))); };
            const int d = rq.dist[vox(p.x) + vox(p.y) * g + vox(p.z) * g * g];
            const double D = double(max(0, d - 1)) * vs;
            skip = D * D + (p.w - wmin) > lim;
        }
        km[u] = ballot(i < rq.n && !skip);
        if (lane == 0) kept[4 * u + wv] = __popcll(km[u]);
    }
    __syncthreads();
    int total = 0, at[4] = {0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < 16; ++k) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (k < 4 * u + wv) at[u] += kept[k];
        total += kept[k];
    }
    if (wv == 0) {
        const int b = tile_prefix(state, tile, total);
        if (lane == 0) {
            before_s = b;
            if (tile == tiles_all - 1) {
                *cnt = b + total;
                if (cnt_host) {
                    *cnt_host = b + total;
                    __threadfence_system();
                }
            }
        }
    }
    __syncthreads();
    const int b = before_s;
#pragma unroll
    for (int u = 0; u < 4; ++u)
        if (in_mask(km[u])) ids_out[b + at[u] + mbcnt(km[u])] = int(rq.base + i0 + 256 * u);
}

}  // namespace rpd

using namespace rpd;

// scratch: M bits per request | ticket, count | a word per tile
static size_t cover_tiles_room(int nreq, int64_t n_total) { return size_t(n_total / kSkipTile) + size_t(nreq) + 1; }

int rpd_cover_prepare(int nreq, int64_t n_total, DevBuf &scratch, int **zero, int *zero_words) {
    const size_t bytes = size_t(nreq) * 8 + 16 + 8 * cover_tiles_room(nreq, n_total);
    if (scratch.ensure(bytes) != RPD_OK) return RPD_E_NOMEM;
    *zero = static_cast<int *>(scratch.ptr);
    *zero_words = int(bytes / 4);
    return RPD_OK;
}

int rpd_cover_skip(hipStream_t st, const CoverArgs *reqs, int nreq, int64_t n_total, DevBuf &scratch, int *ids_out,
                   int *n_out, int *n_out_dev, const int **count_dev) {
    if (n_total <= 0 || nreq <= 0) return RPD_E_ARG;
    auto *mbits = static_cast<unsigned long long *>(scratch.ptr);
    int *ticket = reinterpret_cast<int *>(mbits + nreq), *cnt = ticket + 1;
    unsigned long long *state = mbits + nreq + 2;
    int64_t next = 0, tiles = 0;
    for (int r = 0; r < nreq; ++r) {
        if (reqs[r].base != next || reqs[r].n <= 0) return RPD_E_ARG;
        next += reqs[r].n;
        tiles += (reqs[r].n + kSkipTile - 1) / kSkipTile;
    }
    if (next != n_total || size_t(tiles) > cover_tiles_room(nreq, n_total)) return RPD_E_ARG;
    int tile0 = 0;
    for (int r0 = 0; r0 < nreq; r0 += kCoverSet) {
        CoverSet cs;
        cs.k = std::min(kCoverSet, nreq - r0);
        cs.vb[0] = cs.tb[0] = 0;
        for (int r = 0; r < cs.k; ++r) {
            const CoverArgs &c = reqs[r0 + r];
            cs.r[r] = CoverReq{c.counters, c.dvox, c.dist, c.wdev, c.base, c.n, c.vs,
                               c.wmin,     c.dim,  c.n_dvox, c.g,  c.apply ? 1 : 0};
            cs.vb[r + 1] = cs.vb[r] + (c.apply ? std::min((c.n_dvox + 255) / 256, kCoverBlocks) : 0);
            cs.tb[r + 1] = cs.tb[r] + int((c.n + kSkipTile - 1) / kSkipTile);
        }
        const CoverArgs &c0 = reqs[r0];
        if (cs.vb[cs.k] > 0)
            coverage_kernel<<<unsigned(cs.vb[cs.k]), 256, 0, st>>>(cs, c0.stored64, mbits + r0);
        skip_kernel<<<unsigned(cs.tb[cs.k]), 256, 0, st>>>(cs, c0.stored64, mbits + r0, state, ticket, tile0,
                                                           int(tiles), ids_out, cnt, n_out_dev);
        tile0 += cs.tb[cs.k];
    }
    if (!n_out_dev && hipMemcpyAsync(n_out, cnt, sizeof(int), hipMemcpyDeviceToHost, st) != hipSuccess)
        return RPD_E_DEVICE;
    *count_dev = cnt;
    return hipGetLastError() == hipSuccess ? RPD_OK : RPD_E_DEVICE;
}
