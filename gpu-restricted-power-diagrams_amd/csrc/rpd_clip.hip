// rpd_clip.hip -- per-seed power-cell clipping, restriction to the domain
// grid and fused volume / first-moment integration on gfx950.
//
// Replaces compute_voro_cell (ConvexCell.cl:812-1152) and the ConvexCell
// routines it drives (CCInit :278-308, CCNewPlane :314-333, CCClipByPlane
// :517-563, CCComputeBoundary :463-515, CCVertexIsInHalfSpace :400-461,
// CCIsSecurityRadiusReached :364-382, CCClipTetFromPointsInfinite :565-575,
// CCExportBaryVolume :577-619).
//
// Layout: ONE CELL PER WAVEFRONT.  Vertex j of the cell lives in lane j & 63
// (register slot j >> 6): its three plane ids and its homogeneous
// coordinates (X, Y, Z, W), i.e. the cofactors of CCComputeVertexCoordinates.
// Because det4x4(pi1, pi2, pi3, e) == e . (X, Y, Z, W), the plane-side test
// of CCVertexIsInHalfSpace is one 4-term dot product per lane.  Plane
// equations live in LDS.  A clip removes the vertices with e.v > 0, finds the
// cavity boundary as the edges of removed vertices whose other end is kept
// (checked to be one simple cycle, else inconsistent_boundary), and places one
// new vertex (plane, a, b) per boundary edge a->b into free lanes -- the same
// vertex set CCComputeBoundary + CCNewVertex build.
//
// Two kernels per pass:
//   clip_cells_kernel   the bisector loop for every cell (light, high
//                       occupancy).  A cell that provably misses the domain
//                       ends there with volume 0; a finished cell leaves a
//                       compact record at its item's slot (FP64 planes, vertex
//                       triples and adjacency);
//   finish_cells_kernel restriction to the domain (bbox, voxels, apex, cone
//                       clips per strip of voxel faces or boundary triangle)
//                       and the integration, for the cells with a record.
//
// Everything is in the seed-local frame (origin at the seed, FP64 inputs):
// planes n.y + d with d = (|b|^2 + w_B - w_s) / (2|b|), b = B - s.
//
// Forms: FP64 (all double); mixed: the plane-side tests and the vertex
// registers are FP32 and each test also evaluates a certified bound on its
// FP32 error against the FP64 planes, 2^-18 * (at least the sum of |terms| of
// the det4x4 expansion).  A test inside the bound, and every test of an
// ill-conditioned vertex, is decided in FP64 from the vertex's planes, as the
// FP64 form decides it: the finish kernel has FP64 planes in LDS, the bisector
// kernel FP32 planes, beside which it makes FP64 ones when a test first needs
// them.
// A cavity that such decisions leave inconsistent ends the cell with a status
// that the host re-runs in FP64 to its end.  The records' planes are FP64; the
// cell geometry that produces the results
// (bbox, cone planes, volume and moments) is evaluated in FP64 from them, so
// an unflagged mixed cell has the FP64 combinatorics and FP64 geometry.  FP32
// form: everything in FP32, no filter.  Moments are accumulated in FP64.

#include <hip/hip_runtime.h>
#include <atomic>

#include "rpd_internal.h"
#include "rpd_wave.h"

namespace rpd {

template <typename R>
struct Pl {
    R x, y, z, w;
};

enum ClipResult : int { kNoClip = -1, kClipped = -2 };

struct ClipArgs {
    const double4 *seeds;
    const int *perm;
    const int *ids;
    const int *knn;
    int64_t n_ids;
    int64_t n_seeds;
    int K, P, V, T;
    int apex_mode;
    int g;
    double vs;
    const int8_t *flags;
    const int8_t *centre;
    const double4 *gpts;
    const int *tris;
    const int *tlist;
    const int *toffs;
    double4 *out;
    int *status;
    int *kused;
    int lds_stride;   // LDS bytes of one wave
    int cell_stride;  // LDS bytes shared by the waves of one cell (finish kernel)
    const int *tvoffs;    // per triangle: offsets into tvox
    const uint32_t *tvox; // per triangle: sorted voxels whose list holds it, z<<20 | y<<10 | x
    const uint4 *tinfo;   // per triangle-list entry: its voxel, earlier near voxels holding it
    const int *vfoffs;    // voxel domain: per lattice point, offsets into vface
    const uint2 *vface;   // voxel domain: faces, by the lattice point of their lowest corner
    int security_mode;    // 0 exact power stop, 1 reference stop
    double wmin;          // minimum weight over non-border seeds
    const uint8_t *dist;  // Chebyshev voxel distance to the nearest domain voxel (nullable)
    // Records of the cells (rec_stride bytes, item t's at slot t); one whose
    // header holds no cell (sid -1) is not for the finish kernel.  code[t] is
    // how item t left the bisector kernel (kCode*), from which
    // list_failures_kernel makes the lists: with one wave per cell, counters
    // that every cell adds to cost 9 ns a cell (atomics of one address), more
    // than the cell itself where most cells fail.
    char *rec;
    int rec_stride;
    uint8_t *code;
    // finish kernel: failed cells for the next pass (nullable): fl_cnt[0]
    // exact-predicate entries, stored at fl_eo[-1], fl_eo[-2], ..., [1]
    // overflow entries at fl_eo[0], fl_eo[1], ... (so that both kinds together
    // are one range), [2 + s] cells that ended with status s, [13] the largest
    // triangle union of a cell that overflowed T
    int *fl_cnt, *fl_eo;
    int exact_final;      // FP64 form: exact-predicate failures are final
    // A cell whose list runs out before its security radius is reached can be
    // resumed: its state goes to slot rs_base + t of rs_out (records of
    // rs_out_stride bytes; the slot is kept in rslot[sid]), the stored id of
    // its last neighbour to lastnb[sid].  rs_out may be rec itself (rs_base
    // 0): an item has one record, for the finish kernel or to resume from.
    // rs_out null: a plain overflow.  With rs_in set (FP64 and mixed forms:
    // records of FP64 planes), every cell resumes from record rs_in[rslot[sid]] (written with rs_in_P planes) and
    // its list holds only the neighbours after the ones it has used.
    char *rs_out;
    int rs_out_stride, rs_base;
    const char *rs_in;
    int rs_in_stride, rs_in_P;
    int *rslot, *lastnb;
    // Hessian (finish kernel, H > 0): per original seed up to H entries of
    // hc values in hess and the neighbours' original indices in hids
    double *hess;
    int *hids;
    int H, hc;
    int *dcnt;  // debug counters of this pass (kDcStride ints), nullable
    int keep_exact;  // finish kernel: an exact-predicate failure leaves the outputs as they are
    // finish kernel, a batch with both kinds of domains: 1 only the cells of
    // requests with voxel faces (or no domain), 2 only the others
    int only;
    int count_only;  // finish kernel, triangle lists: only the union counters of the cells whose union fits
    // packed batch (nullable): the fields of request req_of[sid] replace
    // n_seeds, wmin and the domain's
    const ReqDesc *reqs;
    const uint16_t *req_of;
    // finish kernel: work item i is the record at slot slots[i] (nullable:
    // slot i); fl_slot (nullable) receives the record slot of each failure it
    // lists, at the failure's index in fl_eo
    const int *slots;
    int *fl_slot;
    // layout of the records the finish kernel reads: planes and vertex
    // slots they were written with (the finish kernel's own P and S may be
    // larger)
    int rec_P, rec_S;
};

// The arguments in the kernel's argument area (its first parameter), for code
// after the loops: loaded where they are used.
using ColdArgs = const __attribute__((address_space(4))) ClipArgs;
__device__ __forceinline__ ColdArgs *cold_args() {
    auto p = (ColdArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}

// The cell of stored id sid reads its request's seed count, weight minimum
// and domain (packed batch; wave-uniform, so the fields stay in SGPRs).  The
// kernels take it as a template parameter, so that a single diagram's
// kernels keep every field in the kernel arguments.
__device__ __forceinline__ void bind_request(ClipArgs &a, int sid) {
    const ReqDesc &d = a.reqs[uni(int(a.req_of[sid]))];
    a.n_seeds = d.n_seeds;
    a.wmin = d.wmin;
    a.g = d.g;
    a.vs = d.vs;
    a.flags = d.flags;
    a.centre = d.centre;
    a.gpts = d.gpts;
    a.tris = d.tris;
    a.tlist = d.tlist;
    a.toffs = d.toffs;
    a.tvoffs = d.tvoffs;
    a.tvox = d.tvox;
    a.tinfo = d.tinfo;
    a.vfoffs = d.vfoffs;
    a.vface = d.vface;
    a.dist = d.dist;
}

// How an item leaves the bisector kernel: done (no list), queued for the
// finish kernel, or failed with status code - kCodeFailed (code -
// kCodeResume: its state kept, to be resumed).
constexpr uint32_t kCodeDone = 0, kCodeQueued = 1, kCodeFailed = 16, kCodeResume = 32;

__device__ __forceinline__ bool exact_failure(int st) {
    return st == RPD_NEEDS_EXACT_PREDICATES || st == RPD_INCONSISTENT_BOUNDARY ||
           st == RPD_FIND_ANOTHER_BEGINNING_VERTEX;
}

// Whether a cell that ended with status st goes to the failure list:
// overflows (vertex, plane, K, triangle) always; needs_exact_predicates,
// inconsistent_boundary and find_another_beginning_vertex when the form was
// not FP64 (in FP64 a recomputation would fail the same way).
__device__ __forceinline__ bool listed_failure(int exact_final, int st) {
    if (st == RPD_SUCCESS || st == RPD_EMPTY_CELL || st == RPD_HESSIAN_OVERFLOW) return false;
    return !(exact_failure(st) && exact_final);
}

// Finish kernel: appends a failed cell (stored id sid, record slot rslot) to
// the failure list.  One lane.  (Few cells fail here.)
__device__ __forceinline__ void note_failure(const ClipArgs &a, int sid, int st, int rslot) {
    if (!a.fl_cnt || !listed_failure(a.exact_final, st)) return;
    const bool exact = exact_failure(st);
    atomicAdd(a.fl_cnt + 2 + st, 1);
    const int k = atomicAdd(a.fl_cnt + (exact ? 0 : 1), 1);
    a.fl_eo[exact ? -1 - k : k] = sid;
    if (a.fl_slot) a.fl_slot[exact ? -1 - k : k] = rslot;
}

__device__ __forceinline__ uint32_t pack3(uint32_t a, uint32_t b, uint32_t c) { return a | (b << 8) | (c << 16); }
// no vertex (plane triples use 24 bits)
constexpr uint32_t kNoTri = 0xffffffffu;
__device__ __forceinline__ uint32_t t0(uint32_t t) { return t & 0xff; }
__device__ __forceinline__ uint32_t t1(uint32_t t) { return (t >> 8) & 0xff; }
__device__ __forceinline__ uint32_t t2(uint32_t t) { return (t >> 16) & 0xff; }

__device__ __forceinline__ void wsync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename R>
__device__ __forceinline__ Pl<R> rlane_pl(const Pl<R> &p, int l) {
    return Pl<R>{rlane(p.x, l), rlane(p.y, l), rlane(p.z, l), rlane(p.w, l)};
}

template <typename T, typename U>
__device__ __forceinline__ Pl<T> cvt(const Pl<U> &p) {
    return Pl<T>{T(p.x), T(p.y), T(p.z), T(p.w)};
}

// Homogeneous vertex of planes (p1, p2, p3): the cofactors of
// CCComputeVertexCoordinates (ConvexCell.cl:344-362).
template <typename R>
__device__ __forceinline__ void vertex_from_planes(const Pl<R> &p1, const Pl<R> &p2, const Pl<R> &p3, R &X, R &Y,
                                                   R &Z, R &W) {
    const R m12 = p2.x * p3.y - p2.y * p3.x;
    const R m13 = p2.x * p3.z - p2.z * p3.x;
    const R m14 = p2.x * p3.w - p2.w * p3.x;
    const R m23 = p2.y * p3.z - p2.z * p3.y;
    const R m24 = p2.y * p3.w - p2.w * p3.y;
    const R m34 = p2.z * p3.w - p2.w * p3.z;
    X = -p1.w * m23 - p1.y * m34 + p1.z * m24;
    Y = p1.x * m34 + p1.w * m13 - p1.z * m14;
    Z = -p1.x * m24 + p1.y * m14 - p1.w * m12;
    W = p1.x * m23 - p1.y * m13 + p1.z * m12;
}

// Whether the vertex of planes tr lies strictly outside plane e, in FP64:
// the vertex rebuilt from its FP64 planes (as the FP64 form builds it) and
// the FP64 form's test.  (Out of line, the call cost the finish kernel more
// spills than inlined.)
__device__ __forceinline__ bool outside64(const Pl<double> *planes, uint32_t tr, Pl<double> e) {
    double x, y, z, w;
    vertex_from_planes<double>(planes[t0(tr)], planes[t1(tr)], planes[t2(tr)], x, y, z, w);
    return e.x * x + e.y * y + e.z * z + e.w * w > 0.0;
}

// The squared distance from the seed of the vertex of planes tr, in FP64 from
// its FP64 planes.
__device__ __forceinline__ float vertex_r2_64(const Pl<double> *planes, uint32_t tr) {
    double x, y, z, w;
    vertex_from_planes<double>(planes[t0(tr)], planes[t1(tr)], planes[t2(tr)], x, y, z, w);
    return float((x * x + y * y + z * z) / (w * w));
}

// Error bound factor of the mixed form: 64 units in the last place of FP32
// (first-order analysis gives 13: 4 from rounding the FP64 planes, 9 from the
// cofactor and dot-product evaluation).  The bound of a test e.v is
// kappa * (|e.x| MX + |e.y| MY + |e.z| MZ + |e.w| MW) with MX, MY, MZ, MW the
// sums of absolute values of the cofactors' terms.  The planes' normals are
// unit vectors, so by Cauchy-Schwarz MX, MY and MZ are at most M = |w1| + |w2|
// + |w3| (the offsets), and MW, the permanent of three unit vectors, at most
// 2 / sqrt(3): the test takes kappa * ((|e.x| + |e.y| + |e.z|) M + |e.w|
// kMagW), which is not smaller.  M costs 3 instructions of the 28 that the
// sums do; it is about twice as large, but a test it leaves open is decided
// in FP64 in place.
constexpr float kFilterKappa = 0x1.0p-18f;
constexpr float kMagW = 1.1548f;
// vertices with |W| below this are ill-conditioned in FP32: all their tests are
// decided in FP64, and their distance from the seed is taken in FP64
constexpr float kFilterMinW = 1.0e-3f * kMagW;

// apex_mode 1 puts the cone apex at this fraction of a voxel whose interior
// has one known class (in or out).  Any interior point is valid; a generic
// one keeps the cone planes off the voxel lattice and off the CUBE_EPSILON
// box (the voxel centre lies on planes such as y + z = 1000 that contain box
// edges such as y = 1000.1, z = -0.1).
__device__ constexpr double kApexFrac[3] = {0.530901699437495, 0.520710678118655, 0.536602540378444};

// CCInit vertex triples (ConvexCell.cl:299-306), one byte per vertex:
// vertex i has planes (kCube0 >> 8i, kCube1 >> 8i, kCube2 >> 8i) & 0xff.
constexpr uint64_t kCube0 = 0x0402040405010502ull;  // 2 5 1 5 4 4 2 4
constexpr uint64_t kCube1 = 0x0304000201050305ull;  // 5 3 5 1 2 0 4 3
constexpr uint64_t kCube2 = 0x0101030003020000ull;  // 0 0 2 3 0 3 1 1

// Adjacency of the cube's vertices: entry k of vertex i, 5 bits at 16 (i & 3) +
// 5 k of word i >> 2, is (vertex << 2 | edge) of the reverse of edge k of i.
struct CubeAdj {
    uint64_t w[2];
};
constexpr CubeAdj cube_adjacency() {
    CubeAdj c{};
    const uint64_t t[3] = {kCube0, kCube1, kCube2};
    for (int i = 0; i < 8; ++i)
        for (int k = 0; k < 3; ++k) {
            const uint64_t u = (t[k] >> (8 * i)) & 0xff, v = (t[(k + 1) % 3] >> (8 * i)) & 0xff;
            for (int j = 0; j < 8; ++j)
                for (int m = 0; m < 3; ++m)
                    if (((t[m] >> (8 * j)) & 0xff) == v && ((t[(m + 1) % 3] >> (8 * j)) & 0xff) == u)
                        c.w[i >> 2] |= uint64_t(j << 2 | m) << (16 * (i & 3) + 5 * k);
        }
    return c;
}
constexpr CubeAdj kCubeAdj = cube_adjacency();

// A vertex's three adjacency entries as LDS holds them (16 bits each) and as a
// record does (10 bits each).
__device__ __forceinline__ uint2 adj_unpack(uint32_t a) {
    return make_uint2((a & 0x3ffu) | ((a << 6) & 0x3ff0000u), a >> 20);
}
__device__ __forceinline__ uint32_t adj_pack(uint2 a) { return (a.x & 0x3ffu) | ((a.x >> 6) & 0xffc00u) | (a.y << 20); }

// ---------------------------------------------------------------------------
// The cell of one wavefront: vertices in lanes, planes in LDS.
// ---------------------------------------------------------------------------
// The cell of one wavefront.  Planes are stored in LDS in precision PS: the
// bisector kernel keeps them in the test precision R, the finish kernel in
// the geometry precision RP.
//
// Edge k of a vertex (p0, p1, p2) goes from plane p_k to p_(k+1); its reverse
// belongs to the vertex at its other end.  adj holds, per vertex (64 slot +
// lane) and edge, that vertex and which of its edges the reverse is (vertex <<
// 2 | edge, 16 bits).  A clip's boundary edges are those of removed vertices
// whose other end is kept: one LDS read and three bit tests.  (A bit matrix
// of directed edges over pairs of planes, built by LDS atomics in every clip,
// took three atomics, three reads and three writes with an address
// computation each.)
template <typename R, typename RP, bool FILTER, int S, typename PS = RP>
struct WaveCell {
    Pl<PS> *planes;
    uint32_t *nvs;
    uint8_t *nxt;       // boundary successor of a plane (cycle check; 0xff between clips)
    uint8_t *sta, *end;  // new vertex whose boundary edge starts / ends at a plane
    uint2 *adj;
    int P, V, nb_plane, lane;
    uint32_t tri[S];
    R X[S], Y[S], Z[S], W[S], r2[S];
    float M[S];
    uint64_t valid[S];
    // (FILTER) vertices whose tests are all decided in FP64: ill-conditioned
    // in FP32 (small |W|)
    uint64_t x64[S];
    R maxr2;

    // R2: also the vertex's squared distance from the seed (the bisector
    // loop's stop test reads it through maxr2; the finish kernel does not)
    template <bool R2 = true>
    __device__ void set_vertex(int s, uint32_t tr, const Pl<R> &p1, const Pl<R> &p2, const Pl<R> &p3) {
        tri[s] = tr;
        vertex_from_planes<R>(p1, p2, p3, X[s], Y[s], Z[s], W[s]);
        if (FILTER) M[s] = fabsf(float(p1.w)) + fabsf(float(p2.w)) + fabsf(float(p3.w));
        if (R2) {
            // FP32: the hardware reciprocal (1 ulp); r2 is read only by the
            // stop and skip tests, whose radius margin (2e-4) is far larger
            R iw;
            if constexpr (sizeof(R) == 4)
                iw = __builtin_amdgcn_rcpf(W[s]);
            else
                iw = R(1) / W[s];
            const R ix = X[s] * iw, iy = Y[s] * iw, iz = Z[s] * iw;
            r2[s] = ix * ix + iy * iy + iz * iz;
        }
    }

    template <bool R2 = true>
    __device__ void set_vertex_lds(int s, uint32_t tr) {
        set_vertex<R2>(s, tr, cvt<R>(planes[t0(tr)]), cvt<R>(planes[t1(tr)]), cvt<R>(planes[t2(tr)]));
    }

    // The vertices of a record of nent slots (triples rtr, adjacency radj) at
    // their lanes.
    template <bool R2, typename P64>
    __device__ void load_vertices(const uint32_t *rtr, const uint32_t *radj, int nent, P64 planes64) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int j = s * 64 + lane;
            uint32_t tr = kNoTri;
            if (j < nent) {
                tr = rtr[j];
                adj[j] = adj_unpack(radj[j]);
            }
            const bool v = tr != kNoTri;
            if (v) set_vertex_lds<R2>(s, tr);
            valid[s] = ballot(v);
            if (FILTER) x64[s] = ballot(fabsf(float(W[s])) < kFilterMinW) & valid[s];
            if constexpr (FILTER && R2)
                if (x64[s]) {
                    const Pl<double> *p64 = planes64();
                    if (in_mask(x64[s])) r2[s] = vertex_r2_64(p64, tri[s]);
                }
        }
        wsync();
    }

    __device__ void clear_vertices() {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            valid[s] = 0;
            x64[s] = 0;
            tri[s] = 0;
            X[s] = Y[s] = Z[s] = R(0);
            W[s] = R(1);
            r2[s] = R(0);
            M[s] = 0.f;
        }
    }

    __device__ void refresh_max_r2() {
        R m = R(0);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const R x = in_mask(valid[s]) ? r2[s] : R(0);
            m = x > m ? x : m;
        }
        maxr2 = wave_max_pos(m);
    }

    // One clip by plane e (wave-uniform, test precision), which the caller has
    // put at planes[nb_plane].  Returns kNoClip, kClipped or a failure status.
    // R2: keep r2 and maxr2 up to date.  planes64 (FILTER) gives the cell's
    // FP64 planes, that of e at nb_plane.
    //
    // The scalar unit, which the four SIMDs of a CU share, bounds this code as
    // much as the vector ALUs do: masks are combined as masks, edges that are
    // not on the boundary write to a spare word instead of being branched
    // around, and the wave-wide counts are scalar bit counts.
    template <bool R2, typename P64>
    __device__ __forceinline__ int clip(const Pl<R> &e, P64 planes64) {
        uint64_t rem[S], unsure[S];
        uint64_t flag = 0;
        const float ek = kFilterKappa * (fabsf(float(e.x)) + fabsf(float(e.y)) + fabsf(float(e.z))),
                    ewk = kFilterKappa * kMagW * fabsf(float(e.w));
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const R sv = e.x * X[s] + e.y * Y[s] + e.z * Z[s] + e.w * W[s];
            rem[s] = ballot(sv > R(0)) & valid[s];
            unsure[s] = 0;
            if (FILTER) {
                unsure[s] = (ballot(fabsf(float(sv)) <= fmaf(ek, M[s], ewk)) | x64[s]) & valid[s];
                flag |= unsure[s];
            }
        }
        if (FILTER && flag) {
            // the vertices the filter leaves open are rebuilt from their
            // planes in FP64 and tested in FP64, the FP64 form's own
            // evaluation, so the clip decides as the FP64 form does
            const Pl<double> *p64 = planes64();
            const Pl<double> e64 = p64[nb_plane];
#pragma unroll
            for (int s = 0; s < S; ++s) {
                if (!unsure[s]) continue;
                bool out = false;
                if (in_mask(unsure[s])) out = outside64(p64, tri[s], e64);
                rem[s] = (rem[s] & ~unsure[s]) | ballot(out);
            }
        }
        int nr = 0, nvalid = 0;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            nr += __popcll(rem[s]);
            nvalid += __popcll(valid[s]);
        }
        if (nr == 0) return kNoClip;
        if (nr == nvalid) return RPD_EMPTY_CELL;
        const int pid = nb_plane;
        // boundary edges: edges of removed vertices whose other end is kept
        uint32_t en[S][3];
        uint64_t bd[S][3];
        int nb = 0;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const uint2 ad = adj[s * 64 + lane];
            en[s][0] = ad.x & 0xffffu;
            en[s][1] = ad.x >> 16;
            en[s][2] = ad.y;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const uint32_t v = en[s][k] >> 2;
                uint64_t m = rem[0];
#pragma unroll
                for (int u = 1; u < S; ++u)
                    if (v >> 6 == uint32_t(u)) m = rem[u];
                bd[s][k] = ballot((uint32_t(m >> (v & 63u)) & 1u) == 0u) & rem[s];
                nb += __popcll(bd[s][k]);
            }
        }
        if (nvalid - nr + nb > V) return RPD_VERTEX_OVERFLOW;
        // stage the new vertices: (a, b) of the boundary edge and the kept end
        int o = 0;
#pragma unroll
        for (int s = 0; s < S; ++s) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const uint32_t tr = tri[s];
                const uint32_t a = k == 0 ? t0(tr) : (k == 1 ? t1(tr) : t2(tr)),
                               b = k == 0 ? t1(tr) : (k == 1 ? t2(tr) : t0(tr));
                nvs[in_mask(bd[s][k]) ? mbcnt(bd[s][k], o) : 64 * S + lane] = a | (b << 8) | (en[s][k] << 16);
                o += __popcll(bd[s][k]);
            }
        }
        wsync();
        // The cavity must be a disk: its boundary one simple cycle.  With
        // certified signs it always is: the removed vertices are those of a
        // convex polytope strictly on one side of a plane, which, like the
        // kept ones, form a connected set, and every face meets the plane's
        // side in one contiguous arc, so no face is pinched.  Signs decided in
        // FP64 are checked, as CCComputeBoundary does: every start plane
        // written once, and the walk from one start closes after exactly nb
        // steps.
        if (!FILTER || flag) {
            for (int q = lane; q < nb; q += 64) nxt[nvs[q] & 0xffu] = uint8_t(nvs[q] >> 8);
            wsync();
            bool bad = false;
            for (int q = lane; q < nb; q += 64) bad |= nxt[nvs[q] & 0xffu] != ((nvs[q] >> 8) & 0xffu);
            bool inconsistent = ballot(bad) != 0;
            if (!inconsistent) {
                const uint32_t start = uni(nvs[0]) & 0xffu;
                uint32_t cur = start;
                int steps = 0;
                do {
                    cur = uni(uint32_t(nxt[cur]));
                    ++steps;
                } while (cur != start && cur != 0xffu && steps <= nb);
                inconsistent = !(cur == start && steps == nb);
            }
            wsync();
            for (int q = lane; q < nb; q += 64) nxt[nvs[q] & 0xffu] = 0xff;
            if (inconsistent) return RPD_INCONSISTENT_BOUNDARY;
        }
        // new vertices (plane, a, b) fill the lowest free slots
        int carry = 0;
        uint32_t nw[S];
        uint64_t newm[S];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            valid[s] &= ~rem[s];
            const uint64_t fr = ~valid[s];
            const int q = mbcnt(fr, carry);
            newm[s] = ballot(q < nb) & fr;
            nw[s] = 0;
            if (in_mask(newm[s])) {
                const uint32_t w = nvs[q], a = w & 0xffu, b = (w >> 8) & 0xffu, v = uint32_t(s * 64 + lane);
                nw[s] = w;
                set_vertex<R2>(s, pack3(uint32_t(pid), a, b), e, cvt<R>(planes[a]), cvt<R>(planes[b]));
                sta[a] = uint8_t(v);
                end[b] = uint8_t(v);
                // the kept end's edge now leads here (edge 1: a -> b)
                reinterpret_cast<uint16_t *>(adj)[4 * (w >> 18) + ((w >> 16) & 3u)] = uint16_t(v << 2 | 1u);
                if (S == 1) {
                    // edge 0 (pid -> a) meets the new vertex that ends at a,
                    // edge 2 (b -> pid) the one that starts at b
                    wsync();
                    adj[lane] = make_uint2((uint32_t(end[a]) << 2) | 2u | (w & 0xffff0000u), uint32_t(sta[b]) << 2);
                }
            }
            if (FILTER) {
                const uint64_t il = ballot(fabsf(float(W[s])) < kFilterMinW) & newm[s];
                x64[s] = (x64[s] & ~newm[s]) | il;
                if constexpr (R2)
                    if (il) {
                        const Pl<double> *p64 = planes64();
                        if (in_mask(il)) r2[s] = vertex_r2_64(p64, tri[s]);
                    }
            }
            carry += __popcll(fr);
            valid[s] |= newm[s];
        }
        wsync();
        if constexpr (S > 1) {
#pragma unroll
            for (int s = 0; s < S; ++s)
                if (in_mask(newm[s])) {
                    const uint32_t w = nw[s];
                    adj[s * 64 + lane] = make_uint2((uint32_t(end[w & 0xffu]) << 2) | 2u | (w & 0xffff0000u),
                                                    uint32_t(sta[(w >> 8) & 0xffu]) << 2);
                }
            wsync();
        }
        nb_plane = pid + 1;
        if (R2) refresh_max_r2();
        return kClipped;
    }
};

// LDS of one wave: nvs[64S] and 64 spare words | adj[64S] (8 bytes) | chunk /
// cone planes cpl[64] | go_out flags[16] | planes[P] | plane sources src[P]
// (int32) | nxt, sta, end [P rounded up to 16 each] | tail (finish kernel:
// triangle corners tcor[16][9] and the vertex copy; mixed bisector kernel: FP64
// planes).  The parts of a fixed size come first: their
// addresses are constants in the bisector kernel.
__host__ __device__ constexpr size_t up16(size_t b) { return (b + 15) & ~size_t(15); }
template <typename R, typename RP, bool FILTER, int S, typename PS>
__device__ __forceinline__ void bind_lds(char *L, int P, WaveCell<R, RP, FILTER, S, PS> &c, int **src = nullptr,
                                         Pl<PS> **cpl = nullptr, int **goo = nullptr, char **tail = nullptr) {
    c.nvs = reinterpret_cast<uint32_t *>(L);
    size_t off = 4 * (64 * S + 64);
    c.adj = reinterpret_cast<uint2 *>(L + off);
    off += 8 * 64 * S;
    if (cpl) *cpl = reinterpret_cast<Pl<PS> *>(L + off);
    off += 64 * sizeof(Pl<PS>);
    if (goo) *goo = reinterpret_cast<int *>(L + off);
    off += 64;
    c.planes = reinterpret_cast<Pl<PS> *>(L + off);
    off += up16(size_t(P) * sizeof(Pl<PS>));
    if (src) *src = reinterpret_cast<int *>(L + off);
    off += up16(4 * size_t(P));
    c.nxt = reinterpret_cast<uint8_t *>(L + off);
    c.sta = c.nxt + up16(P);
    c.end = c.sta + up16(P);
    off += 3 * up16(P);
    if (tail) *tail = L + off;
}

// A vertex of the finish kernel's cell as the lane-parallel skip tests read
// it: homogeneous coordinates in the test precision and, for the certified
// form, the magnitude of their terms.
template <typename R>
struct VtxRec {
    R X, Y, Z, W;
    float M;
};
constexpr size_t kVtxRecBytes = 40;  // sizeof(VtxRec<double>), the larger one

// LDS bytes of one wave (pl: bytes of one stored plane; tail: bytes after the
// cone planes and flags)
__host__ __device__ constexpr size_t wave_lds(int P, int S, size_t pl, size_t tail) {
    return 4 * (64 * size_t(S) + 64) + 8 * 64 * size_t(S) + 64 * pl + 64 + up16(P * pl) + up16(4 * size_t(P)) +
           3 * up16(P) + up16(tail);
}
// (the bisector kernel; planes in the test precision, the mixed form with room
// for the FP64 planes)
__host__ __device__ constexpr size_t cells_wave_lds(int form, int P, int S) {
    return wave_lds(P, S, form == RPD_PREC_FP64 ? 32 : 16, form == RPD_PREC_MIXED ? 32 * size_t(P) : 0);
}
// (corners: the finish kernel's triangle corners and vertex copy)
__host__ __device__ constexpr size_t finish_wave_lds(int P, int S, size_t pl, bool corners = false) {
    return wave_lds(P, S, pl, corners ? 16 * 9 * 8 + 64 * size_t(S) * kVtxRecBytes : 0);
}
// The voxel form of the finish kernel: room for one plane more (a strip has
// five cone planes, a triangle four), no corners, the vertex copy in the test
// precision (vr bytes each).
__host__ __device__ constexpr size_t finish_vox_wave_lds(int P, int S, size_t vr) {
    return wave_lds(P + 1, S, 32, 64 * size_t(S) * vr);
}
// LDS the Hessian adds to a finish-kernel wave: per plane 4 sums, per vertex
// slot 4 values and a plane id
__host__ __device__ constexpr size_t hessian_wave_lds(int P, int S) {
    return 32 * size_t(P) + 8 * size_t(P) + 64 * 32;
}

// Units (strips of voxel faces, triangles) that a wave of the finish kernel
// tests at once: a lane per cone plane, 5 or 4 a unit.
constexpr int kStripBatch = 12, kTriBatch = 16;

// Power bisector of the seed S0 and neighbour B in the seed-local frame
// (CCNewPlane, ConvexCell.cl:314-333): unit normal -b/|b|, offset
// d = (|b|^2 + w_B - w_s) / (2|b|), b = B - S0; a border neighbour
// (w <= NO_CELL_LIMITS) gives the plane through B.  Evaluated without
// contraction so that every evaluation of one plane has the same bits.
__device__ __forceinline__ Pl<double> bisector_plane(const double4 &S0, const double4 &B, double &bl) {
#pragma clang fp contract(off)
    const double bx = B.x - S0.x, by = B.y - S0.y, bz = B.z - S0.z;
    const double b2 = bx * bx + by * by + bz * bz;
    bl = sqrt(b2);
    const double ib = 1.0 / bl;
    const double d = B.w <= RPD_NO_CELL_LIMITS ? bl : (b2 + (B.w - S0.w)) * (0.5 * ib);
    return Pl<double>{-bx * ib, -by * ib, -bz * ib, d};
}

// Face f of the bounding cube [-eps, 1000 + eps]^3 in the seed-local frame
// (CCInit, ConvexCell.cl:278-297): x >= -eps, x <= 1000 + eps, then y, z.
__device__ __forceinline__ Pl<double> cube_plane(int f, const double4 &S0, double eps) {
    const int ax = f >> 1;
    const double sc = ax == 0 ? S0.x : (ax == 1 ? S0.y : S0.z);
    const double sgn = (f & 1) ? -1.0 : 1.0;
    const double d = (f & 1) ? (1000.0 + eps) - sc : sc + eps;
    return Pl<double>{ax == 0 ? sgn : 0.0, ax == 1 ? sgn : 0.0, ax == 2 ? sgn : 0.0, d};
}

// Record of a cell: header (sid, nb_plane, nent = 64 * S, kused), planes[P] in
// the storage precision, vertex triples[nent] (kNoTri where none) and their
// adjacency[nent] (adj_pack), plane neighbours[P].  The vertices stay at the
// lanes they have, so that a resumed cell has the lanes, and so the sums, of
// one uninterrupted run, and the adjacency stays as it is.
struct RecHeader {
    int sid, nb_plane, nent, kused;
};

// ---------------------------------------------------------------------------
// Kernel A: the bisector loop (ConvexCell.cl:850-917)
// ---------------------------------------------------------------------------
// What bounds it: instruction issue.  The scalar unit serves the four SIMDs of
// a CU, one instruction a cycle; with 4,200 (mixed form) scalar and 6,700
// vector instructions a cell it was as busy as the vector ALUs, and a version
// with fewer vector but more scalar ones (5,600 / 5,900) ran slower.  Hence the
// adjacency (WaveCell), the masks instead of branches, the single exit of the
// loop, and arguments read again after it instead of kept.  1M seeds in a
// torus at 128^3: 1.50 -> 1.17 ms (mixed), 1.90 -> 1.45 ms (FP64); as a packed
// batch of 300,000 cells, where the loop's branches had counted as divergent,
// 3.45 -> 2.33 ms; 1M nearly cospherical seeds, whose cells all failed the
// filter and went to a second kNN and FP64 pass, 15.5 -> 7.9 ms.
//
// Minimum waves per SIMD the bisector kernel is compiled for (one vertex slot
// per lane): occupancy pays more than the few registers the compiler then
// spills, all in the code of open tests.  At 8 waves the compiler has 78 scalar
// registers and spills more of them than at 7 (94): mixed 1.16 against 1.10 ms,
// 1M cospherical seeds 7.9 against 7.6, FP64 the same.  Wider cells (S > 1,
// re-queue passes) are left unconstrained.
template <typename R, int S>
constexpr int kClipWaves = S > 1 ? 1 : 7;

template <typename R, typename RP, bool FILTER, int S, bool BATCH>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kClipWaves<R, S>)))
void clip_cells_kernel(ClipArgs a) {
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    const int lane = lane_id();
    const int64_t t = blockIdx.x;  // one wave per workgroup

    // planes in the test precision; src[p] records where plane p came from
    // (the neighbour's stored id, or -1 - f for cube face f), so that the
    // record of a queued cell carries the planes in the geometry precision
    // and each plane's neighbour (CCPlaneNeighbour, ConvexCell.cl:329-331)
    WaveCell<R, RP, FILTER, S, R> c;
    Pl<R> *chunk = nullptr;  // planes of the current 64 neighbours
    int *src = nullptr;
    char *tail = nullptr;
    bind_lds(lds_raw, a.P, c, &src, &chunk, nullptr, &tail);
    c.P = a.P;
    c.V = a.V;
    c.lane = lane;

    const int sid = uni(a.ids ? a.ids[t] : int(t));
    // the weight minimum and the domain, in a packed batch those of the
    // cell's request
    double wmin = a.wmin, vs = a.vs;
    int g = a.g;
    const uint8_t *dist = a.dist;
    if constexpr (BATCH) {
        const ReqDesc &d = a.reqs[uni(int(a.req_of[sid]))];
        wmin = uni(d.wmin);
        vs = uni(d.vs);
        g = uni(d.g);
        dist = d.dist;
    }
    const double4 S0 = a.seeds[sid];
    const int K = a.K, P = a.P;
    // resumed cells: record of the state, neighbours used before this pass
    const bool resume = sizeof(RP) == 8 && a.rs_in != nullptr;
    const char *rs_rec = resume ? a.rs_in + size_t(a.rslot[sid]) * size_t(a.rs_in_stride) : nullptr;
    const int kbase = resume ? uni(reinterpret_cast<const RecHeader *>(rs_rec)->kused) : 0;

    // The end of an item that is not queued: its outputs and code.  (The
    // arguments are read again from the kernel's argument area: held in
    // registers through the loop, these pointers were spilled to vector lanes
    // and read back one by one.)
    auto finish = [&](int st, double m0, double m1, double m2, double m3, int ku, bool resumable = false) {
        const auto *k = cold_args();
        if (lane == 0) {
            const int orig = k->perm[sid];
            k->out[orig] = make_double4(m0, m1, m2, m3);
            k->status[orig] = st;
            if (k->kused) k->kused[orig] = kbase + ku;
            reinterpret_cast<RecHeader *>(k->rec + size_t(t) * size_t(k->rec_stride))->sid = -1;
            k->code[t] = uint8_t(!listed_failure(k->exact_final, st)
                                     ? kCodeDone
                                     : uint32_t(st) + (resumable ? kCodeResume : kCodeFailed));
        }
    };

    if (S0.w <= RPD_NO_CELL_LIMITS) {  // border seed: copied (ConvexCell.cl:873-876)
        finish(RPD_SUCCESS, S0.x, S0.y, S0.z, S0.w, 0);
        return;
    }
    for (int i = lane; i < P; i += 64) {
        c.nxt[i] = 0xff;
        c.sta[i] = c.end[i] = 0;
    }

    // Domain cull: a seed whose voxel is d >= 2 voxels (Chebyshev) from every
    // voxel that holds triangles or lies inside has no point of the domain
    // within (d - 1) * vs; once the cell's circumradius about the seed is
    // below that, its restriction to the domain is empty (volume 0, as the
    // reference's apex-outside / no-triangle case, ConvexCell.cl:1067-1079).
    double cull_r2 = 0;
    if (g > 0 && dist) {
        auto vox = [&](double x) { return int(fmin(fmax(x / vs, 0.0), double(g - 1))); };
        // (uni: a load through a pointer that is itself loaded, as in a packed
        // batch, counts as differing by lane, and so would the loop's branches)
        const int d = uni(int(dist[vox(S0.x) + vox(S0.y) * g + vox(S0.z) * g * g]));
        if (d >= 2) cull_r2 = double(d - 1) * vs * double(d - 1) * vs;
    }
    const double wgap = S0.w - wmin;  // >= 0 except for the lightest seeds

    const double eps = g > 0 ? 0.1 : 0.0;  // CUBE_EPSILON, voronoi.cpp:929
    c.clear_vertices();
    // (mixed form) the FP64 planes: the first n64 of them are in p64, the
    // others are made when a test or the record first needs them
    Pl<double> *p64 = reinterpret_cast<Pl<double> *>(tail);
    int n64 = 0;
    if (resume) {
        // ---- the state a previous pass left: planes, then the vertices at
        // their lanes (nent = 64 x the S of the pass that left it) ----------
        const RecHeader hd = *reinterpret_cast<const RecHeader *>(rs_rec);
        const int nent = uni(hd.nent);
        c.nb_plane = uni(hd.nb_plane);
        const Pl<RP> *rpl = reinterpret_cast<const Pl<RP> *>(rs_rec + sizeof(RecHeader));
        const uint32_t *rtr =
            reinterpret_cast<const uint32_t *>(rs_rec + sizeof(RecHeader) + size_t(a.rs_in_P) * sizeof(Pl<RP>));
        const int *rnid = reinterpret_cast<const int *>(rtr + 2 * nent);
        for (int p = lane; p < c.nb_plane; p += 64) {
            c.planes[p] = cvt<R>(rpl[p]);
            if constexpr (FILTER) p64[p] = rpl[p];
            src[p] = rnid[p];
        }
        n64 = c.nb_plane;
        wsync();
        c.template load_vertices<true>(rtr, rtr + nent, nent, [&]() -> const Pl<double> * { return p64; });
    } else {
        // ---- CCInit: bounding cube in the local frame ----------------------
        if (lane < 6) {
            const Pl<double> q = cube_plane(lane, S0, eps);
            c.planes[lane] = cvt<R>(q);
            if constexpr (FILTER) p64[lane] = q;
            src[lane] = -1 - lane;
        }
        wsync();
        c.nb_plane = n64 = 6;
        if (lane < 8) {
            const uint32_t sh = 8 * uint32_t(lane);
            c.set_vertex_lds(0, pack3(uint32_t(kCube0 >> sh) & 0xff, uint32_t(kCube1 >> sh) & 0xff,
                                      uint32_t(kCube2 >> sh) & 0xff));
            const uint32_t w = uint32_t(kCubeAdj.w[lane >> 2] >> (16 * (lane & 3)));
            c.adj[lane] = make_uint2((w & 31u) | ((w & 0x3e0u) << 11), (w >> 10) & 31u);
        }
        c.valid[0] = 0xffull;
        wsync();
    }
    c.refresh_max_r2();

    // ---- neighbour loop -----------------------------------------------------
    // The 64 neighbours of a chunk are loaded one per lane: the plane goes to
    // LDS, the distance |b| and plane offset t (signed distance of the
    // bisector from the seed) stay in registers.  A plane with t >= R, R the distance from the seed to the
    // farthest vertex, cannot cut the cell, so instead of visiting every
    // neighbour the wave ballots for the next neighbour whose plane may cut
    // (t < R) and for the first one where the stop test holds, and jumps to
    // the earlier of the two.  Neighbours in between would neither clip nor
    // stop, so the cell, the stop index and the plane-overflow rule (a full
    // plane list fails at the next neighbour, ConvexCell.cl:316-319) are
    // those of the one-by-one loop.
    const int *nrow = a.knn + t * int64_t(K);
    const double rmarg = sizeof(R) == 8 ? 1.0 + 1e-9 : 1.0 + 2e-4;  // FP32 R may be low by ~1e-4
    // the cell's radius (FP32 forms: the hardware square root, 1 ulp, far
    // inside the radius margin)
    auto radius = [&]() -> double {
        if constexpr (sizeof(R) == 4)
            return double(__builtin_amdgcn_sqrtf(c.maxr2));
        else
            return sqrt(double(c.maxr2));
    };
    double Rcur = radius();
    // Stop test: CCIsSecurityRadiusReached (reference stop, weights ignored)
    // or the exact power stop d (d - 2R) >= w_s - w_min.  The exact stop only
    // ever holds when no later bisector can cut, so the FP32 radius's margin
    // merely delays it.  The reference stop can hold while a later bisector of
    // a lighter seed still cuts; there a delayed stop changes the cell.  So in
    // the mixed form a reference-stop test within the FP32 radius's margin
    // (2R / rmarg < d <= 2R rmarg) that the loop reaches ends the cell with
    // needs_exact_predicates: the FP64 pass decides it.
    const bool plain_stop = a.security_mode == 1 || wgap <= 0;
    const bool ref_stop = FILTER && a.security_mode == 1;
    auto fill64 = [&](int upto) {
        wsync();
        for (int p = n64 + lane; p < upto; p += 64) {
            double bl;
            p64[p] = bisector_plane(S0, a.seeds[src[p]], bl);
        }
        wsync();
        n64 = upto;
    };
    // (the plane about to be clipped by lies at nb_plane)
    auto planes64 = [&]() -> const Pl<double> * {
        if constexpr (FILTER) fill64(c.nb_plane + 1);
        return p64;
    };
    // how the loop ends: the list ran out, the radius was reached, every other
    // seed was used, culled, failed (with the status)
    enum { kRanOut = -1, kReached = -2, kComplete = -3, kCulled = -4 };
    int why = kRanOut, kused = 0;
    for (int base = 0; base < K; base += 64) {
        const int j = base + lane;
        const int cnb = j < K ? nrow[j] : -2;  // -1: list exhausted, -2: past K
        double cdl = 0;
        float ct = 0;
        wsync();  // the previous chunk's planes are no longer read
        if (cnb >= 0) {
            double bl;
            const Pl<double> q = bisector_plane(S0, a.seeds[cnb], bl);
            chunk[lane] = cvt<R>(q);
            cdl = bl;
            ct = float(q.w);
        }
        wsync();
        const uint64_t m_has = ballot(cnb >= 0), m_none = ballot(cnb == -1);
        // the neighbours not visited yet, and the one clipped by last, whose
        // stop test comes with the next choice
        uint64_t left = ~0ull, last = 0;
        for (;;) {
            const double Rs = Rcur * rmarg;
            uint64_t m_stop;
            if (plain_stop)
                m_stop = ballot(cdl * cdl > 4.0 * Rs * Rs);
            else
                m_stop = ballot(cdl * (cdl - 2.0 * Rs) >= wgap);
            m_stop &= m_has & (left | last);
            // skip test in FP32: t is rounded to FP32, so the radius gets a
            // margin well above FP32 rounding (a false candidate only costs a
            // no-op clip)
            const float Rskip = float(Rs) * (1.0f + 1e-6f);
            const uint64_t m_clip = ballot(ct < Rskip) & m_has & left;
            const uint64_t m_end = m_none & left;
            uint64_t m_any = m_stop | m_clip | m_end;
            const bool full = c.nb_plane >= P;
            // a full plane list: the next neighbour's plane cannot be stored
            if (full) m_any = (m_stop & last) ? (m_stop & last) : ((m_has | m_none) & left);
            if (FILTER && ref_stop && !full) {
                const double Rl = Rcur / rmarg;
                const uint64_t m_near = ballot(cdl * cdl > 4.0 * Rl * Rl) & ~m_stop & m_has & (left | last);
                if (m_near && (!m_any || lowest_bit(m_near) < lowest_bit(m_any))) {
                    why = RPD_NEEDS_EXACT_PREDICATES;
                    kused = base + lowest_bit(m_near) + 1;
                    break;
                }
            }
            if (!m_any) {
                if (!full) kused = min(K, base + 64);
                break;  // the next chunk
            }
            const int f = lowest_bit(m_any);
            const uint64_t bit = 1ull << f;
            if (full || !(m_clip & bit)) {
                if (m_stop & bit & (full ? last : ~0ull)) {
                    why = kReached;
                    kused = base + f + 1;
                } else if (m_end & bit) {
                    why = kComplete;  // every other seed has been used
                    if (!full) kused = base + f;
                } else {
                    why = RPD_PLANE_OVERFLOW;
                    kused = base + f + 1;
                }
                break;
            }
            // clip by the plane of neighbour base + f
            const Pl<R> e = chunk[f];
            const int nbid = rlane(cnb, f);
            if (lane == 0) {
                src[c.nb_plane] = nbid;
                c.planes[c.nb_plane] = e;
            }
            const int res = c.template clip<true>(e, planes64);
            kused = base + f + 1;
            if (res >= 0) {
                why = res;
                break;
            }
            if (res == kClipped) {
                Rcur = radius();
                if (double(c.maxr2) * 1.001 < cull_r2) {
                    why = kCulled;
                    break;
                }
            } else if (FILTER) {
                n64 = min(n64, c.nb_plane);  // the plane that did not cut gives way
            }
            left = ~1ull << f;  // past f
            last = bit;
        }
        if (why != kRanOut) break;
    }
    if (why >= 0 || why == kCulled) {
        finish(why >= 0 ? why : int(RPD_SUCCESS), 0.0, 0.0, 0.0, 0.0, kused);
        return;
    }
    const auto *k = cold_args();
    // a list that holds every other seed leaves nothing to test: the cell is
    // exact once the list is used up (the reference reads past the seeds there)
    int64_t n_seeds = k->n_seeds;
    if constexpr (BATCH) n_seeds = k->reqs[uni(int(k->req_of[sid]))].n_seeds;
    if (why == kRanOut && int64_t(kbase) + K >= n_seeds - 1) why = kComplete;

    // debug counters (ConvexCell.cl:887-911): K used where the security
    // radius was reached, P and V once the neighbour loop is done
    if (k->dcnt && lane == 0) {
        if (why == kReached) {
            const int ku = min(kbase + kused, 256);
            atomicMax(k->dcnt + kDcMax + 0, ku);
            atomicAdd(k->dcnt + kDcHistK + ku, 1);
        }
        int nv = 0;
#pragma unroll
        for (int s = 0; s < S; ++s) nv += __popcll(c.valid[s]);
        atomicMax(k->dcnt + kDcMax + 1, c.nb_plane);
        atomicAdd(k->dcnt + kDcHistP + min(c.nb_plane, 255), 1);
        atomicMax(k->dcnt + kDcMax + 2, nv);
        atomicAdd(k->dcnt + kDcHistV + min(nv, 256), 1);
    }

    // A finished cell is queued for restriction + integration.  A cell whose
    // list ran out keeps its state when there is room, so that the next pass
    // goes on from here with the neighbours after the last one used.
    const bool ran_out = why == kRanOut;
    if (!ran_out || k->rs_out) {
        const int64_t slot = ran_out ? k->rs_base + t : t;
        // the cell's state as a record: header, planes in the geometry
        // precision, vertex triples and adjacency; P planes' room
        char *rec = ran_out ? k->rs_out + size_t(slot) * size_t(k->rs_out_stride)
                            : k->rec + size_t(slot) * size_t(k->rec_stride);
        Pl<RP> *rpl = reinterpret_cast<Pl<RP> *>(rec + sizeof(RecHeader));
        uint32_t *rtr = reinterpret_cast<uint32_t *>(rec + sizeof(RecHeader) + size_t(P) * sizeof(Pl<RP>));
        int *rnid = reinterpret_cast<int *>(rtr + 128 * S);
        if (lane == 0) {
            *reinterpret_cast<RecHeader *>(rec) = RecHeader{sid, c.nb_plane, 64 * S, kbase + kused};
            if (ran_out) {
                k->rslot[sid] = int(slot);
                k->lastnb[sid] = nrow[K - 1];
            } else {
                k->code[t] = kCodeQueued;
            }
        }
        wsync();
        if constexpr (FILTER) fill64(c.nb_plane);
        for (int p = lane; p < c.nb_plane; p += 64) {
            if constexpr (FILTER)
                rpl[p] = p64[p];
            else
                rpl[p] = cvt<RP>(c.planes[p]);
            rnid[p] = src[p];
        }
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const bool v = in_mask(c.valid[s]);
            rtr[64 * s + lane] = v ? c.tri[s] : kNoTri;
            if (v) rtr[64 * S + 64 * s + lane] = adj_pack(c.adj[64 * s + lane]);
        }
    }
    if (ran_out) finish(RPD_SECURITY_RADIUS_NOT_REACHED, 0.0, 0.0, 0.0, 0.0, kused, k->rs_out != nullptr);
}

// The failure lists of a bisector kernel's items, from their codes: one
// atomic per list and workgroup of 4096 items, entries in item order within a
// workgroup.  Counters as in ClipArgs (cnt[14]: cells to resume, listed in
// sec); *q counts the queued items.  The last workgroup to end copies *q and
// the counters to mapped pinned host memory (nullable) and clears *q, which is
// otherwise left to the caller; q[1], its ticket, it leaves cleared.
struct ListArgs {
    const uint8_t *code;  // room for whole 16-byte groups
    const int *ids;       // nullable: item t is stored id t
    int64_t n;
    int *cnt, *eo, *sec, *q;
    int *q_host, *cnt_host;
};
constexpr int kListPer = 16;    // items of a thread
constexpr int kListBlock = 256;
__global__ __launch_bounds__(kListBlock) void list_failures_kernel(ListArgs a) {
    __shared__ int tot[4][kListBlock / 64], base[3], hist[16], last;
    const int tid = int(threadIdx.x), lane = lane_id(), wv = tid >> 6;
    if (tid < 16) hist[tid] = 0;
    __syncthreads();
    const int64_t i0 = (int64_t(blockIdx.x) * kListBlock + tid) * kListPer;
    uint32_t w[4] = {0, 0, 0, 0};
    if (i0 < a.n) {
        const uint4 v = *reinterpret_cast<const uint4 *>(a.code + i0);
        w[0] = v.x, w[1] = v.y, w[2] = v.z, w[3] = v.w;
    }
    auto code = [&](int j) -> uint32_t { return i0 + j < a.n ? (w[j >> 2] >> (8 * (j & 3))) & 255u : 0u; };
    // exact, overflow, resume, queued
    int num[4] = {0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < kListPer; ++j) {
        const uint32_t cd = code(j);
        const bool failed = cd >= kCodeFailed, resume = cd >= kCodeResume, exact = exact_failure(int(cd & 15u));
        num[0] += failed && !resume && exact;
        num[1] += failed && !resume && !exact;
        num[2] += resume;
        num[3] += cd == kCodeQueued;
        if (failed) atomicAdd(&hist[cd & 15u], 1);
    }
    int at[3];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int incl = wave_incl_scan_op(num[k], 0, [](int x, int y) { return x + y; });
        if (k < 3) at[k] = incl - num[k];
        if (lane == 63) tot[k][wv] = incl;
    }
    __syncthreads();
    if (tid < 4) {
        int n = 0;
        for (int v = 0; v < kListBlock / 64; ++v) {
            const int m = tot[tid][v];
            tot[tid][v] = n;
            n += m;
        }
        if (tid == 3) {
            if (n) atomicAdd(a.q, n);
        } else {
            base[tid] = n ? atomicAdd(a.cnt + (tid == 2 ? 14 : tid), n) : 0;
        }
    } else if (tid >= 64 && tid < 64 + RPD_STATUS_NUM) {
        const int st = tid - 64;
        if (hist[st]) atomicAdd(a.cnt + 2 + st, hist[st]);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 3; ++k) at[k] += base[k] + tot[k][wv];
#pragma unroll
    for (int j = 0; j < kListPer; ++j) {
        const uint32_t cd = code(j);
        if (cd < kCodeFailed) continue;
        const int sid = a.ids ? a.ids[i0 + j] : int(i0 + j);
        if (cd >= kCodeResume)
            a.sec[at[2]++] = sid;
        else if (exact_failure(int(cd & 15u)))
            a.eo[-1 - at[0]++] = sid;
        else
            a.eo[at[1]++] = sid;
    }
    if (!a.q_host && !a.cnt_host) return;
    // the last workgroup's copy to the host
    __threadfence();
    __syncthreads();
    if (tid == 0) last = atomicAdd(a.q + 1, 1) == int(gridDim.x) - 1;
    __syncthreads();
    if (!last) return;
    __threadfence();
    if (a.cnt_host && tid < kFailCounters)
        a.cnt_host[tid] = __hip_atomic_load(a.cnt + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (tid == 0) {
        if (a.q_host) {
            *a.q_host = __hip_atomic_load(a.q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            a.q[0] = 0;
        }
        a.q[1] = 0;
    }
    __threadfence_system();
}

// vface[q] of a voxel domain's face: x, y, z (10 bits each) of its lowest
// lattice point and, in bits 30-31 of .x, the axis it lies across; .y holds
// kVfaceUp when its triangles' normal points along that axis, kVfacePrev when
// the face before it (along x, or along y for faces across x) exists with the
// same normal, and from bit 2 the number of faces from it on that do, itself
// included.
constexpr uint32_t kVfaceUp = 1u, kVfacePrev = 2u;

// tinfo[q] of a triangle-list entry (voxel v): x is v packed as
// z<<20 | y<<10 | x; (z << 32 | y) a 64-bit mask with bit
// (dz+2)*25 + (dy+2)*5 + (dx+2) set when the voxel v + (dx, dy, dz), within 2
// voxels of v per axis, precedes v in scan order and its list holds the same
// triangle (such offsets are the ones below the centre, bit 62, of the
// 5x5x5 block, so the bits are 0..61); kTinfoFar when a preceding voxel
// whose list holds it lies farther away.
constexpr uint64_t kTinfoFar = 1ull << 63;

// Mask of the preceding offsets of the 5x5x5 block (bits as in tinfo) that
// keep voxel (x, y, z) inside the box [mn, mx].
__device__ __forceinline__ uint64_t box_near(int x, int y, int z, const int *mn, const int *mx) {
    // per axis: the offsets d in [-2, 2] with mn <= v + d <= mx, bit d + 2
    auto axis = [](int v, int lo, int hi) -> uint32_t {
        const int a = max(lo - v, -2), b = min(hi - v, 2);
        return a > b ? 0u : ((1u << (b - a + 1)) - 1u) << (a + 2);
    };
    const uint32_t ax = axis(x, mn[0], mx[0]), ay = axis(y, mn[1], mx[1]), az = axis(z, mn[2], mx[2]);
    // the (dy, dx) plane: bit 5 (dy + 2) + dx + 2, i.e. ax repeated at 5 bit k
    // of ay (no carries: the copies are 5 bits apart)
    const uint32_t ry = (ay & 1u) | ((ay & 2u) << 4) | ((ay & 4u) << 8) | ((ay & 8u) << 12) | ((ay & 16u) << 16);
    const uint64_t pyx = uint64_t(ax) * uint64_t(ry);
    // planes dz = -2, -1, 0 at bits 0, 25, 50 (dz > 0 never precedes); bits
    // past 63 of the dz = 0 plane are offsets after the centre, never set
    const uint64_t rz = ((az & 1u) ? 1ull : 0ull) | ((az & 2u) ? 1ull << 25 : 0ull) | ((az & 4u) ? 1ull << 50 : 0ull);
    return pyx * rz;
}

// ---------------------------------------------------------------------------
// Kernel B: restriction to the domain (ConvexCell.cl:918-1116) and the
// integration (CCExportBaryVolume, ConvexCell.cl:577-619) of queued cells.
//
// W waves share one cell (W = 1 for large queues, up to 8 for the short
// re-queue passes whose run time is set by their heaviest cell): every wave
// rebuilds the cell and its list of triangles (or strips), the batches of 16
// (12) units go round the waves.  Each unit starts from the same backed-up
// cell, so its contribution does not depend on which wave computes it.  A
// batch's contributions are added in increasing order, and the batches' sums
// in the batches' order: with W = 1 as they come, with W > 1 from LDS by wave
// 0.  Both make the same additions, so the result of a cell in this form is the
// same bit for bit for every W and every packed batch it is in.
//
// Cone planes are built lane-parallel, 16 triangles x 4 planes per batch.  A
// triangle one of whose four planes removes every vertex of the cell with a
// margin contributes nothing: the reference clips it and ends with
// empty_cell at that plane at the latest (vertices created by earlier cone
// planes lie in the convex hull of the removed ones).  The shortcut is taken
// only when the caps guarantee that those earlier clips could not overflow
// either (at most 3 more planes, at most 2 more vertices per clip), so the
// outcome is the reference's.
//
// VOX: a domain of voxel faces.  What bounds this kernel is the work per
// boundary triangle (cone planes, skip tests, clips, one integration per
// clipped one: 81% of its time on the 1M-seed torus), so a cell is cut by
// strips of faces instead: the faces come from one entry each (a triangle is
// listed by 9 to 12 voxels), side by side ones are one convex unit, their cone
// planes have two components, and five clips and one integration serve two
// triangles or more.  The apex lies in the middle of the cell's box, not in
// its first voxel: cones then only meet the cell where the boundary does.
// 1M seeds, torus in 128^3, mixed: the launch went from 1.43 to 0.67 ms with
// strips, later to 0.61, and to 0.53 ms with batches of equal work and with
// integer and folded wave reductions (VALU-bound: about 1,500 instructions a
// cell before those); 1,000 seeds, sphere in 96^3, where a cell meets hundreds
// of triangles: the whole solve from 3.3 to 1.16 ms with strips.
// ---------------------------------------------------------------------------
template <typename R, typename RP, bool FILTER, int S, bool HESS, bool BATCH, bool VOX>
// 4 waves per SIMD for S = 1 (128 VGPRs): measured at 1M seeds against 5 and
// 6, whose spills cost more than the extra residency gives.  HESS: the
// Hessian variant (one wave per cell).
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(S > 1 ? 1 : (HESS ? 3 : 4))))
void finish_cells_kernel(ClipArgs a, int nq, int W) {
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    const int lane = lane_id();
    const int wv = uni(int(threadIdx.x >> 6));  // wave-uniform: lets ids, seeds and pointers live in SGPRs
    const int wpb = blockDim.x >> 6;
    const int cpb = wpb / W;  // cells per block; W > 1 implies cpb == 1
    const int ci = wv / W, sub = wv - ci * W;
    const int item = int(blockIdx.x) * cpb + ci;
    if (item >= nq) return;  // uniform over the waves of a cell
    const int slot = a.slots ? uni(a.slots[item]) : item;
    if (reinterpret_cast<const RecHeader *>(a.rec + size_t(slot) * size_t(a.rec_stride))->sid < 0)
        return;  // not queued

    char *cell_l = lds_raw + size_t(ci) * a.cell_stride;
    int *fails = reinterpret_cast<int *>(cell_l);                  // [W][2]
    // the units (triangles or strips) that the cell meets: collected by every
    // wave of the cell for itself, all writing the same values
    int *tu = reinterpret_cast<int *>(cell_l + 64);  // [T]
    double *bsum = reinterpret_cast<double *>(cell_l + 64 + up16(4 * size_t(a.T)));  // [4] a batch, W > 1 only
    WaveCell<R, RP, FILTER, S> c;
    int *goo = nullptr;
    Pl<RP> *cpl = nullptr;
    char *tail = nullptr;
    // VOX: a strip's fifth cone plane has room of its own, so that the plane
    // cap is met no earlier than with triangles.  (The vertex cap is met less
    // often: of 3,600 cells of 62 vertices in random domains, without passes
    // to grow the cap, 362 by lists and none by strips, whose cones' planes
    // meet in the middle of the cell, so that the first halves it.)
    const int P = VOX ? a.P + 1 : a.P;
    bind_lds(lds_raw + size_t(cpb) * a.cell_stride + size_t(wv) * a.lds_stride, P, c, nullptr, &cpl, &goo, &tail);
    double *tcor = reinterpret_cast<double *>(tail);  // (not VOX)
    c.P = P;
    c.V = a.V;
    c.lane = lane;

    const char *rec = a.rec + size_t(slot) * size_t(a.rec_stride);
    const RecHeader hd = *reinterpret_cast<const RecHeader *>(rec);
    const int sid = uni(hd.sid);
    if constexpr (BATCH) {
        bind_request(a, sid);
        if (a.only && (a.only == 1) != (a.vface != nullptr || a.g == 0)) return;
    }
    const int kused = uni(hd.kused);
    const int nent = uni(hd.nent);
    c.nb_plane = uni(hd.nb_plane);
    const Pl<RP> *rpl = reinterpret_cast<const Pl<RP> *>(rec + sizeof(RecHeader));
    const uint32_t *rtr =
        reinterpret_cast<const uint32_t *>(rec + sizeof(RecHeader) + size_t(a.rec_P) * sizeof(Pl<RP>));
    for (int p = lane; p < c.nb_plane; p += 64) c.planes[p] = rpl[p];
    for (int i = lane; i < P; i += 64) {
        c.nxt[i] = 0xff;
        c.sta[i] = c.end[i] = 0;
    }
    wsync();
    c.clear_vertices();
    c.template load_vertices<false>(rtr, rtr + nent, nent, 0);
    int nvalid = 0;
#pragma unroll
    for (int s = 0; s < S; ++s) nvalid += __popcll(c.valid[s]);
    // (the vertices' distances from the seed are not kept here: the
    // restriction takes the cell's radius in FP64 below)

    const double4 S0 = a.seeds[sid];
    const int orig = a.perm[sid];
    auto finish = [&](int st, double m0, double m1, double m2, double m3) {
        if (sub == 0 && lane == 0) {
            a.out[orig] = make_double4(m0, m1, m2, m3);
            a.status[orig] = st;
            if (a.kused) a.kused[orig] = kused;
            note_failure(a, sid, st, slot);
        }
    };
    auto fail = [&](int st) {
        if (!(exact_failure(st) && cold_args()->keep_exact)) finish(st, 0.0, 0.0, 0.0, 0.0);
    };

    // vertex coordinates in the geometry precision RP: the registers when
    // R == RP, else recomputed from the stored RP planes
    auto vertex_rp = [&](int s, RP &Ax, RP &Ay, RP &Az) {
        if (sizeof(R) == sizeof(RP)) {
            const RP iw = RP(1) / RP(c.W[s]);
            Ax = RP(c.X[s]) * iw;
            Ay = RP(c.Y[s]) * iw;
            Az = RP(c.Z[s]) * iw;
        } else {
            const uint32_t tr = c.tri[s];
            RP X, Y, Z, W;
            vertex_from_planes<RP>(c.planes[t0(tr)], c.planes[t1(tr)], c.planes[t2(tr)], X, Y, Z, W);
            const RP iw = RP(1) / W;
            Ax = X * iw;
            Ay = Y * iw;
            Az = Z * iw;
        }
    };

    // ---- integration (CCExportBaryVolume): factor/6 * (moments, volume) of
    // the current cell in the local frame, FP64 wave sums; every lane of row r
    // (16 lanes) of the wave returns component r (x, y, z moment, volume) ----
    const RP vol_eps2 = sizeof(RP) == 8 ? RP(1e-12) : RP(1e-6);  // voronoi.cpp:919-922
    // the vertex copy of the skip tests
    VtxRec<R> *vtx = reinterpret_cast<VtxRec<R> *>(VOX ? tcor : tcor + 16 * 9);
    // Hessian sums: per record plane 4 doubles (area-weighted centroid in the
    // local frame, area), and for their reduction a mask of lanes per record
    // plane and 4 doubles per lane
    double *hacc = nullptr, *hval = nullptr;
    unsigned long long *hmask = nullptr;
    const int nbk = c.nb_plane;  // the record's planes; cone planes come after
    const bool hfull = HESS && a.hc != 1;  // centroids beside the areas
    if (HESS) {
        hacc = reinterpret_cast<double *>(reinterpret_cast<char *>(vtx) +
                                          64 * size_t(S) * (VOX ? sizeof(VtxRec<R>) : kVtxRecBytes));
        hval = hacc + 4 * size_t(P);
        hmask = reinterpret_cast<unsigned long long *>(hval + 4 * 64);
        for (int i = lane; i < 4 * nbk; i += 64) hacc[i] = 0.0;
        for (int i = lane; i < nbk; i += 64) hmask[i] = 0;
        wsync();
    }
    auto integrate = [&](double factor) -> double {
        RP sw = 0, sx = 0, sy = 0, sz = 0;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const bool vok = in_mask(c.valid[s]);
            // per plane k of the vertex: area (CCExportBaryVolumeAndArea,
            // ConvexCell.cl:621-674) and area-weighted centroid
            double ha[3] = {0.0, 0.0, 0.0}, hx[3] = {0.0, 0.0, 0.0}, hy[3] = {0.0, 0.0, 0.0},
                   hz[3] = {0.0, 0.0, 0.0};
            uint32_t tr = c.tri[s];
            if (!HESS && !vok) continue;
            if (vok) {
                RP Ax, Ay, Az;
                vertex_rp(s, Ax, Ay, Az);
                const Pl<RP> pl[3] = {c.planes[t0(tr)], c.planes[t1(tr)], c.planes[t2(tr)]};
                if constexpr (sizeof(RP) == 8) {
                    // The reference's six tetrahedra (seed, its foot on plane
                    // i, its foot on the line of planes i and j, vertex A) are
                    // path simplices: the three legs are orthogonal.  With
                    // unit normals, a_i = n_i.A, t = n_k x n_q and T =
                    // (t.A)/|t|^2, the line (k, q) gives the two volumes
                    // (times 6) a_k (a_q - a_k n_k.n_q) T and a_q (a_k - a_q
                    // n_k.n_q) T, and the feet are a_i n_i and A - T t: three
                    // divisions instead of six, and no determinants.
                    RP av[3], ws[3] = {0, 0, 0};
#pragma unroll
                    for (int k = 0; k < 3; ++k) av[k] = pl[k].x * Ax + pl[k].y * Ay + pl[k].z * Az;
                    RP lx = 0, ly = 0, lz = 0;
#pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        const int q = (k + 1) % 3;
                        const Pl<RP> &p = pl[k], &r = pl[q];
                        const RP tx = p.y * r.z - p.z * r.y, ty = p.z * r.x - p.x * r.z, tz = p.x * r.y - p.y * r.x;
                        const RP c2 = tx * tx + ty * ty + tz * tz;
                        const RP d = p.x * r.x + p.y * r.y + p.z * r.z;
                        // (nearly) parallel planes: the reference's foot on the line is the seed
                        const RP T = c2 < vol_eps2 ? RP(0) : (tx * Ax + ty * Ay + tz * Az) / c2;
                        const RP ek = (av[q] - av[k] * d) * T, eq = (av[k] - av[q] * d) * T;
                        const RP wk = av[k] * ek, wq = av[q] * eq;
                        ws[k] += wk;
                        ws[q] += wq;
                        const RP wt = (wk + wq) * T;
                        lx += wt * tx;
                        ly += wt * ty;
                        lz += wt * tz;
                        if (HESS) {
                            // per plane of the line, the triangle (foot on the
                            // plane, foot on the line, A): its area and centroid
                            const double f2 = -0.5 * factor;
                            const double ak = f2 * ek, aq = f2 * eq;
                            const double Lx = Ax - (T * tx) * 0.5, Ly = Ay - (T * ty) * 0.5, Lz = Az - (T * tz) * 0.5;
                            ha[k] += ak;
                            hx[k] += ak * (2.0 * Lx + av[k] * p.x) / 3.0;
                            hy[k] += ak * (2.0 * Ly + av[k] * p.y) / 3.0;
                            hz[k] += ak * (2.0 * Lz + av[k] * p.z) / 3.0;
                            ha[q] += aq;
                            hx[q] += aq * (2.0 * Lx + av[q] * r.x) / 3.0;
                            hy[q] += aq * (2.0 * Ly + av[q] * r.y) / 3.0;
                            hz[q] += aq * (2.0 * Lz + av[q] * r.z) / 3.0;
                        }
                    }
                    // centroid of (seed, a n, A - T t, A)
                    const RP w = ws[0] + ws[1] + ws[2];
                    const RP b0 = ws[0] * av[0], b1 = ws[1] * av[1], b2 = ws[2] * av[2];
                    sw += w;
                    sx += RP(0.5) * w * Ax + RP(0.25) * (b0 * pl[0].x + b1 * pl[1].x + b2 * pl[2].x - lx);
                    sy += RP(0.5) * w * Ay + RP(0.25) * (b0 * pl[0].y + b1 * pl[1].y + b2 * pl[2].y - ly);
                    sz += RP(0.5) * w * Az + RP(0.25) * (b0 * pl[0].z + b1 * pl[1].z + b2 * pl[2].z - lz);
                } else {
                    // FP32 form: the reference's evaluation
                    const RP ACx = -Ax, ACy = -Ay, ACz = -Az;  // seed at the origin
                    RP opx[3], opy[3], opz[3], olx[3], oly[3], olz[3];
    #pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        const RP nn = pl[k].x * pl[k].x + pl[k].y * pl[k].y + pl[k].z * pl[k].z;
                        const RP f = (ACx * pl[k].x + ACy * pl[k].y + ACz * pl[k].z) / nn;
                        opx[k] = ACx - f * pl[k].x;
                        opy[k] = ACy - f * pl[k].y;
                        opz[k] = ACz - f * pl[k].z;
                    }
    #pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        const Pl<RP> &p = pl[k], &q = pl[(k + 1) % 3];
                        const RP cx = p.y * q.z - p.z * q.y, cy = p.z * q.x - p.x * q.z, cz = p.x * q.y - p.y * q.x;
                        const RP c2 = cx * cx + cy * cy + cz * cz;
                        const RP pp = p.x * p.x + p.y * p.y + p.z * p.z, qq = q.x * q.x + q.y * q.y + q.z * q.z;
                        if (c2 < vol_eps2 * pp * qq) {
                            olx[k] = oly[k] = olz[k] = RP(0);
                        } else {
                            const RP f = (ACx * cx + ACy * cy + ACz * cz) / c2;
                            olx[k] = f * cx;
                            oly[k] = f * cy;
                            olz[k] = f * cz;
                        }
                    }
    #pragma unroll
                    for (int k = 0; k < 3; ++k) {
    #pragma unroll
                        for (int st = 0; st < 2; ++st) {
                            const int j = (k + 3 - st) % 3;
                            // det3 of rows AC, onPlane_k, onLine_j (ConvexCell.cl:72-77)
                            const RP d = ACx * (opy[k] * olz[j] - opz[k] * oly[j]) - opx[k] * (ACy * olz[j] - ACz * oly[j]) +
                                         olx[j] * (ACy * opz[k] - ACz * opy[k]);
                            const RP w = st ? d : -d;
                            sw += w;
                            sx += w * (Ax + RP(0.25) * (ACx + opx[k] + olx[j]));
                            sy += w * (Ay + RP(0.25) * (ACy + opy[k] + oly[j]));
                            sz += w * (Az + RP(0.25) * (ACz + opz[k] + olz[j]));
                            if (HESS) {
                                // det3 of rows onPlane_k, onLine_j, n_k, halved
                                const double dt = double(opx[k]) * (double(oly[j]) * pl[k].z - double(olz[j]) * pl[k].y) -
                                                  double(opy[k]) * (double(olx[j]) * pl[k].z - double(olz[j]) * pl[k].x) +
                                                  double(opz[k]) * (double(olx[j]) * pl[k].y - double(oly[j]) * pl[k].x);
                                const double ar = (st ? 0.5 : -0.5) * factor * dt;
                                ha[k] += ar;
                                hx[k] += ar * (double(Ax) + (double(opx[k]) + double(olx[j])) / 3.0);
                                hy[k] += ar * (double(Ay) + (double(opy[k]) + double(oly[j])) / 3.0);
                                hz[k] += ar * (double(Az) + (double(opz[k]) + double(olz[j])) / 3.0);
                            }
                        }
                    }
                }
            }
            if (HESS) {
                // per plane, in a fixed order: plane slot k, then lane; the
                // lane that owns plane p (p = lane, lane + 64, ...) adds.  The
                // lanes that hold a vertex of plane p are the bits of
                // hmask[p] (an OR: the order in which they arrive does not
                // matter), so that a plane reads its own vertices, two or
                // three for each k, and not every lane's, which had bound
                // the Hessian form: 50,021 seeds, torus in a grid of 96^3,
                // 8,567 cells on the boundary: 792 -> 387 us.
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const int pk = int(k == 0 ? t0(tr) : (k == 1 ? t1(tr) : t2(tr)));
                    if (vok && pk < nbk) {
                        atomicOr(hmask + pk, 1ull << lane);
                        if (hfull) {
                            hval[4 * lane + 0] = hx[k];
                            hval[4 * lane + 1] = hy[k];
                            hval[4 * lane + 2] = hz[k];
                        }
                        hval[4 * lane + 3] = ha[k];
                    }
                    wsync();
                    for (int p = lane; p < nbk; p += 64) {
                        unsigned long long m = hmask[p];
                        if (m == 0) continue;
                        hmask[p] = 0;
                        double e0 = 0.0, e1 = 0.0, e2 = 0.0, e3 = 0.0;
                        for (; m; m &= m - 1) {
                            const int j = __builtin_ctzll(m);
                            if (hfull) {
                                e0 += hval[4 * j + 0];
                                e1 += hval[4 * j + 1];
                                e2 += hval[4 * j + 2];
                            }
                            e3 += hval[4 * j + 3];
                        }
                        if (hfull) {
                            hacc[4 * p + 0] += e0;
                            hacc[4 * p + 1] += e1;
                            hacc[4 * p + 2] += e2;
                        }
                        hacc[4 * p + 3] += e3;
                    }
                    wsync();
                }
            }
        }
        return factor / 6.0 * wave_sum4(double(sx), double(sy), double(sz), double(sw));
    };

    // ---- restriction to the domain grid --------------------------------------
    bool add_volume = true;
    int ntri = 0;
    double rcell = 0;  // largest distance of a vertex from the seed (upper bound)
    double P0x = 0, P0y = 0, P0z = 0;  // apex, global frame
    int vmx[3] = {0, 0, 0};
    if (a.g > 0) {
        const int g = a.g;
        const double vs = a.vs;
        // Box of the vertices in voxels, starting from 1000 and 0 as the
        // reference does, (int)(b / vs) clamped to [0, g-1]
        // (ConvexCell.cl:939-940); clamped in floating point first so that
        // inf/NaN from a degenerate vertex cannot produce an out-of-grid range.
        // Division, clamp and truncation are monotone, so the wave reduces
        // integers: the position in 1/1024 voxels, whose high bits are the
        // voxel, as unsigned maxima of one DPP instruction a step (7 FP64
        // reductions had been 245 of the 1,500 VALU instructions of a cell;
        // 1M seeds, torus in 128^3).
        const double top = double(g - 1), x1000 = 1000.0 / vs;
        uint32_t qn[3] = {0, 0, 0}, qx[3] = {0, 0, 0};  // (lows complemented)
        double vr2 = 0.0;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            if (!in_mask(c.valid[s])) continue;
            RP lx, ly, lz;
            vertex_rp(s, lx, ly, lz);
            vr2 = fmax(vr2, double(lx) * double(lx) + double(ly) * double(ly) + double(lz) * double(lz));
            const double v[3] = {(S0.x + double(lx)) / vs, (S0.y + double(ly)) / vs, (S0.z + double(lz)) / vs};
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                qn[d] = max(qn[d], ~uint32_t(fmin(fmax(fmin(x1000, v[d]), 0.0), top) * 1024.0));
                qx[d] = max(qx[d], uint32_t(fmin(fmax(v[d], 0.0), top) * 1024.0));
            }
        }
        // (rounded up: an upper bound is what the tests below need)
        rcell = sqrt(double(wave_max_pos(float(vr2) * (1.0f + 0x1.0p-22f))));
        int vmn[3];
        double mid[3];  // middle of the box, in voxels (VOX)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const uint32_t lo = ~wave_max_u32(qn[d]), hi = wave_max_u32(qx[d]);
            vmn[d] = int(lo >> 10);
            vmx[d] = int(hi >> 10);
            if (vmx[d] < vmn[d]) vmx[d] = vmn[d];
            mid[d] = fmin(fmax((double(lo) + double(hi)) * (0.5 / 1024.0), double(vmn[d])), double(vmx[d]));
        }
        if constexpr (VOX) {
            // ---- voxel domain: every boundary face is a voxel face, and the
            // class of every voxel is known -------------------------------
            // Apex: near the middle of the cell's box, off the lattice and
            // off the middle planes of voxels, in a voxel of known class.
            // From inside the cell the cones only meet it where the boundary
            // does, so fewer strips are clipped than from the box's first
            // voxel.
            int va[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                va[d] = uni(min(int(mid[d]), vmx[d]));
                const double fr = fmin(fmax(mid[d] - double(va[d]), 0.25), 0.75);
                const double P0 = (double(va[d]) + fr + (kApexFrac[d] - 0.5)) * vs;
                if (d == 0) P0x = P0;
                if (d == 1) P0y = P0;
                if (d == 2) P0z = P0;
            }
            const int in_domain = uni(int(a.centre[va[0] + va[1] * g + va[2] * g * g]));
            // Strips: the faces of one orientation side by side along x (faces
            // across y or z) or y (faces across x) within the box.  Faces are
            // listed once, at their lowest lattice point, so the box's faces
            // are one range per row of lattice points; a face whose neighbour
            // before it lies in the box too belongs to that one's strip.
            // Faces on a side of the box inside the frame only touch the
            // cell, which lies on one side of them.
            int nu = 0;
            const int g1 = g + 1;
            const int nx = vmx[0] - vmn[0] + 2, ny = vmx[1] - vmn[1] + 2, nz = vmx[2] - vmn[2] + 2;
            int *seg_off = reinterpret_cast<int *>(cpl), *seg_a = seg_off + 64;
            const int nrows = ny * nz;
            for (int rb = 0; rb < nrows; rb += 64) {
                const int r = rb + lane;
                int sa = 0, len = 0;
                if (r < nrows) {
                    const int id0 = vmn[0] + (vmn[1] + r % ny) * g1 + (vmn[2] + r / ny) * g1 * g1;
                    sa = a.vfoffs[id0];
                    len = a.vfoffs[id0 + nx] - sa;
                }
                const int off = wave_excl_scan(len);
                const int total = uni(rlane(off + len, 63));
                if (total == 0) continue;
                seg_off[lane] = off;
                seg_a[lane] = sa;
                wsync();
                for (int base = 0; base < total; base += 64) {
                    const int e = base + lane;
                    bool keep = false;
                    int q = -1;
                    if (e < total) {
                        // last row whose offset is <= e (empty rows never win)
                        int lo = 0, hi = 63;
                        while (lo < hi) {
                            const int m = (lo + hi + 1) >> 1;
                            if (seg_off[m] <= e)
                                lo = m;
                            else
                                hi = m - 1;
                        }
                        q = seg_a[lo] + (e - seg_off[lo]);
                        const uint2 ent = a.vface[q];
                        const int p[3] = {int(ent.x & 1023u), int((ent.x >> 10) & 1023u), int((ent.x >> 20) & 1023u)};
                        const int ax = int(ent.x >> 30);
                        const bool prev = (ent.y & kVfacePrev) != 0;
                        keep = true;
#pragma unroll
                        for (int d = 0; d < 3; ++d)
                            keep = keep && (d == ax ? (p[d] > vmn[d] || p[d] == 0) && (p[d] <= vmx[d] || p[d] == g)
                                                    : p[d] <= vmx[d]);
                        const bool first = ax == 0 ? p[1] == vmn[1] : p[0] == vmn[0];
                        keep = keep && (first || !prev);
                    }
                    const uint64_t m = ballot(keep);
                    if (keep && nu + mbcnt(m) < a.T) tu[nu + mbcnt(m)] = q;
                    nu += __popcll(m);
                }
                wsync();  // the next rows overwrite seg_off / seg_a
            }
            if (nu > a.T) {
                // the cap a re-queue pass needs for this cell
                if (sub == 0 && lane == 0 && a.fl_cnt) atomicMax(a.fl_cnt + 13, nu);
                fail(RPD_TRIANGLE_OVERFLOW);
                return;
            }
            wsync();
            ntri = nu;
            add_volume = in_domain == 2;
        } else {
            const int nx = vmx[0] - vmn[0] + 1, ny = vmx[1] - vmn[1] + 1, nz = vmx[2] - vmn[2] + 1;
            const int nvox = nx * ny * nz;
            // First voxel of the box, in scan order (x fastest, then y, z),
            // whose flag is not 1 (the reference corner rule) or whose class is
            // known (apex_mode 1); usually the first voxel already.
            int first_ref = -1, first_c = -1, ref_flag = 1, c_flag = 1;
            for (int vb = 0; vb < nvox && (a.apex_mode == 1 ? first_c < 0 : first_ref < 0); vb += 64) {
                const int v = vb + lane;
                const bool in = v < nvox;
                int f = 1, cf = 1;
                if (in) {
                    const int x = vmn[0] + v % nx, y = vmn[1] + (v / nx) % ny, z = vmn[2] + v / (nx * ny);
                    const int id = x + y * g + z * g * g;
                    f = a.flags[id];
                    cf = a.centre ? a.centre[id] : (a.toffs[id + 1] == a.toffs[id] ? f : 1);
                }
                const uint64_t mr = ballot(in && f != 1);
                if (first_ref < 0 && mr) {
                    const int l = lowest_bit(mr);
                    first_ref = vb + l;
                    ref_flag = rlane(f, l);
                }
                const uint64_t mc = ballot(in && cf != 1);
                if (first_c < 0 && mc) {
                    const int l = lowest_bit(mc);
                    first_c = vb + l;
                    c_flag = rlane(cf, l);
                }
            }
            // Union of the voxels' lists (merge, ConvexCell.cl:722-749).  The
            // list entries of one row of the box are one range of tlist; the
            // rows' ranges are spread over the lanes.  An entry is kept in the
            // first voxel of the box, in scan order, whose list holds its
            // triangle: tinfo holds the entry's voxel and a mask of the voxels
            // within 2 of it per axis that precede it and hold the triangle too
            // (or kTinfoFar when one farther away does: then the triangle's own
            // voxel list is read).  Entries are kept in scan order.
            int nu = 0;
            const uint32_t pmn = (uint32_t(vmn[2]) << 20) | (uint32_t(vmn[1]) << 10) | uint32_t(vmn[0]);
            const uint32_t pmx = (uint32_t(vmx[2]) << 20) | (uint32_t(vmx[1]) << 10) | uint32_t(vmx[0]);
            int *seg_off = reinterpret_cast<int *>(cpl), *seg_a = seg_off + 64;
            const int nrows = ny * nz;
            for (int rb = 0; rb < nrows; rb += 64) {
                const int r = rb + lane;
                int sa = 0, len = 0;
                if (r < nrows) {
                    const int id0 = vmn[0] + (vmn[1] + r % ny) * g + (vmn[2] + r / ny) * g * g;
                    sa = a.toffs[id0];
                    len = a.toffs[id0 + nx] - sa;
                }
                const int off = wave_excl_scan(len);
                const int total = uni(rlane(off + len, 63));
                if (total == 0) continue;
                seg_off[lane] = off;
                seg_a[lane] = sa;
                wsync();
                for (int base = 0; base < total; base += 64) {
                    const int e = base + lane;
                    bool keep = false;
                    int t = -1;
                    if (e < total) {
                        // last row whose offset is <= e (empty rows never win)
                        int lo = 0, hi = 63;
                        while (lo < hi) {
                            const int mid = (lo + hi + 1) >> 1;
                            if (seg_off[mid] <= e)
                                lo = mid;
                            else
                                hi = mid - 1;
                        }
                        const int q = seg_a[lo] + (e - seg_off[lo]);
                        t = a.tlist[q];
                        const uint4 inf = a.tinfo[q];
                        const uint32_t pv = inf.x;
                        const uint64_t near = (uint64_t(inf.z) << 32) | inf.y;
                        if (near & kTinfoFar) {
                            keep = true;
                            for (int u = a.tvoffs[t], ue = a.tvoffs[t + 1]; u < ue; ++u) {
                                const uint32_t w = a.tvox[u];
                                if (w >= pv) break;
                                const uint32_t ux = w & 1023u, uy = (w >> 10) & 1023u, uz = w >> 20;
                                if (ux >= (pmn & 1023u) && ux <= (pmx & 1023u) && uy >= ((pmn >> 10) & 1023u) &&
                                    uy <= ((pmx >> 10) & 1023u) && uz >= (pmn >> 20) && uz <= (pmx >> 20)) {
                                    keep = false;  // an earlier voxel of the box holds it
                                    break;
                                }
                            }
                        } else {
                            const int x = int(pv & 1023u), y = int((pv >> 10) & 1023u), z = int(pv >> 20);
                            keep = (near & box_near(x, y, z, vmn, vmx)) == 0;
                        }
                    }
                    const uint64_t m = ballot(keep);
                    if (keep && nu + mbcnt(m) < a.T) tu[nu + mbcnt(m)] = t;
                    nu += __popcll(m);
                }
                wsync();  // the next rows overwrite seg_off / seg_a
            }
            if (a.count_only) {
                if (lane == 0 && a.status[orig] != RPD_TRIANGLE_OVERFLOW) {
                    atomicMax(a.dcnt + kDcMax + 3, nu);
                    atomicAdd(a.dcnt + kDcHistT + min(nu, kDcUnionMax), 1);
                }
                return;
            }
            if (nu > a.T) {
                // the cap a re-queue pass needs for this cell
                if (sub == 0 && lane == 0 && a.fl_cnt) atomicMax(a.fl_cnt + 13, nu);
                fail(RPD_TRIANGLE_OVERFLOW);
                return;
            }
            if (a.dcnt && sub == 0 && lane == 0) {  // ConvexCell.cl:981-982
                atomicMax(a.dcnt + kDcMax + 3, nu);
                atomicAdd(a.dcnt + kDcHistT + min(nu, kDcUnionMax), 1);
            }
            wsync();
            ntri = nu;
            // apex
            int in_domain = 1;
            auto vox_xyz = [&](int v, int &x, int &y, int &z) {
                x = vmn[0] + v % nx;
                y = vmn[1] + (v / nx) % ny;
                z = vmn[2] + v / (nx * ny);
            };
            if (a.apex_mode == 1 && first_c >= 0) {
                int x, y, z;
                vox_xyz(first_c, x, y, z);
                P0x = (x + kApexFrac[0]) * vs;
                P0y = (y + kApexFrac[1]) * vs;
                P0z = (z + kApexFrac[2]) * vs;
                in_domain = c_flag;
            } else if (first_ref >= 0) {
                int x, y, z;
                vox_xyz(first_ref, x, y, z);
                P0x = x * vs;
                P0y = y * vs;
                P0z = z * vs;
                in_domain = ref_flag;
            } else {
                // GRID_OUT_DOMAIN fallback (ConvexCell.cl:985-1051)
                auto flag = [&](int x, int y, int z) { return int(a.flags[x + y * g + z * g * g]); };
                auto setc = [&](int x, int y, int z) {
                    P0x = x * vs;
                    P0y = y * vs;
                    P0z = z * vs;
                };
                if (vmx[2] + 1 < g) {
                    const int z = vmx[2] + 1;
                    for (int y = vmn[1]; y <= vmx[1] + 1 && y < g && in_domain == 1; y++)
                        for (int x = vmn[0]; x <= vmx[0] + 1 && x < g; x++)
                            if (flag(x, y, z) != 1) {
                                in_domain = flag(x, y, z);
                                setc(x, y, z);
                                break;
                            }
                } else {
                    in_domain = 0;
                    setc(vmn[0], vmn[1], vmx[2] + 1);
                }
                if (in_domain == 1 && vmx[1] + 1 < g) {
                    const int y = vmx[1] + 1;
                    for (int z = vmn[2]; z <= vmx[2] && in_domain == 1; z++)
                        for (int x = vmn[0]; x <= vmx[0] + 1 && x < g; x++)
                            if (flag(x, y, z) != 1) {
                                in_domain = flag(x, y, z);
                                setc(x, y, z);
                                break;
                            }
                } else if (in_domain == 1) {
                    in_domain = 0;
                    setc(vmn[0], vmx[1] + 1, vmn[2]);
                }
                if (in_domain == 1 && vmx[0] + 1 < g) {
                    const int x = vmx[0] + 1;
                    for (int z = vmn[2]; z <= vmx[2] && in_domain == 1; z++)
                        for (int y = vmn[1]; y <= vmx[1]; y++)
                            if (flag(x, y, z) != 1) {
                                in_domain = flag(x, y, z);
                                setc(x, y, z);
                                break;
                            }
                } else if (in_domain == 1) {
                    in_domain = 0;
                    setc(vmx[0] + 1, vmn[1], vmn[2]);
                }
                if (in_domain == 1) {
                    fail(RPD_FIND_ANOTHER_BEGINNING_VERTEX);
                    return;
                }
            }
            add_volume = in_domain == 2;
        }
    }
    double cadd = 0.0;  // the whole cell's term
    if (add_volume && sub == 0) cadd = integrate(1.0);

    // The reference clips the triangles in increasing id order and stops at
    // the first failure: the cell's status is that of the smallest failing
    // id.  Triangles are visited here in list order, so after a failure only
    // triangles of smaller id are still clipped.
    int fail_t = 0x7fffffff, fail_st = 0;
    constexpr int kUB = VOX ? kStripBatch : kTriBatch;  // units of a batch
    const int nbat = (ntri + kUB - 1) / kUB;
    double sum = 0.0;  // running sum of the batches (W = 1)
    if (ntri > 0) {
        // backup (ConvexCell.cl:692-715): the vertex registers, their adjacency
        // and the plane count
        const WaveCell<R, RP, FILTER, S> bk = c;
        uint2 bk_adj[S];
#pragma unroll
        for (int s = 0; s < S; ++s) bk_adj[s] = c.adj[s * 64 + lane];
        auto planes64 = [&]() -> const Pl<double> * {
            if constexpr (sizeof(RP) == 8) return c.planes;
            return nullptr;
        };
        constexpr int kPl = VOX ? 5 : 4;    // cone planes of a unit (strip or triangle)
        constexpr uint64_t kUm = (1ull << kPl) - 1;
        const bool may_skip = c.nb_plane + kPl <= P && nvalid + (VOX ? 8 : 6) <= a.V;
        const double lx0 = P0x - S0.x, ly0 = P0y - S0.y, lz0 = P0z - S0.z;
        const double face_margin = sizeof(RP) == 8 ? 1e-7 : 1e-3;
        // The cell's vertices, compacted, for the lane-parallel tests: a cone
        // plane removes every vertex when each one is strictly on its removed
        // side, with a margin: above the certified FP32 error bound (mixed
        // form) or above 2^-33 (FP64) or 2^-16 (FP32 form) times the sum of
        // the test's |terms|.
        int nvc = 0;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            if (in_mask(c.valid[s]))
                vtx[nvc + mbcnt(c.valid[s])] = VtxRec<R>{c.X[s], c.Y[s], c.Z[s], c.W[s], c.M[s]};
            nvc += __popcll(c.valid[s]);
        }
        wsync();
        // A cone plane (unit normal n, offset d) with d < -rcell keeps no point
        // of the ball |y| <= rcell about the seed, which holds the cell: it
        // removes every vertex (kept side n.y + d >= 0), with a margin far
        // above the rounding of d and rcell.
        const double rsk = rcell * (1.0 + 1e-9) + 1e-9;
        // Batch jb is the units jb, jb + nbat, ...: neighbours in the list, of
        // which either all or none are near the cell, go to different batches,
        // so that the batches and with them the waves that take them (sub, sub
        // + W, ...) have about the same number to clip.  Which units a batch
        // has does not depend on W, and the batches' sums are added in order:
        // the result is the same for every W.
        for (int jb = sub; jb < nbat; jb += W) {
            double bs = 0.0;  // the batch's sum
            // cone planes, lane = kPl * unit + plane
            const int i = VOX ? lane / 5 : lane >> 2, f = VOX ? lane - 5 * i : lane & 3;
            const int k = i < kUB ? jb + nbat * i : ntri;
            Pl<RP> pl{RP(0), RP(0), RP(0), RP(0)};
            uint64_t gom = 0;  // VOX: strips whose region counts positive, at lane 5 * strip
            // VOX: the strip in the local frame, across axis ax at rc, from
            // (ru0, rv0) to (ru1, rv1) along its two other axes
            int ax = 0;
            double rc = 0, ru0 = 0, ru1 = 0, rv0 = 0, rv1 = 0;
            if constexpr (VOX) {
                // Cone of a strip from the apex A: for each side, the plane
                // through A and that side, which is parallel to an axis, so
                // its normal has two components; and the strip's own plane.
                bool go = false;
                if (k < ntri) {
                    const uint2 ent = a.vface[tu[k]];
                    const int p0 = int(ent.x & 1023u), p1 = int((ent.x >> 10) & 1023u), p2 = int((ent.x >> 20) & 1023u);
                    ax = int(ent.x >> 30);
                    const int run = int(ent.y >> 2);
                    // axes (u, v) of the strip: x across: (y, z); y: (x, z); z: (x, y)
                    const int pc = ax == 0 ? p0 : (ax == 1 ? p1 : p2);
                    const int pu = ax == 0 ? p1 : p0, pv = ax == 2 ? p1 : p2;
                    const int pu1 = min(pu + run, (ax == 0 ? vmx[1] : vmx[0]) + 1);
                    const double Sc = ax == 0 ? S0.x : (ax == 1 ? S0.y : S0.z), Su = ax == 0 ? S0.y : S0.x,
                                 Sv = ax == 2 ? S0.y : S0.z;
                    const double Ac = ax == 0 ? lx0 : (ax == 1 ? ly0 : lz0), Au = ax == 0 ? ly0 : lx0,
                                 Av = ax == 2 ? ly0 : lz0;
                    rc = pc * a.vs - Sc;
                    ru0 = pu * a.vs - Su;
                    ru1 = pu1 * a.vs - Su;
                    rv0 = pv * a.vs - Sv;
                    rv1 = (pv + 1) * a.vs - Sv;
                    const double da = rc - Ac;  // not 0: the apex is inside a voxel
                    go = (ent.y & kVfaceUp) ? da > 0.0 : da < 0.0;
                    const double sg = da > 0.0 ? 1.0 : -1.0;
                    double nc, nt = 0, nd;
                    if (f < 4) {
                        // sides v0, v1, u0, u1
                        const double At = f < 2 ? Av : Au;
                        const double dt = (f == 0 ? rv0 : (f == 1 ? rv1 : (f == 2 ? ru0 : ru1))) - At;
                        const double il = ((f & 1) ? -1.0 : 1.0) / sqrt(da * da + dt * dt);
                        nt = fabs(da) * il;
                        nc = -sg * dt * il;
                        nd = -(nt * At + nc * Ac);
                    } else {
                        nc = sg;
                        nd = -sg * rc;
                    }
                    // back to x, y, z
                    const bool tu_ = f >= 2;  // the side's axis t is u (else v)
                    const double nu_ = tu_ ? nt : 0.0, nv_ = tu_ ? 0.0 : nt;
                    pl = Pl<RP>{RP(ax == 0 ? nc : nu_), RP(ax == 0 ? nu_ : (ax == 1 ? nc : nv_)),
                                RP(ax == 2 ? nc : nv_), RP(nd)};
                }
                gom = ballot(go);
            }
            // general domain: planes (A,B,C), (A,D,B), (A,C,D), (C,D,B), A =
            // apex (CCClipTetFromPointsInfinite)
            if (!VOX && k < ntri) {
                const int tid = tu[k];
                const double4 G1 = a.gpts[a.tris[3 * tid]];
                double4 G2 = a.gpts[a.tris[3 * tid + 1]], G3 = a.gpts[a.tris[3 * tid + 2]];
                // orientation test in the global frame, as the reference
                const double ux = G1.x - P0x, uy = G1.y - P0y, uz = G1.z - P0z;
                const double vx = G2.x - P0x, vy = G2.y - P0y, vz = G2.z - P0z;
                const double wx = G3.x - P0x, wy = G3.y - P0y, wz = G3.z - P0z;
                const double det = ux * (vy * wz - vz * wy) - vx * (uy * wz - uz * wy) + wx * (uy * vz - uz * vy);
                const bool go_out = det > 0.0;
                if (!go_out) {
                    const double4 tmp = G2;
                    G2 = G3;
                    G3 = tmp;
                }
                if (f == 0) goo[i] = go_out ? 1 : 0;
                // the three points of plane f in the local frame
                const double Bx = G1.x - S0.x, By = G1.y - S0.y, Bz = G1.z - S0.z;
                const double Cx = G2.x - S0.x, Cy = G2.y - S0.y, Cz = G2.z - S0.z;
                const double Dx = G3.x - S0.x, Dy = G3.y - S0.y, Dz = G3.z - S0.z;
                if (f < 3) {  // the corners in the local frame, for the face test
                    const double cx = f == 0 ? Bx : (f == 1 ? Cx : Dx);
                    const double cy = f == 0 ? By : (f == 1 ? Cy : Dy);
                    const double cz = f == 0 ? Bz : (f == 1 ? Cz : Dz);
                    tcor[9 * i + 3 * f] = cx;
                    tcor[9 * i + 3 * f + 1] = cy;
                    tcor[9 * i + 3 * f + 2] = cz;
                }
                double px, py, pz, qx, qy, qz, rx, ry, rz;
                if (f == 3) {
                    px = Cx, py = Cy, pz = Cz;
                    qx = Dx, qy = Dy, qz = Dz;
                    rx = Bx, ry = By, rz = Bz;
                } else {
                    px = lx0, py = ly0, pz = lz0;
                    if (f == 0) {
                        qx = Bx, qy = By, qz = Bz;
                        rx = Cx, ry = Cy, rz = Cz;
                    } else if (f == 1) {
                        qx = Dx, qy = Dy, qz = Dz;
                        rx = Bx, ry = By, rz = Bz;
                    } else {
                        qx = Cx, qy = Cy, qz = Cz;
                        rx = Dx, ry = Dy, rz = Dz;
                    }
                }
                const double e1x = qx - px, e1y = qy - py, e1z = qz - pz;
                const double e2x = rx - px, e2y = ry - py, e2z = rz - pz;
                double nx_ = e1y * e2z - e1z * e2y, ny_ = e1z * e2x - e1x * e2z, nz_ = e1x * e2y - e1y * e2x;
                double nd = -(nx_ * px + ny_ * py + nz_ * pz);
                const double nl = sqrt(nx_ * nx_ + ny_ * ny_ + nz_ * nz_);
                if (nl > 0) {
                    const double il = 1.0 / nl;
                    nx_ *= il;
                    ny_ *= il;
                    nz_ *= il;
                    nd *= il;
                }
                pl = Pl<RP>{RP(nx_), RP(ny_), RP(nz_), RP(nd)};
            }
            cpl[lane] = pl;
            // Skip tests, one lane per cone plane: the ball about the seed,
            // then every vertex.
            bool gone = false;
            if (may_skip && k < ntri) {
                gone = double(pl.w) < -rsk;
                if (!gone) {
                    const Pl<R> e = cvt<R>(pl);
                    const float ek = kFilterKappa * (fabsf(float(e.x)) + fabsf(float(e.y)) + fabsf(float(e.z))),
                                ewk = kFilterKappa * kMagW * fabsf(float(e.w));
                    gone = true;
                    // U vertices a step, their loads issued together (the
                    // last vertex stands in past the end: testing it twice
                    // changes nothing)
                    constexpr int U = sizeof(R) == 4 ? 4 : 2;
                    for (int j0 = 0; j0 < nvc && gone; j0 += U) {
                        VtxRec<R> v[U];
#pragma unroll
                        for (int u = 0; u < U; ++u) v[u] = vtx[min(j0 + u, nvc - 1)];
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                            const R sv = e.x * v[u].X + e.y * v[u].Y + e.z * v[u].Z + e.w * v[u].W;
                            R m;
                            if (FILTER)
                                m = R(fmaf(ek, v[u].M, ewk));
                            else
                                m = R(sizeof(R) == 8 ? 0x1.0p-33 : 0x1.0p-16) *
                                    (fabs(e.x * v[u].X) + fabs(e.y * v[u].Y) + fabs(e.z * v[u].Z) +
                                     fabs(e.w * v[u].W));
                            gone = gone && sv > m;
                        }
                    }
                }
            }
            uint64_t skipm = ballot(gone);
            wsync();
            // The cone region of a triangle (apex A, beyond the triangle) lies
            // strictly outside one of the cell's planes when the triangle's
            // three corners do (with a margin) and the rays from A through
            // them do not turn back towards the plane.  The cell is inside
            // every plane of its list (each one cut it when added), so the two
            // are disjoint: the reference's clip ends empty_cell (same caps
            // guard as above).  Lane 4i + f tests planes f, f + 4, ... against
            // triangle i.
            {
                bool sep = false;
                if constexpr (VOX) {
                    if (may_skip && k < ntri && ((skipm >> (kPl * i)) & kUm) == 0) {
                        // the strip's corner farthest along the plane's normal
                        // decides for all four
                        for (int j = f; j < c.nb_plane && !sep; j += 10) {
                            Pl<RP> q2[2];
#pragma unroll
                            for (int u = 0; u < 2; ++u) q2[u] = c.planes[min(j + 5 * u, c.nb_plane - 1)];
#pragma unroll
                            for (int u = 0; u < 2; ++u) {
                                const double nx = double(q2[u].x), ny = double(q2[u].y), nz = double(q2[u].z),
                                             nw = double(q2[u].w);
                                const double nc = ax == 0 ? nx : (ax == 1 ? ny : nz), nu_ = ax == 0 ? ny : nx,
                                             nv_ = ax == 2 ? ny : nz;
                                const double far = nc * rc + fmax(nu_ * ru0, nu_ * ru1) + fmax(nv_ * rv0, nv_ * rv1);
                                const double m = face_margin * (1.0 + fabs(nw));
                                sep = sep || (far + nw < -m && far - (nx * lx0 + ny * ly0 + nz * lz0) <= 0.0);
                            }
                        }
                    }
                }
                if (!VOX && may_skip && k < ntri && ((skipm >> (4 * i)) & 0xfull) == 0) {
                    double px[3], py[3], pz[3];
#pragma unroll
                    for (int v = 0; v < 3; ++v) {
                        px[v] = tcor[9 * i + 3 * v];
                        py[v] = tcor[9 * i + 3 * v + 1];
                        pz[v] = tcor[9 * i + 3 * v + 2];
                    }
                    // two planes a step, loaded together; past the end the
                    // last plane stands in (any plane of the cell may
                    // separate, and the triangle's other lanes test it too)
                    for (int j = f; j < c.nb_plane && !sep; j += 8) {
                        Pl<RP> q2[2];
#pragma unroll
                        for (int u = 0; u < 2; ++u) q2[u] = c.planes[min(j + 4 * u, c.nb_plane - 1)];
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            const double nx = double(q2[u].x), ny = double(q2[u].y), nz = double(q2[u].z),
                                         nw = double(q2[u].w);
                            const double m = face_margin * (1.0 + fabs(nw));
                            bool out = true;
#pragma unroll
                            for (int v = 0; v < 3; ++v) {
                                out = out && nx * px[v] + ny * py[v] + nz * pz[v] + nw < -m;
                                out = out && nx * (px[v] - lx0) + ny * (py[v] - ly0) + nz * (pz[v] - lz0) <= 0.0;
                            }
                            sep = sep || out;
                        }
                    }
                }
                skipm |= ballot(sep);
            }
            // triangles of the batch that are clipped: none of their four
            // lanes skipped them
            uint32_t todo = 0;
#pragma unroll
            for (int t = 0; t < kUB; ++t)
                if (jb + nbat * t < ntri && ((skipm >> (kPl * t)) & kUm) == 0) todo |= 1u << t;
            // in increasing order (a skipped unit adds nothing)
            while (todo) {
                const int t = __builtin_ctz(todo);
                todo &= todo - 1;
                const int kk = jb + nbat * t;
                // (a strip stands for several triangles: its place in the list)
                const int tid = VOX ? kk : uni(tu[kk]);
                if (tid > fail_t) continue;
                int res = kNoClip;
                // each cone plane read from LDS just before its clip: the four
                // held at once would take 32 registers through the clips
#pragma unroll
                for (int f2 = 0; f2 < kPl; ++f2) {
                    if (res < 0) {
                        const Pl<RP> q = cpl[kPl * t + f2];
                        if (c.nb_plane >= P) {
                            res = RPD_PLANE_OVERFLOW;
                        } else {
                            if (lane == 0) c.planes[c.nb_plane] = q;
                            res = c.template clip<false>(cvt<R>(q), planes64);
                        }
                    }
                }
                if (res >= 0 && res != RPD_EMPTY_CELL) {
                    fail_t = tid;
                    fail_st = res;
                } else if (res != RPD_EMPTY_CELL) {
                    bs += integrate((VOX ? ((gom >> (kPl * t)) & 1) != 0 : goo[t] != 0) ? 1.0 : -1.0);
                }
                c = bk;
#pragma unroll
                for (int s = 0; s < S; ++s) c.adj[s * 64 + lane] = bk_adj[s];
                wsync();
            }
            if (W == 1)
                sum += bs;
            else if ((lane & 15) == 0)
                bsum[4 * jb + (lane >> 4)] = bs;
            wsync();  // the next batch overwrites cpl / goo
        }
    }
    if (lane == 0) {
        fails[2 * sub] = fail_t;
        fails[2 * sub + 1] = fail_st;
    }
    if (W > 1)
        __syncthreads();
    else
        wsync();
    if (sub != 0) return;
    // smallest failing triangle id over the waves
    int fk = 0x7fffffff, fs = 0;
    for (int w = 0; w < W; ++w) {
        const int k = fails[2 * w];
        if (k < fk) {
            fk = k;
            fs = fails[2 * w + 1];
        }
    }
    if (fk != 0x7fffffff) {
        fail(fs);
        return;
    }
    // fixed summation order: the batches in order, then the whole-cell term
    if (W > 1)
        for (int k = 0; k < nbat; ++k) sum += bsum[4 * k + (lane >> 4)];
    sum += cadd;
    const double acc_x = rlane(sum, 0), acc_y = rlane(sum, 16), acc_z = rlane(sum, 32), acc_m = rlane(sum, 48);
    // Hessian entries (ConvexCell.cl:1133-1151): the record's planes towards
    // a seed whose face keeps more than 0.2 of area, in plane order, with the
    // neighbours' original indices; more than H: hessian_overflow, the first
    // H written
    int st_out = RPD_SUCCESS;
    if (HESS) {
        const int *rnid = reinterpret_cast<const int *>(rtr + 128 * a.rec_S);
        const int H = a.H;
        int cnt = 0;
        for (int pb = 0; pb < nbk; pb += 64) {
            const int p = pb + lane;
            int nb = -1;
            bool keep = false;
            if (p < nbk) {
                nb = rnid[p];
                keep = nb >= 0 && hacc[4 * p + 3] > 0.2;
            }
            const uint64_t m = ballot(keep);
            const int pos = cnt + mbcnt(m);
            if (keep && pos < H) {
                const size_t e = size_t(orig) * size_t(H) + size_t(pos);
                const double ar = hacc[4 * p + 3];
                a.hids[e] = a.perm[nb];
                if (a.hc == 1) {
                    a.hess[e] = ar;
                } else {
                    a.hess[4 * e + 0] = hacc[4 * p + 0] + ar * S0.x;
                    a.hess[4 * e + 1] = hacc[4 * p + 1] + ar * S0.y;
                    a.hess[4 * e + 2] = hacc[4 * p + 2] + ar * S0.z;
                    a.hess[4 * e + 3] = ar;
                }
            }
            cnt += __popcll(m);
        }
        if (cnt > H)
            st_out = RPD_HESSIAN_OVERFLOW;
        else if (cnt < H && lane == 0)
            a.hids[size_t(orig) * size_t(H) + size_t(cnt)] = -1;
        if (a.dcnt && lane == 0) atomicMax(a.dcnt + kDcMax + 4, min(cnt, H));  // ConvexCell.cl:1150
    }
    // local first moments -> global frame
    finish(st_out, acc_x + acc_m * S0.x, acc_y + acc_m * S0.y, acc_z + acc_m * S0.z, acc_m);
}

}  // namespace rpd

using namespace rpd;

// Bytes of one stored plane: the planes of the FP64 and mixed forms are FP64.
static size_t plane_bytes(int form) { return form == RPD_PREC_FP32 ? 16 : 32; }

// LDS of a gfx950 CU, shared by the resident workgroups
constexpr size_t kLdsPerCu = 160 * 1024;

// LDS a workgroup may use on the current device (asked once per device)
static size_t lds_limit() {
    static std::atomic<int> cached[64];
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 64 * 1024;
    if (dev >= 0 && dev < 64 && (v = cached[dev].load(std::memory_order_relaxed)) > 0) return size_t(v);
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || v <= 0)
        return 64 * 1024;
    if (dev >= 0 && dev < 64) cached[dev].store(v, std::memory_order_relaxed);
    return size_t(v);
}

// LDS of the cell part of a finish-kernel workgroup: fail slots, the units it
// meets (T) and, when W > 1 waves share the cell, the sums of its batches.
static size_t finish_cell_stride(int T, int W) {
    return 64 + up16(4 * size_t(T)) + (W > 1 ? 32 * ((size_t(T) + kStripBatch - 1) / kStripBatch) : 0);
}

// LDS of one finish-kernel cell handled by a single wave.
static size_t finish_cell_lds(int form, int P, int V, int T, bool hess) {
    const int S = V <= 64 ? 1 : (V <= 128 ? 2 : 4);
    return finish_cell_stride(T, 1) + finish_wave_lds(P, S, plane_bytes(form), true) +
           (hess ? hessian_wave_lds(P, S) : 0);
}

int rpd_clip_max_T(int form, int P, int V, bool hess) {
    const size_t lim = lds_limit();
    int lo = 0, hi = 1 << 20;
    if (finish_cell_lds(form, P, V, 0, hess) > lim) return -1;
    while (lo < hi) {
        const int mid = lo + (hi - lo + 1) / 2;
        if (finish_cell_lds(form, P, V, mid, hess) <= lim)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

int rpd_clip_plane_room(int form, int P, int V, int T, int floor) {
    const int S = V <= 64 ? 1 : (V <= 128 ? 2 : 4);
    if (S != 1) return P;
    // cells per CU at the kernels' residency: 4 waves per SIMD for the
    // finish kernel, kClipWaves for the bisector kernel (one cell a wave)
    const size_t fin_cells = 4 * 4;
    const size_t bis_cells = 4 * size_t(form == RPD_PREC_FP64 ? kClipWaves<double, 1> : kClipWaves<float, 1>);
    for (int p = std::min(floor, 255); p > P; --p)
        if (finish_cell_lds(form, p, V, T, false) * fin_cells <= kLdsPerCu &&
            cells_wave_lds(form, p, S) * bis_cells <= kLdsPerCu)
            return p;
    return P;
}

// header | P planes | 64 S vertex triples, 64 S adjacency words | P plane neighbours (int)
size_t rpd_clip_record_bytes(int form, int P, int V) {
    const int S = V <= 64 ? 1 : (V <= 128 ? 2 : 4);
    const size_t pl = plane_bytes(form);
    return (sizeof(RecHeader) + size_t(P) * pl + 8 * 64 * size_t(S) + 4 * size_t(P) + 15) & ~size_t(15);
}

static int make_args(int form, const ClipLaunch &L, ClipArgs &a) {
    if (L.P < 7 || L.P > 255 || L.V < 8 || L.K < 1) return RPD_E_ARG;
    if (L.V > 256) return RPD_E_LIMIT;
    if (!L.rec) return RPD_E_ARG;
    if (L.reqs && (!L.req_of || (L.hess && L.H > 0))) return RPD_E_ARG;
    a = ClipArgs{};
    a.seeds = L.seeds;
    a.perm = L.perm;
    a.ids = L.ids;
    a.knn = L.knn;
    a.n_ids = L.n_ids;
    a.n_seeds = L.n_seeds;
    a.K = L.K;
    a.P = L.P;
    a.V = L.V;
    a.T = std::max(L.T, 0);
    a.apex_mode = L.apex_mode;
    if (L.dom) {
        a.g = L.dom->g;
        a.vs = L.dom->vs;
        a.flags = L.dom->flags;
        a.centre = L.dom->centre;
        a.gpts = L.dom->pts;
        a.tris = L.dom->tris;
        a.tlist = L.dom->tlist;
        a.toffs = L.dom->toffs;
        a.tvoffs = L.dom->tvoffs;
        a.tvox = L.dom->tvox;
        a.tinfo = L.dom->tinfo;
        a.vfoffs = L.dom->vfoffs;
        a.vface = L.dom->vface;
        a.dist = L.cull ? L.dom->dist : nullptr;
    }
    a.security_mode = L.security_mode;
    a.wmin = L.wmin;
    a.out = L.out;
    a.status = L.status;
    a.kused = L.kused;
    a.rec = static_cast<char *>(L.rec);
    const int rec_P = L.rec_P > 0 ? L.rec_P : L.P, rec_V = L.rec_V > 0 ? L.rec_V : L.V;
    if (rec_P > L.P || rec_V > L.V) return RPD_E_ARG;
    a.rec_stride = int(rpd_clip_record_bytes(form, rec_P, rec_V));
    a.rec_P = rec_P;
    a.rec_S = rec_V <= 64 ? 1 : (rec_V <= 128 ? 2 : 4);
    a.code = L.code;
    a.fl_cnt = L.fl_cnt;
    a.fl_eo = L.fl_eo;
    a.rs_out = L.rs_out;
    a.rs_out_stride = L.rs_out_stride;
    a.rs_base = L.rs_base;
    a.rs_in = form != RPD_PREC_FP32 ? L.rs_in : nullptr;
    a.rs_in_stride = L.rs_in_stride;
    a.rs_in_P = L.rs_in_P;
    a.rslot = L.rslot;
    a.lastnb = L.lastnb;
    a.hess = L.hess;
    a.hids = L.hids;
    a.H = L.hess && L.hids ? L.H : 0;
    a.hc = L.hc == 4 ? 4 : 1;
    a.exact_final = form == RPD_PREC_FP64 ? 1 : 0;
    a.dcnt = L.dcnt;
    a.reqs = L.reqs;
    a.req_of = L.req_of;
    a.slots = L.slots;
    a.fl_slot = L.fl_slot;
    a.keep_exact = L.keep_exact ? 1 : 0;
    return RPD_OK;
}

int rpd_launch_cells(hipStream_t st, int form, const ClipLaunch &L) {
    if (L.n_ids <= 0) return RPD_OK;
    if (!L.code) return RPD_E_ARG;
    ClipArgs a;
    const int r = make_args(form, L, a);
    if (r != RPD_OK) return r;
    const int S = L.V <= 64 ? 1 : (L.V <= 128 ? 2 : 4);
    // kernel A: the bisector loop of every cell
    {
        const size_t stride = cells_wave_lds(form, L.P, S);
        a.lds_stride = int(stride);
        // one wave per workgroup: each cell's wave starts and ends on its own
        const unsigned blocks = unsigned(L.n_ids);
        const dim3 tb(64);
        const size_t shm = stride;
#define RPD_CLIP_A1(R, RP, F, B)                                                      \
    do {                                                                              \
        if (S == 1)                                                                   \
            clip_cells_kernel<R, RP, F, 1, B><<<blocks, tb, shm, st>>>(a);            \
        else if (S == 2)                                                              \
            clip_cells_kernel<R, RP, F, 2, B><<<blocks, tb, shm, st>>>(a);            \
        else                                                                          \
            clip_cells_kernel<R, RP, F, 4, B><<<blocks, tb, shm, st>>>(a);            \
    } while (0)
#define RPD_CLIP_A(R, RP, F)              \
    do {                                  \
        if (a.reqs)                       \
            RPD_CLIP_A1(R, RP, F, true);  \
        else                              \
            RPD_CLIP_A1(R, RP, F, false); \
    } while (0)
        if (form == RPD_PREC_FP64)
            RPD_CLIP_A(double, double, false);
        else if (form == RPD_PREC_MIXED)
            RPD_CLIP_A(float, double, true);
        else
            RPD_CLIP_A(float, float, false);
#undef RPD_CLIP_A
#undef RPD_CLIP_A1
        if (hipGetLastError() != hipSuccess) return RPD_E_DEVICE;
    }
    if (L.ev_mid && hipEventRecord(L.ev_mid, st) != hipSuccess) return RPD_E_DEVICE;
    return RPD_OK;
}

int rpd_launch_lists(hipStream_t st, const ClipLaunch &L, const FailLists &F) {
    if (L.n_ids <= 0) return RPD_OK;
    ListArgs a{};
    a.code = L.code;
    a.ids = L.ids;
    a.n = L.n_ids;
    a.cnt = F.cnt;
    a.eo = F.eo;
    a.sec = F.sec;
    a.q = F.q;
    a.q_host = F.q_host_dev;
    a.cnt_host = F.cnt_host_dev;
    const int64_t per = int64_t(kListBlock) * kListPer;
    list_failures_kernel<<<unsigned((L.n_ids + per - 1) / per), kListBlock, 0, st>>>(a);
    return hipGetLastError() == hipSuccess ? RPD_OK : RPD_E_DEVICE;
}

namespace rpd {
__global__ __launch_bounds__(64) void pin_copy_kernel(const int *src0, int *dst0, int n0, const int *src1,
                                                      int *dst1, int n1) {
    for (int i = int(threadIdx.x); i < n0; i += 64) dst0[i] = src0[i];
    for (int i = int(threadIdx.x); i < n1; i += 64) dst1[i] = src1[i];
    __threadfence_system();  // the host reads them once the stream is done
}
}  // namespace rpd

namespace rpd {
__global__ __launch_bounds__(64) void zero_ints_kernel(int *p, int n) {
    for (int i = int(threadIdx.x); i < n; i += 64) p[i] = 0;
}
}  // namespace rpd

int rpd_zero_ints(hipStream_t st, int *p, int n) {
    zero_ints_kernel<<<1, 64, 0, st>>>(p, n);
    return hipGetLastError() == hipSuccess ? RPD_OK : RPD_E_DEVICE;
}

int rpd_pin_copy(hipStream_t st, const int *src0, int *dst0, int n0, const int *src1, int *dst1, int n1) {
    pin_copy_kernel<<<1, 64, 0, st>>>(src0, dst0, n0, src1, dst1, n1);
    return hipGetLastError() == hipSuccess ? RPD_OK : RPD_E_DEVICE;
}

int rpd_launch_finish(hipStream_t st, int form, const ClipLaunch &L, int nq, int beside) {
    if (nq <= 0) return RPD_OK;
    ClipArgs a;
    const int r = make_args(form, L, a);
    if (r != RPD_OK) return r;
    const int S = L.V <= 64 ? 1 : (L.V <= 128 ? 2 : 4);
    // kernel B: restriction + integration of the queued cells.  Short queues
    // (re-queue passes) spread each cell over W waves.
    const size_t pl = plane_bytes(form);
    const bool hess = a.H > 0;
    // Domains of voxel faces restrict by strips (L.vox); the FP32 form takes
    // the triangle lists.  A batch with both kinds takes two launches: in one,
    // by triangle lists, its voxel requests' bits and speed would depend on
    // what they are packed with.
    // The debug counters count triangles: with strips, a launch of the
    // triangle form for the union's counters alone follows.
    const bool vox = L.vox && form != RPD_PREC_FP32;
    // waves per cell from the cells that share the device: this queue's and
    // those of finish kernels running beside it (the Hessian variant: one wave
    // per cell).  Every wave of a cell sets the cell up anew, so one wave is
    // best as soon as the queue fills the chip (4,096 waves at 4 a SIMD;
    // 20,676 blue-noise cells at two waves 0.28, at one 0.21 ms); 8 up to half
    // of that (947 cells that meet hundreds of strips, those above 256 in
    // further passes: 8 waves 0.91, 2 waves 0.98 ms for the solve).
    // With triangle lists the heaviest cells cost several times as much, and
    // they set the launch's time for longer: more waves up to eight times the
    // queue (uniform seeds, the solve: 30,000 in a torus mesh at 100^3 590 ->
    // 525 us, FP64 695 -> 592; FP32, 30,000 in a voxel torus 1,185 -> 925;
    // 20,000 blue-noise seeds in a sphere mesh, whose cells are all alike, 404
    // -> 426).
    const int64_t load = int64_t(nq) + std::max(beside, 0);
    auto launch = [&](bool vx, bool hs) -> int {
        const size_t wstride =
            (vx ? finish_vox_wave_lds(L.P, S, form == RPD_PREC_FP64 ? sizeof(VtxRec<double>) : sizeof(VtxRec<float>))
                : finish_wave_lds(L.P, S, pl, true)) +
            (hs ? hessian_wave_lds(L.P + (vx ? 1 : 0), S) : 0);
        const size_t kLdsMax = lds_limit();
        if (finish_cell_stride(a.T, 1) + wstride > kLdsMax) return RPD_E_LIMIT;
        int W = 1;
        if (!hs && !a.count_only)
            W = load <= 2048 ? 8 : (vx ? (load <= 4096 ? 2 : 1) : (load <= 8192 ? 4 : (load <= 32768 ? 2 : 1)));
        while (W > 1 && finish_cell_stride(a.T, W) + W * wstride > kLdsMax) W >>= 1;
        a.lds_stride = int(wstride);
        a.cell_stride = int(finish_cell_stride(a.T, W));
        // One cell per workgroup: a workgroup keeps its LDS until its last
        // wave ends, and cell costs are skewed (interior cells are cheap), so
        // several cells per workgroup would hold the LDS of finished cells for
        // the slowest one.  LDS bounds the residency of this kernel.
        const dim3 tb(64 * W);
        const size_t shm = size_t(a.cell_stride) + size_t(W) * wstride;
#define RPD_CLIP_B2(R, RP, F, HS, B, X)                                                    \
    do {                                                                                   \
        if (S == 1)                                                                        \
            finish_cells_kernel<R, RP, F, 1, HS, B, X><<<unsigned(nq), tb, shm, st>>>(a, nq, W); \
        else if (S == 2)                                                                   \
            finish_cells_kernel<R, RP, F, 2, HS, B, X><<<unsigned(nq), tb, shm, st>>>(a, nq, W); \
        else                                                                               \
            finish_cells_kernel<R, RP, F, 4, HS, B, X><<<unsigned(nq), tb, shm, st>>>(a, nq, W); \
    } while (0)
// (the FP32 form has no strips)
#define RPD_CLIP_B1(R, RP, F, HS, B)                       \
    do {                                                   \
        if (sizeof(RP) == 8 && vx)                         \
            RPD_CLIP_B2(R, RP, F, HS, B, sizeof(RP) == 8); \
        else                                               \
            RPD_CLIP_B2(R, RP, F, HS, B, false);           \
    } while (0)
// a packed batch has no Hessian
#define RPD_CLIP_B(R, RP, F)                    \
    do {                                        \
        if (hs)                                 \
            RPD_CLIP_B1(R, RP, F, true, false); \
        else if (a.reqs)                        \
            RPD_CLIP_B1(R, RP, F, false, true); \
        else                                    \
            RPD_CLIP_B1(R, RP, F, false, false); \
    } while (0)
        if (form == RPD_PREC_FP64)
            RPD_CLIP_B(double, double, false);
        else if (form == RPD_PREC_MIXED)
            RPD_CLIP_B(float, double, true);
        else
            RPD_CLIP_B(float, float, false);
#undef RPD_CLIP_B
#undef RPD_CLIP_B1
#undef RPD_CLIP_B2
        return RPD_OK;
    };
    const bool both = vox && L.lists;
    a.only = both ? 1 : 0;
    int rl = launch(vox, hess);
    if (rl == RPD_OK && both) {
        a.only = 2;
        rl = launch(false, hess);
    }
    if (rl == RPD_OK && vox && a.dcnt) {
        a.only = both ? 1 : 0;
        a.count_only = 1;
        a.T = 0;
        rl = launch(false, false);
    }
    if (rl != RPD_OK) return rl;
    return hipGetLastError() == hipSuccess ? RPD_OK : RPD_E_DEVICE;
}
