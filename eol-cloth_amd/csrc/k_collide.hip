// Proximity queries on the GPU (gfx950, FP64): btc::pointTriCollision
// (boxTriCollision.cpp:1067-1224) and btc::boxTriCollision (602-1063).
//
// Compiled with -ffp-contract=off: every expression is evaluated in the order the
// reference (through Eigen's 3-vector kernels) evaluates it -- dot products
// (a0 b0 + a1 b1) + a2 b2, cross products component-wise, normalized() as
// v / sqrt(squaredNorm) when squaredNorm > 0 -- so the records are bitwise equal
// to a CPU evaluation of the same algorithm.  The only transcendental, acos, is
// used in threshold comparisons (E2-E1 test); whenever a compared angle lies
// within kAcosBand of its threshold the pair is flagged and the host decides it
// with the C library's acos, so the pair set does not depend on the device acos.
//
// Work decomposition:
//   k_cd_prep       jittered positions and jittered face normals
//   k_cd_aabb       cloth AABB (min/max are exact: order-free)
//   k_grid_*        uniform-grid hash of the cloth faces: each face is entered in
//                   every cell its AABB, grown by a margin that bounds
//                   |x - projection| and the barycentric rounding, overlaps; faces
//                   too ill-shaped for that bound go to an always-tested list.  A
//                   query point tests the faces of its own cell, so it sees every
//                   face the brute-force loop would accept, and the lexicographic
//                   minimum (dist, face index) reproduces the reference's
//                   "strictly closer wins, first wins ties".
//   k_cd_query      one workgroup per query (point obstacle or box corner), on the grid
//   k_cd_sweep      one thread per face against every query, and k_cd_nearest, the
//                   nearest of a query's candidates: what up to kCdSweepQueries queries
//                   take instead of the grid, which is built anew for every call
//   k_cd_boxes      one thread per cloth vertex (V2-T1) and per cloth edge (which boxes'
//                   faces it reaches), for up to kCdBoxes boxes in one launch
//   k_cd_pairs      E2-E1 of the edges and boxes left, 12 lanes each
//   k_cd_eolpts     one thread per cloth vertex (pointTri EOL branch)
// Variable-length outputs come in the reference's order by count -> scan -> write
// passes (no atomics on record positions); the write pass forms a record anew
// instead of keeping room for one per vertex.
#include <algorithm>
#include <mutex>

#include "eolc_internal.h"
#include "collide_common.h"

using namespace eolc_cd;

namespace {

constexpr double kAcosBand = 1e-12;

__device__ __forceinline__ void ld(const double *p, double *o) { o[0] = p[0]; o[1] = p[1]; o[2] = p[2]; }

// ---------------------------------------------------------------------------
__global__ void k_cd_prep(int N, int F, double thr, const double *__restrict__ x, const double *__restrict__ unit,
                          const int *__restrict__ tri, double *__restrict__ xj, double *__restrict__ fn)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < 3 * N) xj[t] = x[t] + unit[t] * thr * 1e-3;
    (void)F; (void)tri; (void)fn;
}

__global__ void k_cd_fnormals(int F, const double *__restrict__ xj, const int *__restrict__ tri,
                              double *__restrict__ fn)
{
    int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= F) return;
    face_normal(xj + 3 * tri[3 * f], xj + 3 * tri[3 * f + 1], xj + 3 * tri[3 * f + 2], fn + 3 * f);
}

// cloth AABB of the jittered positions: per-block min/max, then a one-block pass
__global__ void __launch_bounds__(256) k_cd_aabb(int N, const double *__restrict__ xj, double *__restrict__ part)
{
    __shared__ double s[6][256];
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x)
        for (int k = 0; k < 3; ++k) {
            double v = xj[3 * i + k];
            lo[k] = fmin(lo[k], v);
            hi[k] = fmax(hi[k], v);
        }
    for (int k = 0; k < 3; ++k) { s[k][threadIdx.x] = lo[k]; s[3 + k][threadIdx.x] = hi[k]; }
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o)
            for (int k = 0; k < 3; ++k) {
                s[k][threadIdx.x] = fmin(s[k][threadIdx.x], s[k][threadIdx.x + o]);
                s[3 + k][threadIdx.x] = fmax(s[3 + k][threadIdx.x], s[3 + k][threadIdx.x + o]);
            }
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int k = 0; k < 6; ++k) part[6 * blockIdx.x + k] = s[k][0];
}

// One workgroup of kAabbParts threads, one partial box each (min and max are order-free).
// A single thread walking the 256 partials took 51-57 us, as long as the query itself.
constexpr int kAabbParts = 256;
__global__ void __launch_bounds__(kAabbParts) k_cd_aabb_final(const double *__restrict__ part, double *__restrict__ out)
{
    __shared__ double s[6][kAabbParts];
    const int t = threadIdx.x;
    for (int k = 0; k < 6; ++k) s[k][t] = part[6 * t + k];
    __syncthreads();
    for (int o = kAabbParts / 2; o > 0; o >>= 1) {
        if (t < o)
            for (int k = 0; k < 3; ++k) {
                s[k][t] = fmin(s[k][t], s[k][t + o]);
                s[3 + k][t] = fmax(s[3 + k][t], s[3 + k][t + o]);
            }
        __syncthreads();
    }
    if (t < 6) out[t] = s[t][0];
}

// ---------------------------------------------------------------------------
// uniform-grid hash
struct GridParams {
    double org[3];
    double inv_cell;
    int dim[3];
    unsigned mask;      // table size - 1 (power of two)
    double margin;
    double cond_max;    // faces with |v0|^2 |v1|^2 / denom above this are always tested
};

__device__ __forceinline__ unsigned cell_hash(int ix, int iy, int iz, unsigned mask)
{
    unsigned h = (unsigned)ix * 73856093u ^ (unsigned)iy * 19349663u ^ (unsigned)iz * 83492791u;
    return h & mask;
}

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

__device__ __forceinline__ void face_cells(const GridParams &g, const double *a, const double *b, const double *c,
                                           int lo[3], int hi[3])
{
    for (int k = 0; k < 3; ++k) {
        double mn = fmin(a[k], fmin(b[k], c[k])) - g.margin;
        double mx = fmax(a[k], fmax(b[k], c[k])) + g.margin;
        lo[k] = clampi((int)floor((mn - g.org[k]) * g.inv_cell), 0, g.dim[k] - 1);
        hi[k] = clampi((int)floor((mx - g.org[k]) * g.inv_cell), 0, g.dim[k] - 1);
    }
}

__device__ __forceinline__ bool ill_shaped(const GridParams &g, const double *a, const double *b, const double *c)
{
    double v0[3], v1[3];
    v_sub(b, a, v0);
    v_sub(c, a, v1);
    double d00 = v_dot(v0, v0), d01 = v_dot(v0, v1), d11 = v_dot(v1, v1);
    double denom = d00 * d11 - d01 * d01;
    return !(denom > 0.0) || d00 * d11 > g.cond_max * denom;
}

// pass 0: count per bucket (and the always-tested list), pass 1: fill
__global__ void k_grid_insert(int F, int pass, GridParams g, const double *__restrict__ xj, const int *__restrict__ tri,
                              unsigned *__restrict__ bucket_cnt, const unsigned *__restrict__ bucket_start,
                              unsigned *__restrict__ cursor, int *__restrict__ entries, unsigned *__restrict__ nalways,
                              int *__restrict__ always)
{
    int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= F) return;
    const double *a = xj + 3 * tri[3 * f], *b = xj + 3 * tri[3 * f + 1], *c = xj + 3 * tri[3 * f + 2];
    if (ill_shaped(g, a, b, c)) {
        if (pass == 1) {
            unsigned p = atomicAdd(nalways, 1u);
            always[p] = f;
        }
        return;
    }
    int lo[3], hi[3];
    face_cells(g, a, b, c, lo, hi);
    for (int iz = lo[2]; iz <= hi[2]; ++iz)
        for (int iy = lo[1]; iy <= hi[1]; ++iy)
            for (int ix = lo[0]; ix <= hi[0]; ++ix) {
                unsigned h = cell_hash(ix, iy, iz, g.mask);
                if (pass == 0) {
                    atomicAdd(&bucket_cnt[h], 1u);
                } else {
                    unsigned p = atomicAdd(&cursor[h], 1u);
                    entries[bucket_start[h] + p] = f;
                }
            }
}

// Exclusive scan of n counts in two launches, kScanItems per workgroup: the sums of
// the workgroups' pieces, then every workgroup adds the sums before its own and scans
// its piece (integers: the order does not matter).  A single workgroup walking the
// array took 1.8 ms for the 2^20 buckets of a 512^2 sheet; this is one read of it,
// another and one write.
constexpr int kScanWG = 512, kScanPer = 16, kScanItems = kScanWG * kScanPer;

__device__ __forceinline__ unsigned scan_wave_sum(unsigned v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__global__ void __launch_bounds__(kScanWG) k_scan_sums(unsigned n, const unsigned *__restrict__ in,
                                                       unsigned *__restrict__ sums)
{
    __shared__ unsigned w[kScanWG / 64];
    const unsigned base = blockIdx.x * kScanItems;
    unsigned v = 0;
#pragma unroll
    for (int k = 0; k < kScanPer; ++k) {
        const unsigned i = base + k * kScanWG + threadIdx.x;
        v += i < n ? in[i] : 0u;
    }
    v = scan_wave_sum(v);
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned s = 0;
        for (int k = 0; k < kScanWG / 64; ++k) s += w[k];
        sums[blockIdx.x] = s;
    }
}

__global__ void __launch_bounds__(kScanWG) k_scan_write(unsigned n, const unsigned *__restrict__ in,
                                                        const unsigned *__restrict__ sums, unsigned *__restrict__ out,
                                                        unsigned *__restrict__ total)
{
    constexpr int NW = kScanWG / 64;
    __shared__ unsigned w[NW], piece[kScanItems + kScanItems / 32];   // one word of padding per 32: a lane's 16 items
    const unsigned base = blockIdx.x * kScanItems;
    const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
    auto at = [](int i) { return i + (i >> 5); };
    unsigned before = 0;
    for (unsigned b = t; b < blockIdx.x; b += kScanWG) before += sums[b];
    before = scan_wave_sum(before);
    if (lane == 0) w[wid] = before;
#pragma unroll
    for (int k = 0; k < kScanPer; ++k) {
        const unsigned i = base + k * kScanWG + t;
        piece[at(k * kScanWG + t)] = i < n ? in[i] : 0u;
    }
    __syncthreads();
    before = 0;
    for (int k = 0; k < NW; ++k) before += w[k];
    __syncthreads();
    // each thread its own kScanPer consecutive items, then the wavefront and the workgroup
    unsigned mine = 0;
#pragma unroll
    for (int k = 0; k < kScanPer; ++k) mine += piece[at(t * kScanPer + k)];
    unsigned inc = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned u = __shfl_up(inc, o, 64);
        if (lane >= o) inc += u;
    }
    if (lane == 63) w[wid] = inc;
    __syncthreads();
    unsigned run = before + inc - mine;
    for (int k = 0; k < wid; ++k) run += w[k];
#pragma unroll
    for (int k = 0; k < kScanPer; ++k) {
        const unsigned v = piece[at(t * kScanPer + k)];
        piece[at(t * kScanPer + k)] = run;
        run += v;
    }
    // the last thread's running sum is the sum of everything up to this piece's end
    if (total && t == kScanWG - 1 && blockIdx.x == gridDim.x - 1) *total = run;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kScanPer; ++k) {
        const unsigned i = base + k * kScanWG + t;
        if (i < n) out[i] = piece[at(k * kScanWG + t)];
    }
}

// ---------------------------------------------------------------------------
// One query point against a set of faces (the loop of boxTriCollision.cpp:782-844
// and 1152-1212); the best (dist, face) pair is kept lexicographically.
struct Best {
    double dist;
    int face;
};

// The reference's tests of one query against one face; its distance when they pass.
__device__ __forceinline__ bool accepts(const double *x1, const double *nor1, double thr, int j2,
                                        const double *__restrict__ xj, const int *__restrict__ tri,
                                        const double *__restrict__ fn, double &dist)
{
    const int *f2 = tri + 3 * j2;
    double nor2[3], dx[3], x2[3];
    ld(fn + 3 * j2, nor2);
    if (v_dot(nor1, nor2) < 0.0) v_neg(nor2);
    v_sub(x1, xj + 3 * f2[0], dx);
    double proj = v_dot(dx, nor2);
    if (proj < 0.0) return false;
    for (int i = 0; i < 3; ++i) x2[i] = x1[i] - proj * nor2[i];
    v_sub(x2, x1, dx);
    dist = v_norm(dx);
    if (dist > 5.0 * thr) return false;
    double u, v;
    barycentric(&u, &v, xj + 3 * f2[0], xj + 3 * f2[1], xj + 3 * f2[2], x1);
    double w = 1.0 - u - v;
    if (u < 0.0 || 1.0 < u || v < 0.0 || 1.0 < v || w < 0.0 || 1.0 < w) return false;
    return true;
}

__device__ __forceinline__ void take(Best &best, double dist, int j2)
{
    if (best.face < 0 || dist < best.dist || (dist == best.dist && j2 < best.face)) {
        best.dist = dist;
        best.face = j2;
    }
}

__device__ __forceinline__ void consider(const double *x1, const double *nor1, double thr, int j2,
                                         const double *__restrict__ xj, const int *__restrict__ tri,
                                         const double *__restrict__ fn, Best &best)
{
    double dist;
    if (accepts(x1, nor1, thr, j2, xj, tri, fn, dist)) take(best, dist, j2);
}

__device__ __forceinline__ Best best_min(Best a, Best b)
{
    if (a.face < 0) return b;
    if (b.face < 0) return a;
    if (b.dist < a.dist || (b.dist == a.dist && b.face < a.face)) return b;
    return a;
}

// Record of a query that found a face (V1-T2 / point-triangle), recomputed from the
// winner exactly as the reference builds it; an empty record without one.
__device__ void query_record(int q, int j2, const double *x1, const double *nor1, const double *__restrict__ xj,
                             const int *__restrict__ tri, const double *__restrict__ fn,
                             eolc_collision *__restrict__ out)
{
    eolc_collision c;
    rec_init(&c);
    if (j2 >= 0) {
        double nor2[3], dx[3], x2[3];
        const int *f2 = tri + 3 * j2;
        ld(fn + 3 * j2, nor2);
        if (v_dot(nor1, nor2) < 0.0) v_neg(nor2);
        v_sub(x1, xj + 3 * f2[0], dx);
        double proj = v_dot(dx, nor2);
        for (int i = 0; i < 3; ++i) x2[i] = x1[i] - proj * nor2[i];
        v_sub(x2, x1, dx);
        double u, v;
        barycentric(&u, &v, xj + 3 * f2[0], xj + 3 * f2[1], xj + 3 * f2[2], x1);
        c.dist = v_norm(dx);
        v_copy(nor1, c.nor1); v_copy(nor2, c.nor2);
        v_copy(x1, c.pos1); v_copy(x2, c.pos2);
        c.count1 = 1; c.count2 = 3;
        c.verts1[0] = q; c.verts1[1] = -1; c.verts1[2] = -1;
        c.verts2[0] = f2[0]; c.verts2[1] = f2[1]; c.verts2[2] = f2[2];
        c.weights1[0] = 1.0;
        c.weights2[0] = u; c.weights2[1] = v; c.weights2[2] = 1.0 - u - v;
        c.tri2 = j2;
    }
    out[q] = c;
}

// Few queries: every face against every query.  A query that lies outside a face's box,
// grown by the grid's margin, cannot pass its tests (face_cells' bound), so a face
// and a query cost six compares, with the query in scalar registers; what passes goes
// to a list (any order: the nearest is taken lexicographically) that k_cd_nearest
// reduces.  Faces too ill-shaped for the bound are tested against all.  A thread takes
// kSweepChunk queries (blockIdx.y the chunk): walking 2,048 took 0.35 ms on a 64^2
// sheet, whose 8,192 faces fill an eighth of the chip.
constexpr int kSweepChunk = 128;
struct Candidate {
    double dist;
    int query, face;
};

__global__ void __launch_bounds__(256)
k_cd_sweep(int F, int Q, const double *__restrict__ qpts, const double *__restrict__ qnrm, double thr, double cond_max,
           const double *__restrict__ clothaabb, const double *__restrict__ xj, const int *__restrict__ tri,
           const double *__restrict__ fn, unsigned cap, unsigned *__restrict__ ncand, Candidate *__restrict__ cand)
{
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= F) return;
    const double *a = xj + 3 * tri[3 * f], *b = xj + 3 * tri[3 * f + 1], *c = xj + 3 * tri[3 * f + 2];
    const double L = fmax(fmax(clothaabb[3] - clothaabb[0], clothaabb[4] - clothaabb[1]),
                          fmax(clothaabb[5] - clothaabb[2], 1e-300));
    GridParams g;
    g.margin = grid_margin(thr, L);
    g.cond_max = cond_max;
    const bool ill = ill_shaped(g, a, b, c);
    double lo[3], hi[3];
    for (int k = 0; k < 3; ++k) {
        lo[k] = ill ? -INFINITY : fmin(a[k], fmin(b[k], c[k])) - g.margin;
        hi[k] = ill ? INFINITY : fmax(a[k], fmax(b[k], c[k])) + g.margin;
    }
    const int q0 = blockIdx.y * kSweepChunk, q1 = min(q0 + kSweepChunk, Q);
#pragma unroll 4
    for (int q = q0; q < q1; ++q) {
        const double *x1 = qpts + 3 * q;
        if (!(x1[0] >= lo[0] && x1[0] <= hi[0] && x1[1] >= lo[1] && x1[1] <= hi[1] && x1[2] >= lo[2] && x1[2] <= hi[2]))
            continue;
        const double pt[6] = {x1[0], x1[1], x1[2], x1[0], x1[1], x1[2]};
        double dist;
        if (!check_aabb(pt, clothaabb) || !accepts(x1, qnrm + 3 * q, thr, f, xj, tri, fn, dist)) continue;
        const unsigned p = atomicAdd(ncand, 1u);
        if (p < cap) cand[p] = Candidate{dist, q, f};
    }
}

// One wavefront per query over the candidate list.
__global__ void __launch_bounds__(64)
k_cd_nearest(const double *__restrict__ qpts, const double *__restrict__ qnrm, const double *__restrict__ xj,
             const int *__restrict__ tri, const double *__restrict__ fn, unsigned cap,
             const unsigned *__restrict__ ncand, const Candidate *__restrict__ cand, eolc_collision *__restrict__ out)
{
    const int q = blockIdx.x;
    const unsigned n = min(*ncand, cap);
    Best best{0.0, -1};
    for (unsigned e = threadIdx.x; e < n; e += 64)
        if (cand[e].query == q) take(best, cand[e].dist, cand[e].face);
    for (int o = 32; o > 0; o >>= 1) {
        const double d = __shfl_xor(best.dist, o, 64);
        const int f = __shfl_xor(best.face, o, 64);
        if (f >= 0) take(best, d, f);
    }
    if (threadIdx.x == 0) {
        double x1[3], n1[3];
        ld(qpts + 3 * q, x1);
        ld(qnrm + 3 * q, n1);
        query_record(q, best.face, x1, n1, xj, tri, fn, out);
    }
}

// qpts/qnrm: query points and their normals; out[q] = the winning face's record.
__global__ void __launch_bounds__(256)
k_cd_query(int Q, GridParams g, const double *__restrict__ qpts, const double *__restrict__ qnrm, double thr,
           const double *__restrict__ clothaabb, const double *__restrict__ xj, const int *__restrict__ tri,
           const double *__restrict__ fn, const unsigned *__restrict__ bstart, const unsigned *__restrict__ bcnt,
           const int *__restrict__ entries, const unsigned *__restrict__ nalways, const int *__restrict__ always,
           eolc_collision *__restrict__ out)
{
    __shared__ double sd[256];
    __shared__ int sf[256];
    const int q = blockIdx.x;
    if (q >= Q) return;
    double x1[3], n1[3];
    ld(qpts + 3 * q, x1);
    ld(qnrm + 3 * q, n1);
    double pt[6] = {x1[0], x1[1], x1[2], x1[0], x1[1], x1[2]};
    Best best{0.0, -1};
    if (check_aabb(pt, clothaabb)) {
        int ix = clampi((int)floor((x1[0] - g.org[0]) * g.inv_cell), 0, g.dim[0] - 1);
        int iy = clampi((int)floor((x1[1] - g.org[1]) * g.inv_cell), 0, g.dim[1] - 1);
        int iz = clampi((int)floor((x1[2] - g.org[2]) * g.inv_cell), 0, g.dim[2] - 1);
        unsigned h = cell_hash(ix, iy, iz, g.mask);
        const unsigned s0 = bstart[h], n = bcnt[h];
        for (unsigned e = threadIdx.x; e < n; e += blockDim.x) consider(x1, n1, thr, entries[s0 + e], xj, tri, fn, best);
        const unsigned na = *nalways;
        for (unsigned e = threadIdx.x; e < na; e += blockDim.x) consider(x1, n1, thr, always[e], xj, tri, fn, best);
    }
    sd[threadIdx.x] = best.dist;
    sf[threadIdx.x] = best.face;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            Best a{sd[threadIdx.x], sf[threadIdx.x]}, b{sd[threadIdx.x + o], sf[threadIdx.x + o]};
            Best m = best_min(a, b);
            sd[threadIdx.x] = m.dist;
            sf[threadIdx.x] = m.face;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) query_record(q, sf[0], x1, n1, xj, tri, fn, out);
}

// ---------------------------------------------------------------------------
// Box V2-T1 (boxTriCollision.cpp:675-764) of one cloth vertex at x2, whose record is
// written to rec when it is not null.
__device__ bool v2t1(int i2, int F, double thr, const BoxGeom &box, const double *x2, const double *__restrict__ fn,
                     eolc_collision *__restrict__ rec, unsigned *__restrict__ err)
{
    const double pt[6] = {x2[0], x2[1], x2[2], x2[0], x2[1], x2[2]};
    if (!check_aabb(pt, box.aabb)) return false;
    for (int j1 = 0; j1 < 24; ++j1) {
        double dx[3];
        v_sub(x2, box.v[kBoxFaces[j1][0]], dx);
        if (v_dot(box.fn[j1], dx) > 0.0) return false;
    }
    eolc_collision best;
    int found = 0;
    for (int j1 = 0; j1 < 24; ++j1) {
        const double *x1a = box.v[kBoxFaces[j1][0]], *x1b = box.v[kBoxFaces[j1][1]], *x1c = box.v[kBoxFaces[j1][2]];
        const double *nor1 = box.fn[j1];
        double dx[3], x1[3];
        v_sub(x2, x1a, dx);
        double proj = v_dot(nor1, dx);
        if (proj > 0.0) continue;
        for (int i = 0; i < 3; ++i) x1[i] = x2[i] - proj * nor1[i];
        v_sub(x2, x1, dx);
        double dist = v_norm(dx);
        if (dist > 5.0 * thr) continue;
        double u, v;
        barycentric(&u, &v, x1a, x1b, x1c, x1);
        double w = 1.0 - u - v;
        if (u < 0.0 || 1.0 < u || v < 0.0 || 1.0 < v || w < 0.0 || 1.0 < w) continue;
        if (i2 >= F) {   // faceNors2.col(i2) would read past the face normals
            atomicOr(err, 1u);
            continue;
        }
        double nor2[3];
        ld(fn + 3 * i2, nor2);
        if (v_dot(nor2, nor1) < 0.0) v_neg(nor2);
        if (!found || dist < best.dist) {
            rec_init(&best);
            best.dist = dist;
            v_copy(nor1, best.nor1); v_copy(nor2, best.nor2);
            v_copy(x1, best.pos1); v_copy(x2, best.pos2);
            best.count1 = 3; best.count2 = 1;
            for (int i = 0; i < 3; ++i) best.verts1[i] = kBoxFaces[j1][i];
            best.verts2[0] = i2; best.verts2[1] = -1; best.verts2[2] = -1;
            best.weights1[0] = u; best.weights1[1] = v; best.weights1[2] = w;
            best.weights2[0] = 1.0;
            best.tri1 = j1;
            found = 1;
        }
    }
    if (found && rec) *rec = best;
    return found != 0;
}

// pointTri EOL branch (boxTriCollision.cpp:1099-1139): nearest point within thr.
// offs null: count (0 or 1 per vertex); else write the records at their offsets.
__global__ void __launch_bounds__(256)
k_cd_eolpts(int N, int P, double thr, const double *__restrict__ pts, const double *__restrict__ nrm,
            const double *__restrict__ xj, unsigned *__restrict__ cnt, const unsigned *__restrict__ offs,
            eolc_collision *__restrict__ out)
{
    int i2 = blockIdx.x * blockDim.x + threadIdx.x;
    if (i2 >= N) return;
    if (offs && !cnt[i2]) return;
    double x2[3];
    ld(xj + 3 * i2, x2);
    int bi = -1;
    double bd = 0.0;
    for (int i1 = 0; i1 < P; ++i1) {
        double dx[3];
        v_sub(x2, pts + 3 * i1, dx);
        double dist = v_norm(dx);
        if (dist < thr && (bi < 0 || dist < bd)) { bi = i1; bd = dist; }
    }
    if (!offs) {
        cnt[i2] = bi >= 0;
        return;
    }
    eolc_collision c;
    rec_init(&c);
    c.dist = bd;
    ld(nrm + 3 * bi, c.nor1); ld(nrm + 3 * bi, c.nor2);
    ld(pts + 3 * bi, c.pos1); v_copy(x2, c.pos2);
    c.count1 = 3; c.count2 = 1;
    c.verts1[0] = bi; c.verts1[1] = -1; c.verts1[2] = -1;
    c.verts2[0] = i2; c.verts2[1] = -1; c.verts2[2] = -1;
    c.weights1[0] = 1.0; c.weights2[0] = 1.0;
    out[offs[i2]] = c;
}

// ---------------------------------------------------------------------------
// The boxes b0 .. b1-1 of a group.  Box b's counts are cnt[b (N + E) ..], vertices then
// edges: one scan gives every record's place.  Count passes:
//   k_cd_boxes  V2-T1 of every cloth vertex (the first blocks_for(N) workgroups, one
//               thread each); every cloth edge (the others) is read once, and where it
//               reaches one of a box's 24 faces' bounds, which ee_pair requires of a box
//               edge's two, it goes to the list of pairs (any order)
//   k_cd_pairs  E2-E1 of the listed pairs, 12 lanes each, a lane per box edge
// With offs both write the records of the non-zero counts, from box b0's first on.
// A pair's tests are a long chain of dependent FP64 work that few edges need: a thread
// walking the 12 box edges of its own edge took 40 us a pass for one box at 64^2 and
// 240 us for four at 512^2, with the chip idle.
constexpr int kBoxWG = 256;
__global__ void __launch_bounds__(kBoxWG)
k_cd_boxes(int N, int E, int F, int b0, int b1, double thr, const BoxGeom *__restrict__ boxes,
           const int *__restrict__ cedges, const double *__restrict__ xj, const double *__restrict__ fn,
           unsigned *__restrict__ cnt, const unsigned *__restrict__ offs, unsigned *__restrict__ npairs,
           unsigned *__restrict__ pairs, unsigned *__restrict__ err, eolc_collision *__restrict__ out)
{
    const int NE = N + E, vblocks = (N + kBoxWG - 1) / kBoxWG;
    if ((int)blockIdx.x < vblocks) {
        const int i = blockIdx.x * kBoxWG + threadIdx.x;
        if (i >= N) return;
        double x2[3];
        ld(xj + 3 * i, x2);
        const unsigned o0 = offs ? offs[(size_t)b0 * NE] : 0u;
        for (int b = b0; b < b1; ++b) {
            const size_t k = (size_t)b * NE + i;
            if (!offs) cnt[k] = v2t1(i, F, thr, boxes[b], x2, fn, nullptr, err) ? 1u : 0u;
            else if (cnt[k]) v2t1(i, F, thr, boxes[b], x2, fn, out + (offs[k] - o0), err);
        }
        return;
    }
    const int k2 = ((int)blockIdx.x - vblocks) * kBoxWG + threadIdx.x;
    if (k2 >= E) return;
    const int *e2 = cedges + 4 * k2;
    double aabbE[6];
    for (int i = 0; i < 3; ++i) {
        double a = xj[3 * e2[0] + i], b = xj[3 * e2[1] + i];
        aabbE[i] = a < b ? a : b;
        aabbE[i + 3] = a < b ? b : a;
    }
    for (int b = b0; b < b1; ++b) {
        const unsigned k = (unsigned)b * (unsigned)NE + (unsigned)(N + k2);
        cnt[k] = 0;
        if (!check_aabb(boxes[b].aabb, aabbE)) continue;
        bool near = false;
        for (int f = 0; f < 24; ++f) near = near || check_aabb(boxes[b].faabb[f], aabbE);
        if (near) pairs[atomicAdd(npairs, 1u)] = k;
    }
}

// Workgroups stride over the listed pairs of the boxes b0 .. b1-1, five to a wavefront.
constexpr int kPairGrid = 1024;
__global__ void __launch_bounds__(64)
k_cd_pairs(int N, int E, int b0, int b1, double thr, const BoxGeom *__restrict__ boxes, const int *__restrict__ cedges,
           const double *__restrict__ x, const double *__restrict__ xj, const int *__restrict__ tri,
           unsigned *__restrict__ cnt, const unsigned *__restrict__ offs, const unsigned *__restrict__ npairs,
           const unsigned *__restrict__ pairs, unsigned *__restrict__ nambig, eolc_collision *__restrict__ out)
{
    const unsigned NE = (unsigned)(N + E), n = *npairs;
    const int lane = threadIdx.x, grp = lane / 12, k1 = lane % 12;
    for (unsigned p0 = 5 * blockIdx.x; p0 < n; p0 += 5 * gridDim.x) {   // uniform in the wavefront
        bool on = grp < 5 && p0 + grp < n;
        const unsigned k = on ? pairs[p0 + grp] : 0u;
        const int b = (int)(k / NE), e = (int)(k % NE) - N;
        if (offs) on = on && b >= b0 && b < b1 && cnt[k];
        ClothEdge ce;
        int hit = 0, amb = 0;
        if (on) {
            cloth_edge(e, cedges, x, xj, tri, ce);
            hit = ee_pair(e, k1, thr, boxes[b], ce, nullptr, &amb, kAcosBand);
        }
        const unsigned bits = (unsigned)(__ballot(hit) >> (12 * grp)) & 0xfffu;
        if (!on) continue;
        if (!offs) {
            if (k1 == 0) cnt[k] = __popc(bits);
            if (amb) atomicOr(&nambig[b], 1u);
        } else if (hit) {
            ee_pair(e, k1, thr, boxes[b], ce,
                    out + (offs[k] - offs[(size_t)b0 * NE]) + __popc(bits & ((1u << k1) - 1)), &amb, kAcosBand);
        }
    }
}

// The acos-ambiguous pairs of one box, per edge (only when k_cd_boxes saw one).
__global__ void __launch_bounds__(256)
k_cd_ambiguous(int E, double thr, const BoxGeom *__restrict__ box, const int *__restrict__ cedges,
               const double *__restrict__ x, const double *__restrict__ xj, const int *__restrict__ tri,
               int *__restrict__ ambig)
{
    const int k2 = blockIdx.x * blockDim.x + threadIdx.x;
    if (k2 >= E) return;
    const int *e2 = cedges + 4 * k2;
    double aabbE[6];
    for (int i = 0; i < 3; ++i) {
        double a = xj[3 * e2[0] + i], b = xj[3 * e2[1] + i];
        aabbE[i] = a < b ? a : b;
        aabbE[i + 3] = a < b ? b : a;
    }
    int mask = 0;
    if (check_aabb(box->aabb, aabbE)) ee_edge(k2, thr, *box, cedges, x, xj, tri, nullptr, &mask, kAcosBand);
    ambig[k2] = mask;
}

// first[2 b], first[2 b + 1]: the offsets of box b's vertex and edge records; first[2 nb]:
// their number (the scan leaves it behind the last offset)
__global__ void k_cd_first(int nb, int N, int NE, const unsigned *__restrict__ offs, unsigned *__restrict__ first)
{
    const int t = threadIdx.x;
    if (t <= 2 * nb) first[t] = offs[(size_t)(t >> 1) * NE + ((t & 1) ? N : 0)];
}

inline int blocks_for(int64_t n, int t = 256) { return (int)((n + t - 1) / t); }

// Device memory of eolc_collide_noalloc: one array per GPU, held from the loading of
// the code object until the process ends.  Host code never passes `scratch` itself
// to a kernel or a copy (in host code the name is a stand-in, not a device address):
// it uses the address that hipGetSymbolAddress returns for the current device.
__device__ __align__(256) unsigned char scratch[eolc::kCollideScratchBytes];

constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxScratchDevices] = {};
std::mutex g_scratch_call_mu[kMaxScratchDevices];

}  // namespace

namespace eolc {

hipError_t collide_scratch(int device, void **ptr)
{
    *ptr = nullptr;
    if (device < 0 || device >= kMaxScratchDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        int cur = -1;
        hipError_t e = hipGetDevice(&cur);
        if (e != hipSuccess) return e;
        if (cur != device && (e = hipSetDevice(device)) != hipSuccess) return e;
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != device) (void)hipSetDevice(cur);
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        g_scratch_ptr[device] = p;
    }
    *ptr = g_scratch_ptr[device];
    return hipSuccess;
}

std::mutex *collide_scratch_lock(int device)
{
    return (device >= 0 && device < kMaxScratchDevices) ? &g_scratch_call_mu[device] : nullptr;
}

// Launch wrappers used by collide_host.cpp --------------------------------------
hipError_t cd_prep(eolc_ctx *c, double thr, double *xj, double *fn, double *aabb_part, double *aabb)
{
    const int N = c->topo.N, F = c->topo.F;
    hipLaunchKernelGGL(k_cd_prep, dim3(blocks_for(3 * N)), dim3(256), 0, c->stream, N, F, thr, c->x, c->cd_unit,
                       c->tri, xj, fn);
    hipLaunchKernelGGL(k_cd_fnormals, dim3(blocks_for(F)), dim3(256), 0, c->stream, F, xj, c->tri, fn);
    hipLaunchKernelGGL(k_cd_aabb, dim3(kAabbParts), dim3(256), 0, c->stream, N, xj, aabb_part);
    hipLaunchKernelGGL(k_cd_aabb_final, dim3(1), dim3(kAabbParts), 0, c->stream, aabb_part, aabb);
    return hipGetLastError();
}

size_t cd_scan_words(size_t n) { return (n + kScanItems - 1) / kScanItems; }

// Exclusive scan of in[0..n) into out, the sum into *total; sums: cd_scan_words(n).
hipError_t cd_scan(eolc_ctx *c, unsigned n, const unsigned *in, unsigned *out, unsigned *sums, unsigned *total)
{
    const int nb = (int)std::max<size_t>(cd_scan_words(n), 1);
    hipLaunchKernelGGL(k_scan_sums, dim3(nb), dim3(kScanWG), 0, c->stream, n, in, sums);
    hipLaunchKernelGGL(k_scan_write, dim3(nb), dim3(kScanWG), 0, c->stream, n, in, sums, out, total);
    return hipGetLastError();
}

hipError_t cd_grid_build(eolc_ctx *c, const eolc_cd::CdGrid &gp, const double *xj, unsigned *bcnt, unsigned *bstart,
                         unsigned *cursor, int *entries, unsigned *nalways, int *always, unsigned *sums, unsigned *total,
                         bool fill)
{
    const int F = c->topo.F;
    GridParams g;
    for (int k = 0; k < 3; ++k) { g.org[k] = gp.org[k]; g.dim[k] = gp.dim[k]; }
    g.inv_cell = gp.inv_cell;
    g.mask = gp.mask;
    g.margin = gp.margin;
    g.cond_max = gp.cond_max;
    if (!fill) {
        hipLaunchKernelGGL(k_grid_insert, dim3(blocks_for(F)), dim3(256), 0, c->stream, F, 0, g, xj, c->tri, bcnt,
                           bstart, cursor, entries, nalways, always);
        const hipError_t e = cd_scan(c, gp.mask + 1, bcnt, bstart, sums, total);
        if (e != hipSuccess) return e;
    } else {
        hipLaunchKernelGGL(k_grid_insert, dim3(blocks_for(F)), dim3(256), 0, c->stream, F, 1, g, xj, c->tri, bcnt,
                           bstart, cursor, entries, nalways, always);
    }
    return hipGetLastError();
}

hipError_t cd_query(eolc_ctx *c, const eolc_cd::CdGrid &gp, int Q, const double *qpts, const double *qnrm, double thr,
                    const double *aabb, const double *xj, const double *fn, const unsigned *bstart, const unsigned *bcnt,
                    const int *entries, const unsigned *nalways, const int *always, eolc_collision *rec)
{
    if (Q <= 0) return hipSuccess;
    GridParams g;
    for (int k = 0; k < 3; ++k) { g.org[k] = gp.org[k]; g.dim[k] = gp.dim[k]; }
    g.inv_cell = gp.inv_cell;
    g.mask = gp.mask;
    g.margin = gp.margin;
    g.cond_max = gp.cond_max;
    hipLaunchKernelGGL(k_cd_query, dim3(Q), dim3(256), 0, c->stream, Q, g, qpts, qnrm, thr, aabb, xj, c->tri, fn,
                       bstart, bcnt, entries, nalways, always, rec);
    return hipGetLastError();
}

hipError_t cd_sweep(eolc_ctx *c, int Q, const double *qpts, const double *qnrm, double thr, const double *aabb,
                    const double *xj, const double *fn, unsigned *ncand, void *cand, eolc_collision *rec)
{
    if (Q <= 0) return hipSuccess;
    const int F = c->topo.F;
    Candidate *cd = static_cast<Candidate *>(cand);
    if (F > 0)
        hipLaunchKernelGGL(k_cd_sweep, dim3(blocks_for(F), blocks_for(Q, kSweepChunk)), dim3(256), 0, c->stream, F, Q, qpts, qnrm, thr,
                           eolc_cd::kGridCondMax, aabb, xj, c->tri, fn, kCdCandidates, ncand, cd);
    hipLaunchKernelGGL(k_cd_nearest, dim3(Q), dim3(64), 0, c->stream, qpts, qnrm, xj, c->tri, fn, kCdCandidates, ncand,
                       cd, rec);
    return hipGetLastError();
}

hipError_t cd_eolpts(eolc_ctx *c, int P, double thr, const double *pts, const double *nrm, const double *xj,
                     unsigned *cnt, const unsigned *offs, eolc_collision *out)
{
    const int N = c->topo.N;
    hipLaunchKernelGGL(k_cd_eolpts, dim3(blocks_for(N)), dim3(256), 0, c->stream, N, P, thr, pts, nrm, xj, cnt, offs,
                       out);
    return hipGetLastError();
}

hipError_t cd_boxes(eolc_ctx *c, int b0, int b1, double thr, const eolc_cd::BoxGeom *boxes, const double *xj,
                    const double *fn, unsigned *cnt, const unsigned *offs, unsigned *npairs, unsigned *pairs,
                    unsigned *nambig, unsigned *err, eolc_collision *out)
{
    const int N = c->topo.N, E = c->n_cedges;
    // the record pass reads the edges from the list alone
    const int blocks = blocks_for(N, kBoxWG) + (offs ? 0 : blocks_for(E, kBoxWG));
    hipLaunchKernelGGL(k_cd_boxes, dim3(blocks), dim3(kBoxWG), 0, c->stream, N, E, c->topo.F, b0, b1, thr, boxes,
                       c->cedges, xj, fn, cnt, offs, npairs, pairs, err, out);
    if (E > 0)
        hipLaunchKernelGGL(k_cd_pairs, dim3(kPairGrid), dim3(64), 0, c->stream, N, E, b0, b1, thr, boxes, c->cedges,
                           c->x, xj, c->tri, cnt, offs, npairs, pairs, nambig, out);
    return hipGetLastError();
}

hipError_t cd_ambiguous(eolc_ctx *c, double thr, const eolc_cd::BoxGeom *box, const double *xj, int *ambig)
{
    const int E = c->n_cedges;
    if (E == 0) return hipSuccess;
    hipLaunchKernelGGL(k_cd_ambiguous, dim3(blocks_for(E)), dim3(256), 0, c->stream, E, thr, box, c->cedges, c->x, xj,
                       c->tri, ambig);
    return hipGetLastError();
}

hipError_t cd_first(eolc_ctx *c, int nb, const unsigned *offs, unsigned *first)
{
    static_assert(2 * kCdBoxes < 64, "one wavefront");
    hipLaunchKernelGGL(k_cd_first, dim3(1), dim3(64), 0, c->stream, nb, c->topo.N, c->topo.N + c->n_cedges, offs,
                       first);
    return hipGetLastError();
}

}  // namespace eolc
