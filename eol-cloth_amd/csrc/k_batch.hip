// Batched cloths (gfx950): many independent cloth instances, concatenated into one
// context, solved in ONE persistent launch.
//
// Every instance's vertex range is padded to a multiple of 64, so each 64-row
// SELL slice of the concatenated matrix belongs to exactly one instance; padding
// vertices are isolated and fixed.  Workgroup w of the persistent solve owns
// instance order[w] (largest first, so consecutive large instances land on
// different XCDs, which receive workgroups round-robin) and runs that instance's
// whole mixed-precision PCG -- the velocity solve of GeneralizedSolver::velocitySolve
// for solver "none" (GeneralizedSolver.cpp:107-172) -- to its own tolerance:
//   FP32 difference-form SpMV (row mass plus S'_ij (p_j - p_i), the diagonal
//   entry skipped) and block-Jacobi, FP64 dot products, FP64 true
//   residual at every reliable update (delta), iterate accumulated in FP64.
// No grid-wide synchronisation exists: the instances are independent, a workgroup
// only touches its own rows, and an instance that has converged simply leaves
// (its workgroup exits) -- the per-instance convergence mask.
//
// Reductions: each wave reduces its slice's 64 rows with a fixed shuffle tree and
// writes one partial per slice; after a barrier wave 0 sums the instance's slice
// partials in slice order.  The result does not depend on the workgroup size, so
// the autotuned launch shape never changes the answer.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "eolc_internal.h"

// Multiply-adds are written out (fma where fused); the compiler contracts nothing,
// so every workgroup-size instantiation rounds identically.
#pragma clang fp contract(off)

namespace {

constexpr int SL = eolc::kSlice;

inline int blocks_for(int64_t n, int t = 256) { return (int)((n + t - 1) / t); }

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}

// Sum over the instance's slices of K per-row values; the result is returned to
// every thread.  part: K x nslices scratch, red: K doubles of LDS.
template <int K>
__device__ __forceinline__ void inst_sum(double (&v)[K], const eolc::BatchInst &I, const double *__restrict__ part,
                                         int nslices, double *red)
{
    __syncthreads();   // the per-slice partials of every wave are written
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (wave == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            double s = 0.0;
            for (int sl = I.s0 + lane; sl < I.s1; sl += 64) s += part[k * nslices + sl];
            s = wave_sum(s);
            if (lane == 0) red[k] = s;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = red[k];
}

// Per-slice partial of K values held one per lane (all 64 lanes of the wave).
template <int K>
__device__ __forceinline__ void slice_partial(const double (&v)[K], int sl, double *__restrict__ part, int nslices)
{
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const double s = wave_sum(v[k]);
        if ((threadIdx.x & 63) == 0) part[k * nslices + sl] = s;
    }
}

// Products of a row's SELL entries added in order, AH entries' loads in flight: a
// workgroup owns a whole instance, so a wavefront walks up to 17 slices one after the
// other and every dependent load is waited for.  apply(j, a): one entry's block (9
// values) on column j.
template <class T, int AH, class Apply>
__device__ __forceinline__ void row_entries(const T *__restrict__ A, int64_t nbs, const int *__restrict__ cl, int base,
                                            int len, Apply apply)
{
    for (int k0 = 0; k0 < len; k0 += AH) {
        T a[AH][9];
        int j[AH];
#pragma unroll
        for (int u = 0; u < AH; ++u)
            if (k0 + u < len) {
                const int e = base + (k0 + u) * SL;
                j[u] = cl[e];
#pragma unroll
                for (int c = 0; c < 9; ++c) a[u][c] = A[c * nbs + e];
            }
        apply(j, a, len - k0);
    }
}

// FP64 row product y = (A x)_row over the SELL entries of one row.
__device__ __forceinline__ void row_spmv64(const double *__restrict__ A, int64_t nbs, const int *__restrict__ cl,
                                           int base, int len, const double *__restrict__ x, double &y0, double &y1,
                                           double &y2)
{
    y0 = y1 = y2 = 0.0;
    constexpr int AH = 2;   // four spill at 1,024 threads
    row_entries<double, AH>(A, nbs, cl, base, len, [&](const int (&j)[AH], const double (&a)[AH][9], int n) {
        double u[AH][3];
#pragma unroll
        for (int t = 0; t < AH; ++t)
            if (t < n)
#pragma unroll
                for (int c = 0; c < 3; ++c) u[t][c] = x[3 * j[t] + c];
#pragma unroll
        for (int t = 0; t < AH; ++t)
            if (t < n) {
                y0 += fma(a[t][2], u[t][2], fma(a[t][1], u[t][1], a[t][0] * u[t][0]));
                y1 += fma(a[t][5], u[t][2], fma(a[t][4], u[t][1], a[t][3] * u[t][0]));
                y2 += fma(a[t][8], u[t][2], fma(a[t][7], u[t][1], a[t][6] * u[t][0]));
            }
    });
}

// FP32 difference form: y += S'_ij (p_j - p_i) over the entries, p by get(j, c).
template <class Get>
__device__ __forceinline__ void row_spmv32(const float *__restrict__ S, int64_t nbs, const int *__restrict__ cl,
                                           int base, int len, float ui0, float ui1, float ui2, double &y0, double &y1,
                                           double &y2, Get get)
{
    constexpr int AH = 4;
    row_entries<float, AH>(S, nbs, cl, base, len, [&](const int (&j)[AH], const float (&a)[AH][9], int n) {
        float u[AH][3];
#pragma unroll
        for (int t = 0; t < AH; ++t)
            if (t < n)
#pragma unroll
                for (int c = 0; c < 3; ++c) u[t][c] = get(j[t], c);
#pragma unroll
        for (int t = 0; t < AH; ++t)
            if (t < n) {
                const float d0 = u[t][0] - ui0, d1 = u[t][1] - ui1, d2 = u[t][2] - ui2;
                y0 += (double)fmaf(a[t][2], d2, fmaf(a[t][1], d1, a[t][0] * d0));
                y1 += (double)fmaf(a[t][5], d2, fmaf(a[t][4], d1, a[t][3] * d0));
                y2 += (double)fmaf(a[t][8], d2, fmaf(a[t][7], d1, a[t][6] * d0));
            }
    });
}

// Runs load and then use on the instance's slices, two slices a trip.  The vector passes take the rows in vertex order (slice s
// holds the vertices 64 s .. 64 s + 63), without the storage order's index load.
template <int WGS, class Slice, class Load, class Use>
__device__ __forceinline__ void each_slice(const eolc::BatchInst &I, Load load, Use use)
{
    constexpr int NW = WGS / 64;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int sl = I.s0 + wave; sl < I.s1; sl += 2 * NW) {
        Slice a, b;
        const bool two = sl + NW < I.s1;   // uniform in the wavefront
        load(a, sl * SL + lane);
        if (two) load(b, (sl + NW) * SL + lane);
        use(a, sl, sl * SL + lane);
        if (two) use(b, sl + NW, (sl + NW) * SL + lane);
    }
}

// out = b - A x (masked), returns ||out||^2 over the instance.  b may be null.
template <int WGS>
__device__ double inst_residual64(const eolc::BatchInst &I, const int *__restrict__ slice_off,
                                  const int *__restrict__ srow, const int *__restrict__ slen,
                                  const int *__restrict__ scol, const double *__restrict__ A, int64_t nbs,
                                  const unsigned char *__restrict__ fixmask, const double *__restrict__ x,
                                  const double *__restrict__ b, double *__restrict__ out, double *part, int nslices,
                                  double *red)
{
    constexpr int NW = WGS / 64;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int sl = I.s0 + wave; sl < I.s1; sl += NW) {
        const int g = sl * SL + lane;
        const int row = srow[g];
        double y0, y1, y2;
        row_spmv64(A, nbs, scol, slice_off[sl] + lane, slen[g], x, y0, y1, y2);
        double o0 = (b ? b[3 * row] : 0.0) - y0, o1 = (b ? b[3 * row + 1] : 0.0) - y1,
               o2 = (b ? b[3 * row + 2] : 0.0) - y2;
        const unsigned fm = fixmask[row];
        if (fm & 1) o0 = 0.0;
        if (fm & 2) o1 = 0.0;
        if (fm & 4) o2 = 0.0;
        out[3 * row] = o0; out[3 * row + 1] = o1; out[3 * row + 2] = o2;
        const double v[1] = {(o0 * o0 + o1 * o1) + o2 * o2};
        slice_partial<1>(v, sl, part, nslices);
    }
    double s[1];
    inst_sum<1>(s, I, part, nslices, red);
    return s[0];
}

// r32 = (float) r64, z = D r32; returns (r.z, r.r) over the instance.
template <int WGS>
__device__ void inst_precond(const eolc::BatchInst &I, int N, const float *__restrict__ D,
                             const double *__restrict__ r64, float *__restrict__ r32, float *__restrict__ z32,
                             double *part, int nslices, double *red, double &rz, double &rr)
{
    struct In { double r[3]; float d[6]; };
    each_slice<WGS, In>(
        I,
        [&](In &x, int i) {
#pragma unroll
            for (int c = 0; c < 3; ++c) x.r[c] = r64[3 * i + c];
#pragma unroll
            for (int c = 0; c < 6; ++c) x.d[c] = D[c * N + i];
        },
        [&](const In &x, int sl, int i) {
            const float r0 = (float)x.r[0], r1 = (float)x.r[1], r2 = (float)x.r[2];
            r32[3 * i] = r0; r32[3 * i + 1] = r1; r32[3 * i + 2] = r2;
            const double s0 = r0, s1 = r1, s2 = r2;
            const double e00 = x.d[0], e01 = x.d[1], e02 = x.d[2], e11 = x.d[3], e12 = x.d[4], e22 = x.d[5];
            const float z0 = (float)fma(e02, s2, fma(e01, s1, e00 * s0));
            const float z1 = (float)fma(e12, s2, fma(e11, s1, e01 * s0));
            const float z2 = (float)fma(e22, s2, fma(e12, s1, e02 * s0));
            z32[3 * i] = z0; z32[3 * i + 1] = z1; z32[3 * i + 2] = z2;
            const double v[2] = {(s0 * (double)z0 + s1 * (double)z1) + s2 * (double)z2, (s0 * s0 + s1 * s1) + s2 * s2};
            slice_partial<2>(v, sl, part, nslices);
        });
    double s[2];
    inst_sum<2>(s, I, part, nslices, red);
    rz = s[0];
    rr = s[1];
}

// Multilevel coarse levels inside the persistent solve: the hierarchy of the
// concatenated topology never spans two instances, and its hierarchical numbering
// gives every instance a contiguous aggregate range per level (lo), so a workgroup
// applies its instance's levels alone, with workgroup barriers between levels.
struct BatchML {
    eolc::MLLevels lv;
    const int *hord, *ptr1, *agg1, *par, *cptr;
    const int *lo;   // (B + 1) x (kMLMaxLevels + 1): first aggregate of instance b at level l
    const double *Dinv;
    double *R, *C;
};

__device__ __forceinline__ void ml_inv_apply(const double *__restrict__ d, double r0, double r1, double r2, double &c0,
                                             double &c1, double &c2)
{
    c0 = fma(d[2], r2, fma(d[1], r1, d[0] * r0));
    c1 = fma(d[4], r2, fma(d[3], r1, d[1] * r0));
    c2 = fma(d[5], r2, fma(d[4], r1, d[2] * r0));
}

// Sum of n 3-vectors in order, eight loads in flight; get(k, c): component c of the kth.
template <class Get> __device__ __forceinline__ void sum3(int k0, int k1, double (&t)[3], Get get)
{
    t[0] = t[1] = t[2] = 0.0;
    for (int k = k0; k < k1; k += 8) {
        double v[8][3];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int q = min(k + u, k1 - 1);
            get(q, v[u]);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (k + u < k1)
#pragma unroll
                for (int c = 0; c < 3; ++c) t[c] += v[u][c];
    }
}

// z = D r + sum_l Z_l D_l^-1 Z_l^T r over instance b (r32 of its rows complete);
// returns r.z over the instance.  Sums in member / child order, FP64.
template <int WGS>
__device__ double inst_ml_apply(const eolc::BatchInst &I, int b, const BatchML &m, int N, const float *__restrict__ D,
                                const float *__restrict__ r32, float *__restrict__ z32,
                                const unsigned char *__restrict__ fixmask, double *part, int nslices, double *red)
{
    constexpr int S = eolc::kMLMaxLevels + 1;
    const int L = m.lv.L;
    __syncthreads();   // every row's r32 is written
    {
        const int lo = m.lo[b * S + 1], hi = m.lo[(b + 1) * S + 1];
        for (int a = lo + (int)threadIdx.x; a < hi; a += WGS) {
            double t[3];
            sum3(m.ptr1[a], m.ptr1[a + 1], t, [&](int k, double (&v)[3]) {
                const int i = m.hord[k];
#pragma unroll
                for (int c = 0; c < 3; ++c) v[c] = (double)r32[3 * i + c];
            });
#pragma unroll
            for (int c = 0; c < 3; ++c) m.R[3 * a + c] = t[c];
        }
    }
    __syncthreads();
    for (int l = 2; l <= L; ++l) {
        const int lo = m.lo[b * S + l], hi = m.lo[(b + 1) * S + l];
        for (int A = lo + (int)threadIdx.x; A < hi; A += WGS) {
            double t[3];
            sum3(m.cptr[m.lv.coff[l] + A], m.cptr[m.lv.coff[l] + A + 1], t, [&](int a, double (&v)[3]) {
                const double *q = m.R + 3 * (int64_t)(m.lv.off[l - 1] + a);
#pragma unroll
                for (int c = 0; c < 3; ++c) v[c] = q[c];
            });
            double *o = m.R + 3 * (int64_t)(m.lv.off[l] + A);
#pragma unroll
            for (int c = 0; c < 3; ++c) o[c] = t[c];
        }
        __syncthreads();
    }
    for (int l = L; l >= 1; --l) {
        const int lo = m.lo[b * S + l], hi = m.lo[(b + 1) * S + l];
        for (int a = lo + (int)threadIdx.x; a < hi; a += WGS) {
            const int64_t g = m.lv.off[l] + a;
            double c0, c1, c2;
            ml_inv_apply(m.Dinv + 6 * g, m.R[3 * g], m.R[3 * g + 1], m.R[3 * g + 2], c0, c1, c2);
            if (l < L) {
                const double *up = m.C + 3 * (int64_t)(m.lv.off[l + 1] + m.par[g]);
                c0 += up[0]; c1 += up[1]; c2 += up[2];
            }
            m.C[3 * g] = c0; m.C[3 * g + 1] = c1; m.C[3 * g + 2] = c2;
        }
        __syncthreads();
    }
    struct In { float r[3], d[6]; double c[3]; unsigned fm; };
    each_slice<WGS, In>(
        I,
        [&](In &x, int i) {
            const double *cc = m.C + 3 * (int64_t)m.agg1[i];
#pragma unroll
            for (int c = 0; c < 6; ++c) x.d[c] = D[c * N + i];
#pragma unroll
            for (int c = 0; c < 3; ++c) x.r[c] = r32[3 * i + c];
            x.fm = fixmask[i];
#pragma unroll
            for (int c = 0; c < 3; ++c) x.c[c] = cc[c];
        },
        [&](const In &x, int sl, int i) {
            const float r0 = x.r[0], r1 = x.r[1], r2 = x.r[2];
            float f0, f1, f2;
            eolc::apply_sym3<float>(x.d, 1, r0, r1, r2, f0, f1, f2);
            const float z0 = (x.fm & 1u) ? 0.0f : (float)((double)f0 + x.c[0]);
            const float z1 = (x.fm & 2u) ? 0.0f : (float)((double)f1 + x.c[1]);
            const float z2 = (x.fm & 4u) ? 0.0f : (float)((double)f2 + x.c[2]);
            z32[3 * i] = z0; z32[3 * i + 1] = z1; z32[3 * i + 2] = z2;
            const double v[1] = {((double)r0 * (double)z0 + (double)r1 * (double)z1) + (double)r2 * (double)z2};
            slice_partial<1>(v, sl, part, nslices);
        });
    double s[1];
    inst_sum<1>(s, I, part, nslices, red);
    return s[0];
}

// r32 = (float) r64 and r.r over the instance (the multilevel path forms z after).
template <int WGS>
__device__ double inst_convert(const eolc::BatchInst &I, const double *__restrict__ r64, float *__restrict__ r32,
                               double *part, int nslices, double *red)
{
    constexpr int NW = WGS / 64;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int sl = I.s0 + wave; sl < I.s1; sl += NW) {
        const int i = sl * SL + lane;
        const float r0 = (float)r64[3 * i], r1 = (float)r64[3 * i + 1], r2 = (float)r64[3 * i + 2];
        r32[3 * i] = r0; r32[3 * i + 1] = r1; r32[3 * i + 2] = r2;
        const double s0 = r0, s1 = r1, s2 = r2;
        const double v[1] = {(s0 * s0 + s1 * s1) + s2 * s2};
        slice_partial<1>(v, sl, part, nslices);
    }
    double s[1];
    inst_sum<1>(s, I, part, nslices, red);
    return s[0];
}

struct BatchArgs {
    const eolc::BatchInst *inst;
    const int *order;
    const int *slice_off, *srow, *slen, *scol;
    const double *A64;
    const float *S32, *M32, *D32;
    int64_t nbs;
    int N, nslices;
    const unsigned char *fixmask;
    const double *vfix, *rhs;
    double *v, *xs64, *r64, *b64;
    float *r32, *z32, *q32, *xl32, *p32a, *p32b;
    double *part;
    double tol2, delta2;
    int maxit;
    int *stats;
    double *dstats;
    int stage;   // rows of LDS (3 floats each) the launch provides
    BatchML ml;
};

// Persistent mixed-precision PCG, one workgroup per instance.  ML: the preconditioner
// adds the instance's multilevel coarse levels to the block-Jacobi blocks.  The search
// direction of an instance of at most `stage` rows is kept in LDS for the product, whose
// column gathers (six dwords a block from two vectors) otherwise take more of the compute
// unit's address rate than the block's own nine.  A 96 x 96 sheet's iteration takes 95 us
// (190 us with one entry's loads at a time and the direction gathered from global
// memory): 51 the product, the rest the passes over its vectors at 80 GB/s and the
// barriers.  The next entries loaded ahead (56-60 us a product), the direction in LDS
// alone and the levels >= 2 in LDS gained nothing.
template <int WGS, bool ML>
__global__ void __launch_bounds__(WGS) k_batch_pcg(BatchArgs a)
{
    constexpr int NW = WGS / 64;
    __shared__ double red[4];
    extern __shared__ float su[];   // 3 per row of a staged instance
    const int b = a.order[blockIdx.x];
    const eolc::BatchInst I = a.inst[b];
    const bool staged = I.v1 - I.v0 <= a.stage;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int N = a.N, ns = a.nslices;
    const int64_t nbs = a.nbs;

    // b_red = rhs - A vfix (masked); x0 = masked v_old; r = b_red - A x0
    const double bnorm2 = inst_residual64<WGS>(I, a.slice_off, a.srow, a.slen, a.scol, a.A64, nbs, a.fixmask, a.vfix,
                                               a.rhs, a.b64, a.part, ns, red);
    for (int sl = I.s0 + wave; sl < I.s1; sl += NW) {
        const int i = a.srow[sl * SL + lane];
        const unsigned fm = a.fixmask[i];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            a.xs64[3 * i + c] = ((fm >> c) & 1) ? 0.0 : a.v[3 * i + c];
            a.xl32[3 * i + c] = 0.0f;
            a.p32a[3 * i + c] = 0.0f;
        }
    }
    __syncthreads();
    double rmax2 = inst_residual64<WGS>(I, a.slice_off, a.srow, a.slen, a.scol, a.A64, nbs, a.fixmask, a.xs64, a.b64,
                                        a.r64, a.part, ns, red);
    double rz, rr;
    if constexpr (ML) {
        rr = inst_convert<WGS>(I, a.r64, a.r32, a.part, ns, red);
        rz = inst_ml_apply<WGS>(I, b, a.ml, N, a.D32, a.r32, a.z32, a.fixmask, a.part, ns, red);
    } else {
        inst_precond<WGS>(I, N, a.D32, a.r64, a.r32, a.z32, a.part, ns, red, rz, rr);
    }
    double rz_prev = 1.0;
    int k = 0, first = 0, refinements = 0, status = EOLC_ERR_MAXIT;
    float *pold = a.p32a, *pnew = a.p32b;
    const double thr_final = a.tol2 * bnorm2;
    for (;;) {
        const double thr = fmax(thr_final, a.delta2 * rmax2);
        if (!isfinite(rr) || !isfinite(rz)) {
            status = EOLC_ERR_NONFINITE;
            break;
        }
        if (rr <= thr) {
            // reliable update: fold the FP32 correction in, FP64 true residual
            for (int sl = I.s0 + wave; sl < I.s1; sl += NW) {
                const int i = a.srow[sl * SL + lane];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    a.xs64[3 * i + c] += (double)a.xl32[3 * i + c];
                    a.xl32[3 * i + c] = 0.0f;
                }
            }
            __syncthreads();
            rmax2 = inst_residual64<WGS>(I, a.slice_off, a.srow, a.slen, a.scol, a.A64, nbs, a.fixmask, a.xs64, a.b64,
                                         a.r64, a.part, ns, red);
            ++refinements;
            if (!isfinite(rmax2)) {
                status = EOLC_ERR_NONFINITE;
                break;
            }
            if (rmax2 <= thr_final) {
                status = EOLC_OK;
                break;
            }
            if (k >= a.maxit || refinements > eolc::kMaxRefinements) break;
            if constexpr (ML) {
                rr = inst_convert<WGS>(I, a.r64, a.r32, a.part, ns, red);
                rz = inst_ml_apply<WGS>(I, b, a.ml, N, a.D32, a.r32, a.z32, a.fixmask, a.part, ns, red);
            } else {
                inst_precond<WGS>(I, N, a.D32, a.r64, a.r32, a.z32, a.part, ns, red, rz, rr);
            }
            continue;
        }
        if (k >= a.maxit) break;
        const double beta = (k == first) ? 0.0 : rz / rz_prev;
        const float betaT = (float)beta;
        // p_new = z + beta p_old of every row, then q = A p_new with p_new from LDS (from
        // global memory when the instance is too large for it)
        {
            struct In { float z[3], p[3]; };
            each_slice<WGS, In>(
                I,
                [&](In &x, int i) {
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        x.z[c] = a.z32[3 * i + c];
                        x.p[c] = pold[3 * i + c];
                    }
                },
                [&](const In &x, int sl, int i) {
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        const float u = fmaf(betaT, x.p[c], x.z[c]);
                        pnew[3 * i + c] = u;
                        if (staged) su[3 * (i - I.v0) + c] = u;
                    }
                });
        }
        __syncthreads();
        for (int sl = I.s0 + wave; sl < I.s1; sl += NW) {
            const int g = sl * SL + lane;
            const int row = a.srow[g], len = a.slen[g] - 1;   // the diagonal (last entry) is skipped
            const int base = a.slice_off[sl] + lane;
            const float mb = a.M32[row];
            const unsigned fm = a.fixmask[row];
            double y0, y1, y2;
            float ui0, ui1, ui2;
            auto rows = [&](auto get) {
                ui0 = get(row, 0); ui1 = get(row, 1); ui2 = get(row, 2);
                y0 = (double)(mb * ui0); y1 = (double)(mb * ui1); y2 = (double)(mb * ui2);
                row_spmv32(a.S32, nbs, a.scol, base, len, ui0, ui1, ui2, y0, y1, y2, get);
            };
            if (staged) rows([&](int j, int c) { return su[3 * (j - I.v0) + c]; });
            else rows([&](int j, int c) { return pnew[3 * j + c]; });
            if (fm & 1) y0 = 0.0;
            if (fm & 2) y1 = 0.0;
            if (fm & 4) y2 = 0.0;
            const float q0 = (float)y0, q1 = (float)y1, q2 = (float)y2;
            a.q32[3 * row] = q0; a.q32[3 * row + 1] = q1; a.q32[3 * row + 2] = q2;
            const double v[1] = {((double)ui0 * (double)q0 + (double)ui1 * (double)q1) + (double)ui2 * (double)q2};
            slice_partial<1>(v, sl, a.part, ns);
        }
        double pq[1];
        inst_sum<1>(pq, I, a.part, ns, red);
        if (!(pq[0] > 0.0)) {
            status = isfinite(pq[0]) ? EOLC_ERR_NOT_SPD : EOLC_ERR_NONFINITE;
            break;
        }
        const double alpha = rz / pq[0];
        const float alphaT = (float)alpha;
        // x += alpha p, r -= alpha q, z = D r
        {
            struct In { float p[3], q[3], r[3], x[3], d[ML ? 1 : 6]; };
            each_slice<WGS, In>(
                I,
                [&](In &x, int i) {
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        x.p[c] = pnew[3 * i + c];
                        x.q[c] = a.q32[3 * i + c];
                        x.r[c] = a.r32[3 * i + c];
                        x.x[c] = a.xl32[3 * i + c];
                    }
                    if constexpr (!ML)
#pragma unroll
                        for (int c = 0; c < 6; ++c) x.d[c] = a.D32[c * N + i];
                },
                [&](const In &x, int sl, int i) {
#pragma unroll
                    for (int c = 0; c < 3; ++c) a.xl32[3 * i + c] = fmaf(alphaT, x.p[c], x.x[c]);
                    const float r0 = fmaf(-alphaT, x.q[0], x.r[0]);
                    const float r1 = fmaf(-alphaT, x.q[1], x.r[1]);
                    const float r2 = fmaf(-alphaT, x.q[2], x.r[2]);
                    a.r32[3 * i] = r0; a.r32[3 * i + 1] = r1; a.r32[3 * i + 2] = r2;
                    if constexpr (ML) {
                        const double v[1] = {((double)r0 * (double)r0 + (double)r1 * (double)r1) + (double)r2 * (double)r2};
                        slice_partial<1>(v, sl, a.part, ns);
                    } else {
                        float z0, z1, z2;
                        eolc::apply_sym3<float>(x.d, 1, r0, r1, r2, z0, z1, z2);
                        a.z32[3 * i] = z0; a.z32[3 * i + 1] = z1; a.z32[3 * i + 2] = z2;
                        const double v[2] = {((double)r0 * (double)z0 + (double)r1 * (double)z1) + (double)r2 * (double)z2,
                                             ((double)r0 * (double)r0 + (double)r1 * (double)r1) + (double)r2 * (double)r2};
                        slice_partial<2>(v, sl, a.part, ns);
                    }
                });
        }
        rz_prev = rz;
        if constexpr (ML) {
            double s1[1];
            inst_sum<1>(s1, I, a.part, ns, red);
            rr = s1[0];
            rz = inst_ml_apply<WGS>(I, b, a.ml, N, a.D32, a.r32, a.z32, a.fixmask, a.part, ns, red);
        } else {
            double s2[2];
            inst_sum<2>(s2, I, a.part, ns, red);
            rz = s2[0];
            rr = s2[1];
        }
        float *t = pold;
        pold = pnew;
        pnew = t;
        ++k;
    }
    if (status != EOLC_OK && status != EOLC_ERR_NOT_SPD) {
        for (int sl = I.s0 + wave; sl < I.s1; sl += NW) {
            const int i = a.srow[sl * SL + lane];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                a.xs64[3 * i + c] += (double)a.xl32[3 * i + c];
                a.xl32[3 * i + c] = 0.0f;
            }
        }
    }
    // v = fixed ? vfix : x
    for (int sl = I.s0 + wave; sl < I.s1; sl += NW) {
        const int i = a.srow[sl * SL + lane];
        const unsigned fm = a.fixmask[i];
#pragma unroll
        for (int c = 0; c < 3; ++c) a.v[3 * i + c] = ((fm >> c) & 1) ? a.vfix[3 * i + c] : a.xs64[3 * i + c];
    }
    __syncthreads();
    const double true_rr = inst_residual64<WGS>(I, a.slice_off, a.srow, a.slen, a.scol, a.A64, nbs, a.fixmask, a.v,
                                                a.rhs, a.r64, a.part, ns, red);
    if (threadIdx.x == 0) {
        a.stats[4 * b + 0] = k;
        a.stats[4 * b + 1] = refinements;
        a.stats[4 * b + 2] = status;
        a.dstats[4 * b + 0] = bnorm2;
        a.dstats[4 * b + 1] = true_rr;
        a.dstats[4 * b + 2] = bnorm2 > 0.0 ? sqrt(rr / bnorm2) : 0.0;
    }
}

// Fixed values of the caller's fixed nodes (all three DOFs), Constraints.cpp:114-119:
// v_fixed = (1 - 0.01) v_old + scripted velocity.
__global__ void k_batch_vfix(int n, const int *__restrict__ nodes, const double *__restrict__ scripted,
                             const double *__restrict__ v, double *__restrict__ vfix)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 3 * n) return;
    const int i = nodes[t / 3], c = t % 3;
    vfix[3 * i + c] = (1 - 0.01) * v[3 * i + c] + scripted[t];
}

// All DOFs of the listed nodes fixed (set once per batch topology).
__global__ void k_batch_fixmask(int n, const int *__restrict__ nodes, unsigned char *__restrict__ fixmask)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) fixmask[nodes[t]] = 7;
}

// Rows whose direction fits the LDS of a compute unit beside the kernel's own few words;
// the launch asks for what its largest such instance needs, for every workgroup alike.  In a
// batch of more instances than compute units that leaves the smaller ones fewer workgroups
// on a unit, but the registers admit only one of 1,024 threads anyway (two of 512, four of
// 256), and the largest instance's chain of iterations counts for more.  Without LDS (the
// direction gathered, one entry at a time), with this rule, and with the staged rows limited
// to what leaves each unit its share of the instances, ms a step with 256, 512 and 1,024
// threads: 4,095 cloths of 20^2 quads and one of 115^2 185 117 80, 88 60 53, 99 68 53; 2,047
// of 40^2 and one of 115^2 234 164 121, 118 88 83, 148 112 84; 2,047 of 40^2 and one of 64^2
// 116 117 107, 88 87 76, 92 87 76; 600 of 8^2 to 96^2 180 122 89, 84 71 69, 97 81 69.
constexpr int kBatchStage = (160 * 1024 - 256) / 12;

template <int WGS>
hipError_t launch_batch(eolc_ctx *c, BatchArgs args, bool ml)
{
    const auto fn = ml ? k_batch_pcg<WGS, true> : k_batch_pcg<WGS, false>;
    args.stage = 0;
    for (const eolc::BatchInst &I : c->batch.inst)
        if (I.v1 - I.v0 <= kBatchStage) args.stage = std::max(args.stage, I.v1 - I.v0);
    const size_t lds = 12 * (size_t)args.stage;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(fn),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)(12 * kBatchStage));
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(fn, dim3(c->batch.B), dim3(WGS), lds, c->stream, args);
    return hipGetLastError();
}

}  // namespace

namespace eolc {

hipError_t batch_set_fixmask(eolc_ctx *c, const int *d_nodes, int n)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_batch_fixmask, dim3(blocks_for(n)), dim3(256), 0, c->stream, n, d_nodes, c->fixmask);
    return hipGetLastError();
}

// Enqueue the solve part of one batched step: fixed values, block-Jacobi blocks and
// the persistent PCG (all kernels, no host synchronisation: capturable).
hipError_t batch_solve_async(eolc_ctx *c, double tol, int maxit, int variant)
{
    BatchState &S = c->batch;
    const Topology &t = c->topo;
    const int nu = (int)S.user_fixed.size();
    if (nu > 0)
        hipLaunchKernelGGL(k_batch_vfix, dim3(blocks_for(3 * nu)), dim3(256), 0, c->stream, nu, S.d_user_fixed, S.d_scripted,
                           c->v, c->vfix);
    const bool ml = S.ml && S.d_ml_lo && c->ml.lv.L > 0;
    c->ml_on = ml;   // pcg_setup then also forms the coarse levels' blocks (translations only)
    hipError_t e = pcg_setup(c, true, 0, false);
    c->ml_on = false;
    if (e != hipSuccess) return e;
    BatchArgs a;
    a.inst = S.d_inst; a.order = S.d_order;
    a.slice_off = c->slice_off; a.srow = c->srow; a.slen = c->slen; a.scol = c->scol;
    a.A64 = c->A64; a.S32 = c->S32; a.M32 = c->M32; a.D32 = c->D32;
    a.nbs = t.nbs; a.N = t.N; a.nslices = t.nslices;
    a.fixmask = c->fixmask; a.vfix = c->vfix; a.rhs = c->rhs;
    a.v = c->v; a.xs64 = c->xs64; a.r64 = c->r64; a.b64 = c->b64;
    a.r32 = c->r32; a.z32 = c->z32; a.q32 = c->q32; a.xl32 = c->xl32; a.p32a = c->p32[0]; a.p32b = c->p32[1];
    a.part = S.slice_part;
    a.tol2 = tol * tol; a.delta2 = c->batch_delta * c->batch_delta; a.maxit = maxit;
    a.stats = S.stats; a.dstats = S.dstats;
    const MLState &m = c->ml;
    a.ml = BatchML{m.lv, m.hord, m.ptr1, m.agg1, m.par, m.cptr, S.d_ml_lo, m.Dinv, m.R, m.C};
    switch (variant) {
    case 0: return launch_batch<256>(c, a, ml);
    case 1: return launch_batch<512>(c, a, ml);
    default: return launch_batch<1024>(c, a, ml);
    }
}

}  // namespace eolc
