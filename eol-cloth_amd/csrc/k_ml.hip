// Additive multilevel preconditioner over an aggregation hierarchy (gfx950).
//
//   z = D0 r + sum_{l = 1..L} Z_l D_l^-1 Z_l^T r
//
// D0 holds the fine 3x3 blocks (block-Jacobi inverse, or the learned blocks).  Level
// l groups the vertices into nested aggregates (ml_host.cpp); Z_l is the piecewise-
// constant prolongation that copies one 3-vector per aggregate to its member
// vertices (zero on fixed DOFs), and D_l is the 3x3 diagonal block of the Galerkin
// operator Z_l^T A Z_l: the sum of all blocks A_ij, fixed DOFs masked, whose two
// vertices lie in the same level-l aggregate.  Each term is symmetric positive
// (semi-)definite for an SPD A, so z = P r defines an SPD preconditioner: an additive
// multilevel method of the BPX family (Bramble, Pasciak and Xu 1990) with
// aggregation coarse spaces.  The coarse terms carry the smooth, slowly converging
// modes (sheet-wide translations and bending) that no per-vertex block reaches.
//
// Set-up per matrix (ml_setup): k_ml_diag1 sums, per level-1 aggregate, the blocks
// of its member rows bucketed by the first level whose aggregate holds both vertices
// (`lam`, precomputed per SELL entry); k_ml_diagup adds children upwards.  Every
// level's blocks are inverted in FP64.
//
// Per PCG iteration, after the product (ml_apply):
//   k_ml_update   : on large meshes the vector update x += alpha p, r -= alpha q (on others
//                   the restriction updates r, the prolongation x)
//   k_ml_restrict : one wavefront per level-2 aggregate, vertices staged through LDS:
//                   R_1(a) = sum of r over a's members, R_2 = sum of the children's R_1,
//                   and per level-1 aggregate a, C(a) = D_1^-1 R_1(a) + D_2^-1 R_2(parent)
//   k_ml_coarse   : one workgroup (levels >= 3 only): R_l for l >= 3, then
//                   C_l = D_l^-1 R_l + C_{l+1}(parent) from the top level down to 3
//   k_ml_prolong  : z_i = D0 r_i + C(a_i) + C_3(level-3 aggregate of i); r.z partials
// All coarse arithmetic is FP64 in a fixed order, so the result does not depend on
// the launch shape.
//
// Linear coarse fields (single-cloth solves, levels >= kMLLinFrom = 3): there Z_l
// carries, per aggregate A and component, the basis phi = (1, (X - c_A) / s_A) of
// the material coordinates X (c_A the centroid, s_A the RMS radius of A's members),
// so a coarse correction is a field linear on each aggregate instead of a constant,
// and D_l is the 9 x 9 diagonal block of Z_l^T A Z_l, applied through the LDL^T
// factors of its unit-diagonal scaling, which leave out a basis function whose
// scaled pivot falls to 1e-10 (fact9_psd).  The smooth bending modes of a sheet are linear to
// first order over an aggregate; at 512^2 this cut the PCG iterations by a quarter
// (826 -> 617 at step 0, 890 -> 696 at step 6 of the benchmark trajectory).  The
// restriction forms the first moments sum (phi_1, phi_2) r of each level-2 aggregate,
// from which the coarse kernel gets every level >= 3 by the exact change of
// centroid and radius; the prolongation evaluates the level-3 field at each vertex.
// The batched solve keeps the translations on every level.
#include <algorithm>
#include <type_traits>

#include "eolc_internal.h"
#include "pcg_device.h"

using eolc::MLLevels;
using eolc::SolverScalars;

namespace {

constexpr int kML = eolc::kMLMaxLevels;

// Inverse of a symmetric 3x3 block (upper entries out).  A component whose diagonal
// is not positive (all of the aggregate's DOFs in it fixed) is left out: its row
// and column of the inverse are zero.  A block that is not positive definite on
// the remaining components gives a zero inverse (no correction from it).
__device__ __forceinline__ void inv_spd3(const double a[9], double *__restrict__ out)
{
    double s00 = a[0], s11 = a[4], s22 = a[8];
    double s01 = 0.5 * (a[1] + a[3]), s02 = 0.5 * (a[2] + a[6]), s12 = 0.5 * (a[5] + a[7]);
    const bool k0 = s00 > 0.0, k1 = s11 > 0.0, k2 = s22 > 0.0;
    if (!k0) { s00 = 1.0; s01 = 0.0; s02 = 0.0; }
    if (!k1) { s11 = 1.0; s01 = 0.0; s12 = 0.0; }
    if (!k2) { s22 = 1.0; s02 = 0.0; s12 = 0.0; }
    const double c00 = s11 * s22 - s12 * s12, c01 = s02 * s12 - s01 * s22, c02 = s01 * s12 - s02 * s11;
    const double m2 = s00 * s11 - s01 * s01;
    const double det = s00 * c00 + s01 * c01 + s02 * c02;
    double o[6] = {0, 0, 0, 0, 0, 0};
    if (s00 > 0.0 && m2 > 0.0 && det > 0.0 && isfinite(det)) {
        const double id = 1.0 / det;
        o[0] = c00 * id;
        o[1] = c01 * id;
        o[2] = c02 * id;
        o[3] = (s00 * s22 - s02 * s02) * id;
        o[4] = (s01 * s02 - s00 * s12) * id;
        o[5] = m2 * id;
        if (!k0) { o[0] = 0.0; o[1] = 0.0; o[2] = 0.0; }
        if (!k1) { o[1] = 0.0; o[3] = 0.0; o[4] = 0.0; }
        if (!k2) { o[2] = 0.0; o[4] = 0.0; o[5] = 0.0; }
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) out[k] = o[k];
}

__device__ __forceinline__ void apply_inv(const double *__restrict__ d, double r0, double r1, double r2, double &c0,
                                          double &c1, double &c2)
{
    c0 = fma(d[2], r2, fma(d[1], r1, d[0] * r0));
    c1 = fma(d[4], r2, fma(d[3], r1, d[1] * r0));
    c2 = fma(d[5], r2, fma(d[4], r1, d[2] * r0));
}

// The block of entry e with its fixed rows and columns zeroed (loads first: none waits on
// the masks).
__device__ __forceinline__ void masked9(const double *__restrict__ A, int64_t nbs, int64_t e, unsigned fi, unsigned fj,
                                        double (&b)[9])
{
#pragma unroll
    for (int c = 0; c < 9; ++c) b[c] = A[(int64_t)c * nbs + e];
#pragma unroll
    for (int c = 0; c < 9; ++c)
        if (((fi >> (c / 3)) | (fj >> (c % 3))) & 1u) b[c] = 0.0;
}

// V_1[m](a) = sum over level-1 aggregate a's member rows of the blocks (fixed DOFs masked)
// whose first common level is <= m + 1, m = 0..L-1; D_1^-1 from V_1[0].  An entry is a
// chain of dependent loads and an aggregate has about 12 rows of 13: kDiagLanes lanes to
// an aggregate, a row each, their sums added in a fixed tree.  With a thread to an
// aggregate 131 x 97 quads ran on four workgroups: 241 us,
// 30 now; 64 meshes of 32^2 to 96^2 quads 395 and 132; 512^2 quads 385 and 130.
constexpr int kDiagLanes = 16;
__global__ void __launch_bounds__(256) k_ml_diag1(MLLevels lv, const int *__restrict__ hord,
                                                  const int *__restrict__ ptr1, const int *__restrict__ gpos,
                                                  const int *__restrict__ slice_off, const int *__restrict__ slen,
                                                  const int *__restrict__ scol, const unsigned char *__restrict__ lam,
                                                  const double *__restrict__ A, int64_t nbs,
                                                  const unsigned char *__restrict__ fixmask, double *__restrict__ V,
                                                  double *__restrict__ Dinv)
{
    const int a = (int)(((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kDiagLanes);
    const int sub = threadIdx.x % kDiagLanes;
    const int n1 = lv.n[1], L = lv.L;
    if (a >= n1) return;   // all lanes of an aggregate together
    double acc[kML][9];
#pragma unroll
    for (int m = 0; m < kML; ++m)
#pragma unroll
        for (int c = 0; c < 9; ++c) acc[m][c] = 0.0;
    const int k1 = ptr1[a + 1];
    for (int k = ptr1[a] + sub; k < k1; k += kDiagLanes) {
        const int i = hord[k];
        const int g = gpos[i];
        const int len = slen[g];
        const int base = slice_off[g / eolc::kSlice] + (g % eolc::kSlice);
        const unsigned fi = fixmask[i];
        for (int kk = 0; kk < len; ++kk) {
            const int e = base + kk * eolc::kSlice;
            const int lm = lam[e];
            if (lm > L) continue;
            double b[9];
            masked9(A, nbs, e, fi, fixmask[scol[e]], b);
#pragma unroll
            for (int m = 0; m < kML; ++m)
                if (m < L && lm <= m + 1)
#pragma unroll
                    for (int c = 0; c < 9; ++c) acc[m][c] += b[c];
        }
    }
#pragma unroll
    for (int m = 0; m < kML; ++m)
        if (m < L)
#pragma unroll
            for (int c = 0; c < 9; ++c) {
                double v = acc[m][c];
#pragma unroll
                for (int o = kDiagLanes / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kDiagLanes);
                acc[m][c] = v;
                if (sub == (9 * m + c) % kDiagLanes) V[(int64_t)(m * 9 + c) * n1 + a] = v;
            }
    if (sub == 0) inv_spd3(acc[0], Dinv + 6 * (int64_t)a);
}

// One wavefront per level-l aggregate (l >= 2), a lane per sum: V_l[m] = sum of the
// children's V_{l-1}[m] for m >= l - 1; D_l^-1 from V_l[l - 1].  (One thread per aggregate
// ran a few of them at a time through every sum: 82 us for
// the three levels of 131 x 97 quads, 14 now.)
__global__ void __launch_bounds__(64) k_ml_diagup(int l, MLLevels lv, const int *__restrict__ cptr,
                                                  double *__restrict__ V, double *__restrict__ Dinv)
{
    __shared__ double d[9];
    const int A = blockIdx.x;
    const int L = lv.L, nl = lv.n[l], nc = lv.n[l - 1];
    const double *__restrict__ Vc = V + (int64_t)9 * L * lv.off[l - 1];
    double *__restrict__ Vl = V + (int64_t)9 * L * lv.off[l];
    const int c0 = cptr[lv.coff[l] + A], c1 = cptr[lv.coff[l] + A + 1];
    for (int t = 9 * (l - 1) + (int)threadIdx.x; t < 9 * L; t += 64) {
        double s = 0.0;
#pragma unroll 4
        for (int a = c0; a < c1; ++a) s += Vc[(int64_t)t * nc + a];
        Vl[(int64_t)t * nl + A] = s;
        if (t < 9 * l) d[t - 9 * (l - 1)] = s;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double v[9];
#pragma unroll
        for (int c = 0; c < 9; ++c) v[c] = d[c];
        inv_spd3(v, Dinv + 6 * (int64_t)(lv.off[l] + A));
    }
}

// Upper triangle of a symmetric 9 x 9 block, row by row: 45 entries.
__device__ __forceinline__ constexpr int pk9(int p, int q) { return p * 9 - p * (p - 1) / 2 + (q - p); }
// Strictly lower triangle of a 9 x 9 factor, row by row: 36 entries.
__device__ __forceinline__ constexpr int lo9(int i, int j) { return i * (i - 1) / 2 + j; }

constexpr double kPivotTol = 1e-10;
constexpr int kFact9 = 54;   // per aggregate: 36 factor entries, 9 inverse pivots, 9 scales

// Factorisation of a symmetric positive semi-definite 9 x 9 block G (packed) for
// applying its inverse: with the scales s_p = G_pp^-1/2 the scaled block s G s has
// a unit diagonal; LDL^T of it in index order leaves out a basis function whose
// pivot is at or below kPivotTol (its share of the block not spanned by the earlier
// ones), or whose diagonal is not positive, and inverts the rest.  Stored: the unit
// lower factor (its columns of left-out functions zero), 1/d (0 when left out) and
// s.  The scaling keeps a block whose stretch modes are 1e10 times stiffer than its
// translations (a collapsed element inside the aggregate) from losing the
// translations, and applying the factors keeps the operator positive where an
// explicit inverse of such a block would not be.  The factors go out with stride `ld`,
// so that the coarse kernel, one aggregate per thread, reads them coalesced.
__device__ void fact9_psd(const double *__restrict__ G, double *__restrict__ F, int ld)
{
    double Lm[9][9], d[9], sc[9];
    bool kept[9];
    for (int p = 0; p < 9; ++p) {
        const double g = G[pk9(p, p)];
        sc[p] = (g > 0.0 && isfinite(g)) ? 1.0 / sqrt(g) : 0.0;
    }
    for (int k = 0; k < 9; ++k) {
        double dk = sc[k] * sc[k] * G[pk9(k, k)];
        for (int j = 0; j < k; ++j)
            if (kept[j]) dk -= Lm[k][j] * Lm[k][j] * d[j];
        kept[k] = sc[k] > 0.0 && dk > kPivotTol && isfinite(dk);
        for (int i = 0; i < 9; ++i) Lm[i][k] = 0.0;
        d[k] = 0.0;
        if (!kept[k]) continue;
        d[k] = dk;
        for (int i = k + 1; i < 9; ++i) {
            double v = sc[k] * sc[i] * G[pk9(k, i)];
            for (int j = 0; j < k; ++j)
                if (kept[j]) v -= Lm[i][j] * Lm[k][j] * d[j];
            Lm[i][k] = v / dk;
        }
    }
    for (int i = 1; i < 9; ++i)
        for (int j = 0; j < i; ++j) F[(int64_t)lo9(i, j) * ld] = Lm[i][j];
    for (int p = 0; p < 9; ++p) {
        F[(int64_t)(36 + p) * ld] = kept[p] ? 1.0 / d[p] : 0.0;
        F[(int64_t)(45 + p) * ld] = sc[p];
    }
}

// out = G^+ r from fact9_psd's factors (here one after the other): s L^-T D^-1 L^-1 s r.
__device__ __forceinline__ void apply9(const double *__restrict__ F, const double *r, double *out)
{
    double y[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        double v = F[45 + i] * r[i];
#pragma unroll
        for (int j = 0; j < i; ++j) v = fma(-F[lo9(i, j)], y[j], v);
        y[i] = v;
    }
#pragma unroll
    for (int i = 0; i < 9; ++i) y[i] *= F[36 + i];
#pragma unroll
    for (int i = 8; i >= 0; --i) {
        double v = y[i];
#pragma unroll
        for (int j = i + 1; j < 9; ++j) v = fma(-F[lo9(j, i)], y[j], v);
        y[i] = v;
    }
#pragma unroll
    for (int i = 0; i < 9; ++i) out[i] = F[45 + i] * y[i];
}

// One workgroup per set-up chunk (level l, aggregate g, hord positions [k0, k1)):
// sum over the chunk's rows i and their entries (i, j) inside g (first common level
// <= l) of phi(i) phi(j)^T (x) A_ij, fixed DOFs masked, in the aggregate's basis;
// the upper triangle (45 sums) in a fixed order per thread, then over the workgroup.
// 131 x 97 quads: 177 us in chunks of 2,048 rows, 37 in chunks of 256.
constexpr int kGalWG = 256;
__global__ void __launch_bounds__(kGalWG) k_ml_gal9_part(const int *__restrict__ gchunk, const int *__restrict__ hord,
                                                         const int *__restrict__ gpos,
                                                         const int *__restrict__ slice_off,
                                                         const int *__restrict__ slen, const int *__restrict__ scol,
                                                         const unsigned char *__restrict__ lam,
                                                         const double *__restrict__ A, int64_t nbs,
                                                         const unsigned char *__restrict__ fixmask,
                                                         const double *__restrict__ X, const double *__restrict__ geo,
                                                         double *__restrict__ gpart)
{
    __shared__ double red[kGalWG / 64][45];
    const int ch = blockIdx.x;
    const int l = gchunk[4 * ch], g = gchunk[4 * ch + 1], k0 = gchunk[4 * ch + 2], k1 = gchunk[4 * ch + 3];
    const double cu = geo[4 * (int64_t)g], cv = geo[4 * (int64_t)g + 1], is = geo[4 * (int64_t)g + 3];
    double acc[45];
#pragma unroll
    for (int p = 0; p < 45; ++p) acc[p] = 0.0;
    for (int k = k0 + (int)threadIdx.x; k < k1; k += kGalWG) {
        const int i = hord[k];
        const int gp = gpos[i];
        const int len = slen[gp];
        const int base = slice_off[gp / eolc::kSlice] + (gp % eolc::kSlice);
        const unsigned fi = fixmask[i];
        const double pi[3] = {1.0, (X[2 * (int64_t)i] - cu) * is, (X[2 * (int64_t)i + 1] - cv) * is};
        for (int kk = 0; kk < len; ++kk) {
            const int e = base + kk * eolc::kSlice;
            if ((int)lam[e] > l) continue;
            const int j = scol[e];
            const unsigned fj = fixmask[j];
            const double pj[3] = {1.0, (X[2 * (int64_t)j] - cu) * is, (X[2 * (int64_t)j + 1] - cv) * is};
            double b[9];
            masked9(A, nbs, e, fi, fj, b);
#pragma unroll
            for (int p = 0; p < 9; ++p)
#pragma unroll
                for (int q = p; q < 9; ++q) acc[pk9(p, q)] = fma(pi[p / 3] * pj[q / 3], b[(p % 3) * 3 + q % 3], acc[pk9(p, q)]);
        }
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int p = 0; p < 45; ++p) {
        const double v = wave_sum(acc[p]);
        if (lane == 0) red[wid][p] = v;
    }
    __syncthreads();
    if (threadIdx.x < 45) {
        double v = 0.0;
#pragma unroll
        for (int w = 0; w < kGalWG / 64; ++w) v += red[w][threadIdx.x];
        gpart[45 * (int64_t)ch + threadIdx.x] = v;
    }
}

// One wavefront per aggregate of levels >= 3: its chunks' sums in order, a lane per
// value, then the block's factors.
__global__ void __launch_bounds__(64) k_ml_gal9_fin(int n_hi, const int *__restrict__ gcp,
                                                    const double *__restrict__ gpart, double *__restrict__ D9)
{
    __shared__ double sG[45];
    const int h = blockIdx.x, p = threadIdx.x;
    if (p < 45) {
        const int c1 = gcp[h + 1];
        double v = 0.0;
#pragma unroll 8
        for (int ch = gcp[h]; ch < c1; ++ch) v += gpart[45 * (int64_t)ch + p];
        sG[p] = v;
    }
    __syncthreads();
    if (p == 0) fact9_psd(sG, D9 + h, n_hi);
}

// Ordering of LDS traffic between the lanes of one wavefront (no workgroup barrier:
// the wavefronts of a workgroup run different trip counts).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Restriction of r to levels 1 and 2: one wavefront per level-2 aggregate.  Its
// vertices are a contiguous range of hord; the lanes stage up to kStageRows of them in
// LDS, four per lane with the loads of all four together, then each lane sums the
// members of one level-1 child that fall in the stage, in member order.  R_2 is the
// wavefront sum of the children's R_1 (fixed shuffle tree).  With a single level, a
// wavefront takes 64 level-1 aggregates.
// two wavefronts per workgroup: 13.9 us per restriction at 1024^2, against 14.8 (1),
// 14.2 (4) and 14.4 (8) in the same kernel trace
constexpr int kRestrictWG = 128;
constexpr int kStageRows = 256;

// The PCG's residual update r -= alpha q, done by the restriction as it reads r (UPD): the
// residual is written once and read once, and a launch is saved.  The members of an
// aggregate are a compact patch of the sheet, so their scattered pieces share most cache
// lines; still they cost more than a pass in row order does, and far more on a renumbered
// mesh, so x += alpha p is left to the prolongation, which goes over the rows in order
// (restriction + prolongation, us, before and now: 22,000 remeshed
// vertices in FP64 24.6 + 6.7 and 18.1 + 7.0, 1024^2 mixed 50.5 + 19.0 and 38.3 + 29.6, 512^2
// 20.0 + 6.9 and 16.9 + 10.0; a renumbered 700^2 step 158 and 129 ms).
template <class T> struct VecUpdate {
    const T *q;
    T *r;
    T alpha;
};

__device__ __forceinline__ void lift9(const double *__restrict__ q, double al, double bu, double bv, double *sm)
{
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        sm[a] += q[a];
        sm[3 + a] += fma(al, q[3 + a], bu * q[a]);
        sm[6 + a] += fma(al, q[6 + a], bv * q[a]);
    }
}
__device__ __forceinline__ void lower9(const double *__restrict__ P, double al, double bu, double bv, double *cf)
{
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        cf[a] += fma(bv, P[6 + a], fma(bu, P[3 + a], P[a]));
        cf[3 + a] = fma(al, P[3 + a], cf[3 + a]);
        cf[6 + a] = fma(al, P[6 + a], cf[6 + a]);
    }
}

// The restriction of one level-2 aggregate w by one wavefront (two levels or more),
// or of the 64 level-1 aggregates from w * 64 (one level).  Writes R_1 of its
// children, R_2(w) and C of its children; returns R_2(w) in every lane and, with
// feat2 (the members' level-2 coordinate features in hord order), the first moments
// sum phi_1 r and sum phi_2 r in lane 0.  srr += r.r of the lane's members.
template <class T, bool LIN, bool UPD>
__device__ __forceinline__ void restrict_wave(const MLLevels &lv, int w, const int *__restrict__ hord,
                                              const int *__restrict__ ptr1, const int *__restrict__ cptr,
                                              const int *__restrict__ kptr2, const VecUpdate<T> &up,
                                              double *__restrict__ R, const double *__restrict__ Dinv,
                                              double *__restrict__ C, const double *__restrict__ feat2,
                                              double *__restrict__ buf, double &s0, double &s1, double &s2,
                                              double (&mom)[6], double &srr)
{
    constexpr int NC = kStageRows / 64;
    const int lane = threadIdx.x % 64;
    const bool two = lv.L >= 2;
    int a0, a1, ka = 0, kz = 0;
    if (two) {
        a0 = cptr[lv.coff[2] + w];
        a1 = cptr[lv.coff[2] + w + 1];
        ka = kptr2[w];
        kz = kptr2[w + 1];
    } else {
        a0 = w * 64;
        a1 = min(a0 + 64, lv.n[1]);
    }
    s0 = s1 = s2 = 0.0;
    double f0 = 0.0, f1 = 0.0, f2 = 0.0;   // R_1 of this lane's first child
    double mu0 = 0.0, mu1 = 0.0, mu2 = 0.0, mv0 = 0.0, mv1 = 0.0, mv2 = 0.0;
    int k0 = two ? ka : ptr1[a0];
    for (int g0 = a0; g0 < a1; g0 += 64) {   // groups of up to 64 children
        const int g1 = min(g0 + 64, a1);
        const int a = g0 + lane;
        const bool mine = a < g1;
        const int m0 = mine ? ptr1[a] : 0, m1 = mine ? ptr1[a + 1] : 0;
        const int k1 = (two && g1 == a1) ? kz : ptr1[g1];
        double t0 = 0.0, t1 = 0.0, t2 = 0.0;
        for (int kb = k0; kb < k1; kb += kStageRows) {
            int i[NC];
            double u[NC], v[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const int k = kb + 64 * c + lane;
                if (k < k1) {
                    i[c] = hord[k];
                    if (LIN) {
                        u[c] = feat2[2 * (int64_t)k];
                        v[c] = feat2[2 * (int64_t)k + 1];
                    }
                }
            }
            // (the compiler otherwise issues the features' loads after the gathers below)
            if (LIN) asm volatile("" ::: "memory");
            T qv[NC][3], rv[NC][3];
#pragma unroll
            for (int c = 0; c < NC; ++c)
                if (kb + 64 * c + lane < k1)
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        const int64_t j = 3 * (int64_t)i[c] + d;
                        rv[c][d] = up.r[j];
                        if (UPD) qv[c][d] = up.q[j];
                    }
#pragma unroll
            for (int c = 0; c < NC; ++c)
                if (kb + 64 * c + lane < k1) {
                    double q[3];
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        if (UPD) {
                            const int64_t j = 3 * (int64_t)i[c] + d;
                            rv[c][d] = fma(-up.alpha, qv[c][d], rv[c][d]);
                            up.r[j] = rv[c][d];
                        }
                        q[d] = (double)rv[c][d];
                        srr += q[d] * q[d];
                        buf[3 * (64 * c + lane) + d] = q[d];
                    }
                    if (LIN) {
                        mu0 = fma(u[c], q[0], mu0); mu1 = fma(u[c], q[1], mu1); mu2 = fma(u[c], q[2], mu2);
                        mv0 = fma(v[c], q[0], mv0); mv1 = fma(v[c], q[1], mv1); mv2 = fma(v[c], q[2], mv2);
                    }
                }
            wave_sync();
            const int e0 = max(m0, kb), e1 = min(m1, kb + kStageRows);
            for (int m = e0; m < e1; ++m) {
                t0 += buf[3 * (m - kb)];
                t1 += buf[3 * (m - kb) + 1];
                t2 += buf[3 * (m - kb) + 2];
            }
            wave_sync();
        }
        if (mine) {
            R[3 * a] = t0; R[3 * a + 1] = t1; R[3 * a + 2] = t2;
            s0 += t0; s1 += t1; s2 += t2;
            if (g0 == a0) { f0 = t0; f1 = t1; f2 = t2; }
        }
        k0 = k1;   // the next group starts where this one ends
    }
    if (!two) return;
    // inverse blocks of the level-2 aggregate and of this lane's first child
    double dw[6], da[6] = {0, 0, 0, 0, 0, 0};
    {
        const int64_t gw = lv.off[2] + w;
#pragma unroll
        for (int k = 0; k < 6; ++k) dw[k] = Dinv[6 * gw + k];
        if (a0 + lane < a1)
#pragma unroll
            for (int k = 0; k < 6; ++k) da[k] = Dinv[6 * (int64_t)(a0 + lane) + k];
    }
    // wave_sum leaves the total in lane 0; every lane needs it below
    s0 = __shfl(wave_sum(s0), 0, 64);
    s1 = __shfl(wave_sum(s1), 0, 64);
    s2 = __shfl(wave_sum(s2), 0, 64);
    if (lane == 0) {
        double *o = R + 3 * (lv.off[2] + (int64_t)w);
        o[0] = s0; o[1] = s1; o[2] = s2;
    }
    if (LIN) {
        mom[0] = wave_sum(mu0); mom[1] = wave_sum(mu1); mom[2] = wave_sum(mu2);
        mom[3] = wave_sum(mv0); mom[4] = wave_sum(mv1); mom[5] = wave_sum(mv2);
    }
    // levels 1 and 2 of each child, for the prolongation: C(a) = D_1^-1 R_1(a) +
    // D_2^-1 R_2(w)
    double e0, e1, e2, c0, c1, c2;
    apply_inv(dw, s0, s1, s2, e0, e1, e2);
    if (a0 + lane < a1) {
        const int64_t a = a0 + lane;
        apply_inv(da, f0, f1, f2, c0, c1, c2);
        C[3 * a] = c0 + e0; C[3 * a + 1] = c1 + e1; C[3 * a + 2] = c2 + e2;
    }
    // more than 64 children: each lane re-reads the R_1 it wrote above
    for (int g0 = a0 + 64; g0 < a1; g0 += 64) {
        const int a = g0 + lane;
        if (a < a1) {
            apply_inv(Dinv + 6 * (int64_t)a, R[3 * a], R[3 * a + 1], R[3 * a + 2], c0, c1, c2);
            C[3 * a] = c0 + e0; C[3 * a + 1] = c1 + e1; C[3 * a + 2] = c2 + e2;
        }
    }
}

// What the two restriction kernels share.  In an iteration (UPD) alpha = r.z / p.q from
// the partials of the product (Ga) and of the prolongation (Gz), left in the scalars for
// the prolongation, and the stop on p.q <= 0.  Every workgroup leaves its r.r in PB[parity].
struct RestrictArgs {
    MLLevels lv;
    const int *hord, *ptr1, *cptr, *kptr2;
    double *R, *C;
    const double *Dinv, *feat2, *geo;
    double *R9p;
    SolverScalars *scal;
    double *partials;
    int k, Ga, Gz;        // iteration and partial counts (the vector update)
    int parity;
    bool check;           // no-op once the solve has stopped
};

// alpha of the iteration; false: the solve stops here (the flag is set by workgroup 0).
template <class T, int W>
__device__ __forceinline__ bool restrict_alpha(const RestrictArgs &g, VecUpdate<T> &up, double &alpha, double *lds)
{
    double v[2];
    reduce_partials<2, W>({PA(g.partials), PB(g.partials, g.k & 1)}, {g.Ga, g.Gz}, v, lds);
    const double pq = v[0], rz = v[1];
    SolverScalars *scal = g.scal;
    if (!(pq > 0.0)) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            scal->done = 1;
            scal->reason = isfinite(pq) ? 2 : 4;
            scal->pq = pq;
        }
        return false;
    }
    alpha = rz / pq;
    up.alpha = (T)alpha;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        scal->iters = g.k + 1;
        scal->pq = pq;
        scal->alpha = alpha;
    }
    return true;
}

// The vector update of a large mesh on its own (ml_update_apart), x += alpha p and r -=
// alpha q over the flat arrays: four consecutive values a thread, 16 bytes a load (two for
// FP64), bound by the bytes.
template <class T>
__global__ void __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(8, 8)))
k_ml_update(RestrictArgs g, VecUpdate<T> up, int n3, const T *__restrict__ p, double *__restrict__ x)
{
    typedef T v4 __attribute__((ext_vector_type(4)));
    typedef double x4 __attribute__((ext_vector_type(4)));
    __shared__ double lds[2 * (WG / 64) + 2];
    if (g.scal->done) return;
    const int G = gridDim.x, chunk = (((n3 + G - 1) / G) + 3) & ~3;
    const int b = min(logical_wg() * chunk, n3), e = min(b + chunk, n3), i0 = b + 4 * (int)threadIdx.x;
    // mixed precision: the first trip's x (half the bytes read) loads before the partial
    // sums are reduced; more would spill at eight waves per SIMD
    constexpr bool PRE = sizeof(T) == 4;
    x4 xv0 = {};
    if (PRE && i0 + 3 < e) xv0 = *reinterpret_cast<const x4 *>(x + i0);
    double alpha;
    if (!restrict_alpha<T, WG>(g, up, alpha, lds)) return;
    for (int i = i0; i < e; i += 4 * WG) {
        if (i + 3 < e) {   // i is a multiple of 4: aligned vectors
            const v4 pv = *reinterpret_cast<const v4 *>(p + i), qv = *reinterpret_cast<const v4 *>(up.q + i);
            const v4 rv = *reinterpret_cast<const v4 *>(up.r + i);
            const x4 xv = (PRE && i == i0) ? xv0 : *reinterpret_cast<const x4 *>(x + i);
            x4 xo;
            v4 ro;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                xo[c] = fma(alpha, (double)pv[c], xv[c]);
                ro[c] = fma(-up.alpha, qv[c], rv[c]);
            }
            *reinterpret_cast<x4 *>(x + i) = xo;
            *reinterpret_cast<v4 *>(up.r + i) = ro;
        } else {
            for (int c = i; c < e; ++c) {
                x[c] = fma(alpha, (double)p[c], x[c]);
                up.r[c] = fma(-up.alpha, up.q[c], up.r[c]);
            }
        }
    }
}

// Translations only: one wavefront per level-2 aggregate (or per 64 level-1 ones), on at
// most kRestrictGrid workgroups (every workgroup of the next product sums their r.r).
constexpr int kRestrictGrid = 4096;
template <class T, bool UPD>
__global__ void __launch_bounds__(kRestrictWG) k_ml_restrict(RestrictArgs g, VecUpdate<T> up)
{
    constexpr int NW = kRestrictWG / 64;
    __shared__ double stage[NW][3 * kStageRows];
    __shared__ double lds[2 * NW + 2];
    if (g.check && g.scal->done) return;
    double alpha;
    if (UPD && !restrict_alpha<T, kRestrictWG>(g, up, alpha, lds)) return;
    double s0, s1, s2, mom[6], srr[1] = {0.0};
    const int waves = g.lv.L >= 2 ? g.lv.n[2] : (g.lv.n[1] + 63) / 64;
    for (int w = logical_wg() * NW + (int)threadIdx.x / 64; w < waves; w += gridDim.x * NW)   // uniform
        restrict_wave<T, false, UPD>(g.lv, w, g.hord, g.ptr1, g.cptr, g.kptr2, up, g.R, g.Dinv, g.C, nullptr,
                                     stage[threadIdx.x / 64], s0, s1, s2, mom, srr[0]);
    write_partials<1, kRestrictWG>(srr, PB(g.partials, g.parity) + eolc::kMaxPartials, lds);
}

// Linear coarse fields: kRestrict3Parts workgroups per level-3 aggregate U, whose
// kRestrict3Parts x (kRestrict3WG / 64) wavefronts take U's level-2 children in turn
// (wavefront g of U takes children c0 + g, c0 + g + 16, ...).  Each child's R_2 and
// first moments are re-expressed on U's basis, (R_2, alpha M_1 + beta_u R_2, alpha
// M_2 + beta_v R_2) with alpha = s_w / s_U and beta = (c_w - c_U) / s_U, summed per
// wavefront in child order and over the workgroup's wavefronts in order: one partial
// R9 per workgroup, which the coarse kernel adds in order.  With the residual update, FP32
// (us): 131 x 97 quads 8.7, 512^2 16.9, 1024^2 38.3.  There it is bound by the scattered
// pieces and its chain of dependent rounds (59 MB of vectors): slower without the
// workgroups in XCD order, the same with 128 or 256 members staged at once and with four
// wavefronts per SIMD instead of three; with eight parts to an aggregate it takes 15.0 at
// 512^2 but 47.7 at 1024^2, and the coarse kernel twice as long.
constexpr int kRestrict3WG = 256;
using eolc::kRestrict3Parts;
template <class T, bool UPD>
__global__ void __launch_bounds__(kRestrict3WG) k_ml_restrict3(RestrictArgs g, VecUpdate<T> up)
{
    constexpr int NW = kRestrict3WG / 64;
    __shared__ double stage[NW][3 * kStageRows];
    __shared__ double red[NW][9];
    __shared__ double lds[2 * NW + 2];
    const MLLevels &lv = g.lv;
    // consecutive aggregates on one XCD: neighbouring patches share cache lines of the
    // vectors (the grid is padded to a multiple of 8; a workgroup without one only
    // leaves its empty r.r)
    const int lw = logical_wg();
    const int U = min(lw / kRestrict3Parts, lv.n[3] - 1), part = lw % kRestrict3Parts;
    const bool own = lw < lv.n[3] * kRestrict3Parts;
    const int lane = threadIdx.x % 64, wid = threadIdx.x / 64;
    const int c0 = g.cptr[lv.coff[3] + U], c1 = own ? g.cptr[lv.coff[3] + U + 1] : 0;
    const int64_t gU = lv.off[3] + U;
    const double cu = g.geo[4 * gU], cv = g.geo[4 * gU + 1], is = g.geo[4 * gU + 3];
    if (g.check && g.scal->done) return;
    double alpha;
    if (UPD && !restrict_alpha<T, kRestrict3WG>(g, up, alpha, lds)) return;
    // lane 0 keeps the wavefront's running sum in LDS
    if (lane == 0)
#pragma unroll
        for (int q = 0; q < 9; ++q) red[wid][q] = 0.0;
    double srr[1] = {0.0};
    for (int w = c0 + part * NW + wid; w < c1; w += NW * kRestrict3Parts) {
        double s0, s1, s2, mom[6];
        restrict_wave<T, true, UPD>(lv, w, g.hord, g.ptr1, g.cptr, g.kptr2, up, g.R, g.Dinv, g.C, g.feat2, stage[wid],
                                    s0, s1, s2, mom, srr[0]);
        if (lane == 0) {
            const int64_t gw = lv.off[2] + w;
            const double al = g.geo[4 * gw + 2] * is, bu = (g.geo[4 * gw] - cu) * is, bv = (g.geo[4 * gw + 1] - cv) * is;
            double t[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
            const double q[9] = {s0, s1, s2, mom[0], mom[1], mom[2], mom[3], mom[4], mom[5]};
            lift9(q, al, bu, bv, t);
#pragma unroll
            for (int k = 0; k < 9; ++k) red[wid][k] += t[k];
        }
    }
    __syncthreads();
    if (own && threadIdx.x < 9) {
        double v = 0.0;
#pragma unroll
        for (int k = 0; k < NW; ++k) v += red[k][threadIdx.x];
        g.R9p[(int64_t)threadIdx.x * (kRestrict3Parts * lv.n[3]) + lw] = v;
    }
    write_partials<1, kRestrict3WG>(srr, PB(g.partials, g.parity) + eolc::kMaxPartials, lds, lw);
}

// Levels >= 3 in one workgroup: R_l from the children (l = 3..L), then from the top
// down C_l = D_l^-1 R_l + C_{l+1}(parent) (l = L..3).  These levels hold a few hundred
// aggregates for a million vertices: up to kCoarseWG, each thread owns one, their R and C
// live in LDS and only C_3 is written out.  Larger hierarchies loop over global memory.
constexpr int kCoarseWG = 1024;

// The levels >= 3, at most one aggregate to a thread of the workgroup: C_l of aggregate
// off[3] + j in Cl[3 j ..], visible to all; false: the solve has stopped.
__device__ __forceinline__ bool coarse_levels(const MLLevels &lv, const int *__restrict__ cptr,
                                              const int *__restrict__ par, const double *__restrict__ Dinv,
                                              const double *__restrict__ R, const SolverScalars *scal, int check_done,
                                              double *__restrict__ Rl, double *__restrict__ Cl)
{
    // one aggregate per thread: its inverse block, parent and child range are
    // loaded up front (with level 3's children sums), then every phase runs in LDS
    const int L = lv.L, base = lv.off[3], M = lv.off[L + 1] - base;
    const int j = threadIdx.x;
    int l = 0, pa = 0, c0 = 0, c1 = 0, offm1 = 0, offp1 = 0;
    double d[6] = {0, 0, 0, 0, 0, 0};
    if (j < M) {
        // the level and its neighbours' offsets from constant indices into the
        // arguments (scalar loads; a variable index costs a vector load per use)
        l = 3;
        int offl = lv.off[3], coffl = lv.coff[3];
        offm1 = lv.off[2];
        offp1 = lv.off[4];
#pragma unroll
        for (int k = 4; k <= eolc::kMLMaxLevels; ++k)
            if (k <= L && j >= lv.off[k] - base) {   // offsets increase with the level
                l = k;
                offl = lv.off[k];
                coffl = lv.coff[k];
                offm1 = lv.off[k - 1];
                offp1 = lv.off[k + 1];
            }
        const int a = j - (offl - base);
        const int64_t g = base + j;
#pragma unroll
        for (int k = 0; k < 6; ++k) d[k] = Dinv[6 * g + k];
        if (l < L) pa = par[g];
        c0 = cptr[coffl + a];
        c1 = cptr[coffl + a + 1];
    }
    // the stop flag is read with the first loads (uniform: every thread leaves
    // before the first barrier, or none does)
    if (check_done && scal->done) return false;
    if (j < M) {
        if (l == 3) {
            const double *src = R + 3 * (int64_t)lv.off[2];
            double s0 = 0.0, s1 = 0.0, s2 = 0.0;
            for (int b = c0; b < c1; b += 8) {   // children in order, 8 loads in flight
                double v[8][3];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const bool ok = b + u < c1;
                    const double *q = src + 3 * (ok ? b + u : c0);
                    v[u][0] = ok ? q[0] : 0.0;
                    v[u][1] = ok ? q[1] : 0.0;
                    v[u][2] = ok ? q[2] : 0.0;
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    s0 += v[u][0]; s1 += v[u][1]; s2 += v[u][2];
                }
            }
            Rl[3 * j] = s0; Rl[3 * j + 1] = s1; Rl[3 * j + 2] = s2;
        }
    }
    __syncthreads();
    for (int lev = 4; lev <= L; ++lev) {
        if (j < M && l == lev) {
            const int cb = offm1 - base;   // level lev - 1
            double s0 = 0.0, s1 = 0.0, s2 = 0.0;
            for (int b = c0; b < c1; ++b) {
                s0 += Rl[3 * (cb + b)]; s1 += Rl[3 * (cb + b) + 1]; s2 += Rl[3 * (cb + b) + 2];
            }
            Rl[3 * j] = s0; Rl[3 * j + 1] = s1; Rl[3 * j + 2] = s2;
        }
        __syncthreads();
    }
    for (int lev = L; lev >= 3; --lev) {
        if (j < M && l == lev) {
            double e0, e1, e2;
            apply_inv(d, Rl[3 * j], Rl[3 * j + 1], Rl[3 * j + 2], e0, e1, e2);
            if (lev < L) {
                const int up = offp1 - base + pa;   // the parent on level lev + 1
                e0 += Cl[3 * up]; e1 += Cl[3 * up + 1]; e2 += Cl[3 * up + 2];
            }
            Cl[3 * j] = e0; Cl[3 * j + 1] = e1; Cl[3 * j + 2] = e2;
        }
        __syncthreads();
    }
    return true;
}

__global__ void __launch_bounds__(kCoarseWG) k_ml_coarse(MLLevels lv, const int *__restrict__ cptr,
                                                         const int *__restrict__ par, const double *__restrict__ Dinv,
                                                         double *__restrict__ R, double *__restrict__ C,
                                                         const SolverScalars *scal, int check_done)
{
    __shared__ double lds[6 * kCoarseWG];
    const int L = lv.L;
    const int base = lv.off[3];
    const int M = lv.off[L + 1] - base;   // aggregates of levels >= 3
    if (M <= kCoarseWG) {
        double *Cl = lds + 3 * kCoarseWG;
        if (!coarse_levels(lv, cptr, par, Dinv, R, scal, check_done, lds, Cl)) return;
        for (int t = threadIdx.x; t < 3 * lv.n[3]; t += kCoarseWG) C[3 * (int64_t)base + t] = Cl[t];
        return;
    }
    if (check_done && scal->done) return;
    double *Rb = R + 3 * (int64_t)base, *Cb = C + 3 * (int64_t)base;   // level l at off[l] - off[3]
    for (int l = 3; l <= L; ++l) {
        for (int A = threadIdx.x; A < lv.n[l]; A += kCoarseWG) {
            const int c0 = cptr[lv.coff[l] + A], c1 = cptr[lv.coff[l] + A + 1];
            const double *src = (l == 3) ? R + 3 * (int64_t)lv.off[2] : Rb + 3 * (lv.off[l - 1] - base);
            double s0 = 0.0, s1 = 0.0, s2 = 0.0;
            // children in order; the loads of 8 children are issued before their sums
            // (a missing child adds an exact 0)
            for (int a = c0; a < c1; a += 8) {
                double v[8][3];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const bool ok = a + u < c1;
                    const double *q = src + 3 * (ok ? a + u : c0);
                    v[u][0] = ok ? q[0] : 0.0;
                    v[u][1] = ok ? q[1] : 0.0;
                    v[u][2] = ok ? q[2] : 0.0;
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    s0 += v[u][0]; s1 += v[u][1]; s2 += v[u][2];
                }
            }
            double *o = Rb + 3 * (lv.off[l] - base + A);
            o[0] = s0; o[1] = s1; o[2] = s2;
        }
        __syncthreads();
    }
    for (int l = L; l >= 3; --l) {
        for (int a = threadIdx.x; a < lv.n[l]; a += kCoarseWG) {
            const int g = lv.off[l] + a;
            const double *q = Rb + 3 * (g - base);
            double c0, c1, c2;
            apply_inv(Dinv + 6 * (int64_t)g, q[0], q[1], q[2], c0, c1, c2);
            if (l < L) {
                const double *up = Cb + 3 * (lv.off[l + 1] - base + par[g]);
                c0 += up[0]; c1 += up[1]; c2 += up[2];
            }
            double *o = Cb + 3 * (g - base);
            o[0] = c0; o[1] = c1; o[2] = c2;
        }
        __syncthreads();
    }
}

// Levels >= 3 with linear fields, in one workgroup, from the level-3 sums R9_3 of
// the restriction: R9_l (l > 3) = sum over the level-(l-1) children c of (R9_c[0],
// alpha R9_c[1] + beta_u R9_c[0], alpha R9_c[2] + beta_v R9_c[0]) with alpha = s_c /
// s_A, beta = (c_c - c_A) / s_A (the child's basis on the parent's; R9_c[m] the
// three components of feature m).  Then from the top down C9_l = D9_l^+ R9_l plus the
// parent's field re-expressed on the aggregate's basis (the same alpha, beta); the
// level-3 fields go to C9.
// One aggregate per thread (the linear fields apply when these levels hold at most
// kCoarse9WG aggregates, ml_prepare_linear): every load (the level-3 sums, geometry,
// parents, child ranges and the thread's own factors) is issued in one round, then
// the levels run in LDS and registers.  One workgroup, so bound by its chain of dependent
// steps: a child lifts its own sums to its parent's basis, nine threads a parent add
// them, every level's factors are applied at once, and the way down only re-expresses the
// parents' fields.  The factors and partial sums are stored one value of every aggregate
// after the other.  The bytes that one CU can read count too: a workgroup reads the
// factors of its own 64 level-3 aggregates only, and repeats the levels above.
// 379 aggregates on level 3 (1024^2): 17.0 us with the parents lifting their children one
// by one and a level's factors applied after the other, 11.2 now with one workgroup, 9.0
// with six; 512^2 8.4 and 5.4; a dozen aggregates 3.8 either way.
using eolc::kCoarse9WG;

// One aggregate of the levels >= 3 to a thread (W threads, at least as many): the fields
// of the level-3 aggregates [own0, own1), and of every one above, in sC[9 h ..], visible
// to all; false: the solve has stopped.  LDS: sT and sC 9 values an aggregate, sg 4, sc 2.
template <int W>
__device__ __forceinline__ bool coarse9_levels(const MLLevels &lv, const int *__restrict__ cptr,
                                               const int *__restrict__ par, const double *__restrict__ geo,
                                               const double *__restrict__ D9, const double *__restrict__ R9p,
                                               const SolverScalars *scal, int check_done, int own0, int own1,
                                               double *__restrict__ sT, double *__restrict__ sC,
                                               double *__restrict__ sg, int *__restrict__ sc)
{
    const int L = lv.L, base = lv.off[3];
    const int M = lv.off[L + 1] - base, n3 = lv.n[3];
    const int h = threadIdx.x;   // this thread's aggregate (levels >= 3 concatenated)
    const bool mine = h >= n3 || (h >= own0 && h < own1);
    // Every load is issued before the first wait, without branches between them (clamped
    // indexes).  The level and the offsets of its neighbour levels come from the uniform
    // offsets with constant indices (scalar loads; a variable index reads the argument
    // block with a vector load, one more memory round per level), and the LDS stores
    // follow the loads.
    int l = h < M ? 3 : 0;
    int offl = lv.off[3], coffl = 0, offm1 = lv.off[2], offp1 = lv.off[4];
#pragma unroll
    for (int k = 4; k <= eolc::kMLMaxLevels; ++k)
        if (k <= L && h >= lv.off[k] - base) {   // offsets increase with the level
            l = h < M ? k : 0;
            offl = lv.off[k];
            coffl = lv.coff[k];
            offm1 = lv.off[k - 1];
            offp1 = lv.off[k + 1];
        }
    const int ci = l > 3 ? coffl + h - (offl - base) : 0;
    double r3[kRestrict3Parts][9], F[kFact9], g4[4] = {0, 0, 0, 0};
    int pp = 0, ca = 0, cz = 0;
    if (h < M) {   // (wavefronts without an aggregate load nothing)
        const int h3 = min(h, n3 - 1);
#pragma unroll
        for (int q = 0; q < kRestrict3Parts; ++q)
#pragma unroll
            for (int k = 0; k < 9; ++k) r3[q][k] = R9p[((int64_t)k * n3 + h3) * kRestrict3Parts + q];
#pragma unroll
        for (int k = 0; k < 4; ++k) g4[k] = geo[4 * (int64_t)(base + h) + k];
        pp = par[min(base + h, lv.off[L] - 1)];
        ca = cptr[ci];
        cz = cptr[ci + 1];
        if (mine)
#pragma unroll
            for (int k = 0; k < kFact9; ++k) F[k] = D9[(int64_t)k * M + h];
    }
    // the children and the parent as threads
    const int c0 = offm1 - base + ca, c1 = offm1 - base + cz;
    const int hp = l < L ? offp1 - base + pp : 0;
    if (check_done && scal->done) return false;
    if (h < M) {
#pragma unroll
        for (int k = 0; k < 4; ++k) sg[4 * h + k] = g4[k];
        sc[2 * h] = c0;
        sc[2 * h + 1] = c1;
    }
    // the level-3 sums: the restriction's partial sums of each aggregate, in order
    double R[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (h < n3)
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            double v = r3[0][k];
#pragma unroll
            for (int q = 1; q < kRestrict3Parts; ++q) v += r3[q][k];
            R[k] = v;
        }
    __syncthreads();
    // this aggregate's basis on its parent's
    double al = 0.0, bu = 0.0, bv = 0.0;
    if (h < M && l < L) {
        const double ip = sg[4 * hp + 3];
        al = g4[2] * ip;
        bu = (g4[0] - sg[4 * hp]) * ip;
        bv = (g4[1] - sg[4 * hp + 1]) * ip;
    }
    for (int lev = 4; lev <= L; ++lev) {
        if (l == lev - 1) {   // (threads without an aggregate have l = 0)
            double t[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
            lift9(R, al, bu, bv, t);
#pragma unroll
            for (int q = 0; q < 9; ++q) sT[9 * h + q] = t[q];
        }
        __syncthreads();
        const int p0 = lv.off[lev] - base;
        for (int t = h; t < 9 * lv.n[lev]; t += W) {
            const int p = p0 + t / 9, q = t % 9, e = sc[2 * p + 1];
            double v = 0.0;
#pragma unroll 4
            for (int ch = sc[2 * p]; ch < e; ++ch) v += sT[9 * ch + q];
            sT[9 * p + q] = v;
        }
        __syncthreads();
        if (l == lev)
#pragma unroll
            for (int q = 0; q < 9; ++q) R[q] = sT[9 * h + q];
    }
    double cf[9];
    if (h < M && mine) apply9(F, R, cf);
    for (int lev = L; lev >= 3; --lev) {
        if (l == lev && mine) {
            if (lev < L) lower9(sC + 9 * hp, al, bu, bv, cf);
#pragma unroll
            for (int q = 0; q < 9; ++q) sC[9 * h + q] = cf[q];
        }
        __syncthreads();
    }
    return true;
}

__global__ void __launch_bounds__(kCoarse9WG) k_ml_coarse9(MLLevels lv, const int *__restrict__ cptr,
                                                           const int *__restrict__ par, const double *__restrict__ geo,
                                                           const double *__restrict__ D9, const double *__restrict__ R9p,
                                                           double *__restrict__ C9, const SolverScalars *scal,
                                                           int check_done)
{
    __shared__ double sT[9 * kCoarse9WG], sC[9 * kCoarse9WG], sg[4 * kCoarse9WG];
    __shared__ int sc[2 * kCoarse9WG];
    // this workgroup's 64 of level 3
    const int own0 = 64 * blockIdx.x, own1 = min(own0 + 64, lv.n[3]);
    if (!coarse9_levels<kCoarse9WG>(lv, cptr, par, geo, D9, R9p, scal, check_done, own0, own1, sT, sC, sg, sc)) return;
    for (int t = 9 * own0 + (int)threadIdx.x; t < 9 * own1; t += kCoarse9WG) C9[t] = sC[t];
}

// z = D0 r + coarse correction (zero on fixed DOFs); r.z partials -> PB[parity] slot 0.
// Levels 1 and 2 are applied here, per vertex, from the restricted sums; levels >= 3
// arrive accumulated in C_3.
// In an iteration (x given) x += alpha p too, with the restriction's alpha.
// FINE = false: the coarse corrections alone (z_i = C(a_i) + C_3), for the learned
// blocks' training loss, whose fine term is the network's.
template <class T, bool FINE, int W>
__global__ void __launch_bounds__(W) __attribute__((amdgpu_waves_per_eu(8, 8)))
k_ml_prolong(int parity, int N, MLLevels lv, const int *__restrict__ agg1, const int *__restrict__ anc3,
             const double *__restrict__ Dinv, const double *__restrict__ R, const double *__restrict__ C,
             const T *__restrict__ D, const T *__restrict__ r, T *__restrict__ z,
             const unsigned char *__restrict__ fixmask, const SolverScalars *scal, double *partials, int check_done,
             const double *__restrict__ feat3, const double *__restrict__ C9, const T *__restrict__ p,
             double *__restrict__ x)
{
    __shared__ double lds[2 * (W / 64) + 2];
    int rb, re;
    wg_rows(N, &rb, &re);
    const int i0 = rb + (int)threadIdx.x;
    // the first vertex's aggregate indices are read together with the stop flag, so
    // both corrections below load in one round
    int a = 0, u = 0;
    if (i0 < re) {
        a = agg1[i0];
        if (lv.L >= 3) u = anc3[i0];
    }
    if (check_done && scal->done) return;
    const double alpha = x ? scal->alpha : 0.0;
    double srz = 0.0;
    for (int i = i0; i < re; i += W) {
        if (i != i0) {
            a = agg1[i];
            if (lv.L >= 3) u = anc3[i];
        }
        double c0, c1, c2;
        if (lv.L >= 2) {
            // levels 1 and 2, combined per level-1 aggregate by the restriction
            c0 = C[3 * a]; c1 = C[3 * a + 1]; c2 = C[3 * a + 2];
            if (lv.L >= 3) {
                if (C9) {   // the level-3 aggregate's linear field at this vertex
                    const double *P = C9 + 9 * (int64_t)(u - lv.off[3]);
                    const double gu = feat3[2 * (int64_t)i], gv = feat3[2 * (int64_t)i + 1];
                    c0 += fma(gv, P[6], fma(gu, P[3], P[0]));
                    c1 += fma(gv, P[7], fma(gu, P[4], P[1]));
                    c2 += fma(gv, P[8], fma(gu, P[5], P[2]));
                } else {
                    const double *up = C + 3 * (int64_t)u;
                    c0 += up[0]; c1 += up[1]; c2 += up[2];
                }
            }
        } else {
            apply_inv(Dinv + 6 * (int64_t)a, R[3 * a], R[3 * a + 1], R[3 * a + 2], c0, c1, c2);
        }
        const T r0 = r[3 * i], r1 = r[3 * i + 1], r2 = r[3 * i + 2];
        if (x)
#pragma unroll
            for (int c = 0; c < 3; ++c) x[3 * (int64_t)i + c] = fma(alpha, (double)p[3 * (int64_t)i + c], x[3 * (int64_t)i + c]);
        double g0 = 0.0, g1 = 0.0, g2 = 0.0;
        if constexpr (FINE) {
            T f0, f1, f2;
            eolc::apply_sym3<T>(D + i, N, r0, r1, r2, f0, f1, f2);
            g0 = (double)f0; g1 = (double)f1; g2 = (double)f2;
        }
        const unsigned fm = fixmask[i];
        const T z0 = (fm & 1u) ? (T)0 : (T)(g0 + c0);
        const T z1 = (fm & 2u) ? (T)0 : (T)(g1 + c1);
        const T z2 = (fm & 4u) ? (T)0 : (T)(g2 + c2);
        z[3 * i] = z0; z[3 * i + 1] = z1; z[3 * i + 2] = z2;
        srz += ((double)r0 * (double)z0 + (double)r1 * (double)z1) + (double)r2 * (double)z2;
    }
    double v[1] = {srz};
    write_partials<1, W>(v, PB(partials, parity), lds);
}

// The prolongation of a small mesh, a vertex to a thread, with the levels >= 3 formed by
// every workgroup for itself: the same operations as the coarse kernels, so the same z, a
// launch less and most of its latency hidden.  131 x 97 quads, mixed: 3.8 us and 4.0 in two
// kernels, 4.9 in one.
constexpr int kFusedCoarse = 64, kFusedLinear = 40;
template <class T, bool LIN>
__global__ void __launch_bounds__(eolc::kVecWG)
k_ml_prolong_coarse(int parity, int N, MLLevels lv, const int *__restrict__ agg1, const int *__restrict__ anc3,
                    const int *__restrict__ cptr, const int *__restrict__ par, const double *__restrict__ geo,
                    const double *__restrict__ D9, const double *__restrict__ R9p, const double *__restrict__ Dinv,
                    const double *__restrict__ R, const double *__restrict__ C, const T *__restrict__ D,
                    const T *__restrict__ r, T *__restrict__ z, const unsigned char *__restrict__ fixmask,
                    const SolverScalars *scal, double *partials, int check_done, const double *__restrict__ feat3,
                    const T *__restrict__ p, double *__restrict__ x)
{
    constexpr int W = eolc::kVecWG, K = kFusedCoarse;
    __shared__ double lds[2 * (W / 64) + 2];
    __shared__ double sT[9 * K], sC[9 * K], sg[4 * K];
    __shared__ int sc[2 * K];
    int rb, re;
    wg_rows(N, &rb, &re);
    const int i = rb + (int)threadIdx.x;
    const bool on = i < re;
    // the vertex's own values are on their way while the levels are formed
    int a = 0, u = 0;
    double gu = 0.0, gv = 0.0;
    T rv[3] = {0, 0, 0}, f[3] = {0, 0, 0}, pv[3];
    double xv[3];
    unsigned fm = 0;
    if (on) {
        if (x)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                pv[c] = p[3 * i + c];
                xv[c] = x[3 * i + c];
            }
        a = agg1[i];
        u = anc3[i];
#pragma unroll
        for (int c = 0; c < 3; ++c) rv[c] = r[3 * i + c];
        fm = fixmask[i];
        if (LIN) {
            gu = feat3[2 * (int64_t)i];
            gv = feat3[2 * (int64_t)i + 1];
        }
    }
    double c[3] = {0, 0, 0};
    if (on) {
#pragma unroll
        for (int k = 0; k < 3; ++k) c[k] = C[3 * a + k];
        eolc::apply_sym3<T>(D + i, N, rv[0], rv[1], rv[2], f[0], f[1], f[2]);
    }
    if (LIN) {
        if (!coarse9_levels<W>(lv, cptr, par, geo, D9, R9p, scal, check_done, 0, lv.n[3], sT, sC, sg, sc)) return;
    } else {
        if (!coarse_levels(lv, cptr, par, Dinv, R, scal, check_done, sT, sC)) return;
    }
    double v[1] = {0.0};
    if (on) {
        if (x) {
            const double alpha = scal->alpha;
#pragma unroll
            for (int k = 0; k < 3; ++k) x[3 * i + k] = fma(alpha, (double)pv[k], xv[k]);
        }
        const double *P = sC + (LIN ? 9 : 3) * (u - lv.off[3]);
        T zv[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            if (LIN) c[k] += fma(gv, P[6 + k], fma(gu, P[3 + k], P[k]));
            else c[k] += P[k];
            zv[k] = ((fm >> k) & 1u) ? (T)0 : (T)((double)f[k] + c[k]);
            z[3 * i + k] = zv[k];
        }
        v[0] = ((double)rv[0] * (double)zv[0] + (double)rv[1] * (double)zv[1]) + (double)rv[2] * (double)zv[2];
    }
    write_partials<1, W>(v, PB(partials, parity), lds);
}

inline int blocks_for(int64_t n, int t = 256) { return (int)((n + t - 1) / t); }

}  // namespace

namespace eolc {

hipError_t ml_setup(eolc_ctx *c, bool linear)
{
    MLState &m = c->ml;
    const MLLevels &lv = m.lv;
    m.lin_on = false;
    if (lv.L <= 0) return hipSuccess;
    const Topology &t = c->topo;
    hipLaunchKernelGGL(k_ml_diag1, dim3(blocks_for((int64_t)lv.n[1] * kDiagLanes)), dim3(256), 0, c->stream, lv, m.hord, m.ptr1, m.gpos,
                       c->slice_off, c->slen, c->scol, m.lam, c->A64, t.nbs, c->fixmask, m.V, m.Dinv);
    for (int l = 2; l <= lv.L; ++l)
        hipLaunchKernelGGL(k_ml_diagup, dim3(lv.n[l]), dim3(64), 0, c->stream, l, lv, m.cptr, m.V,
                           m.Dinv);
    if (linear && m.lin_ok) {
        const int n_hi = lv.off[lv.L + 1] - lv.off[kMLLinFrom];
        hipLaunchKernelGGL(k_ml_gal9_part, dim3(m.nchunks), dim3(kGalWG), 0, c->stream, m.gchunk, m.hord, m.gpos,
                           c->slice_off, c->slen, c->scol, m.lam, c->A64, t.nbs, c->fixmask, c->X, m.geo, m.gpart);
        hipLaunchKernelGGL(k_ml_gal9_fin, dim3(n_hi), dim3(64), 0, c->stream, n_hi, m.gcp, m.gpart,
                           m.D9);
        m.lin_on = true;
    }
    return hipGetLastError();
}

static bool ml_linear_on(const eolc_ctx *c) { return c->ml.lin_on && c->ml.lv.L >= kMLLinFrom; }

static_assert(kRestrictGrid <= kMaxPartials && kCoarse9WG * kRestrict3Parts + 7 <= kMaxPartials, "partials of r.r");
int ml_restrict_grid(const eolc_ctx *c)
{
    const MLLevels &lv = c->ml.lv;
    if (ml_linear_on(c)) return (lv.n[3] * kRestrict3Parts + 7) & ~7;   // (a multiple of 8, as logical_wg needs)
    const int waves = lv.L >= 2 ? lv.n[2] : (lv.n[1] + 63) / 64;
    return std::min((blocks_for((int64_t)64 * waves, kRestrictWG) + 7) & ~7, kRestrictGrid);
}

// The prolongation forms the levels >= 3 where a vertex kernel has 256 threads a workgroup
// and these levels hold few aggregates: every workgroup reads all their factors.  Steps of
// n^2 quads, two kernels and one (ms): linear fields 48: 3.83 3.51, 131: 6.11 5.52, 200: 8.53
// 7.93, 300 (37 aggregates): 16.1 15.5, 380 (57): 27.5 29.0; translations, whose factors are a
// ninth, 131: 6.00 5.55, 300: 22.4 21.8, 380: 40.0 39.1.
static bool ml_fused(const eolc_ctx *c)
{
    const MLLevels &lv = c->ml.lv;
    return lv.L >= 3 && lv.off[lv.L + 1] - lv.off[3] <= (ml_linear_on(c) ? kFusedLinear : kFusedCoarse) && vec_wg(c->topo.N) == kVecWG;
}

// On large meshes the vectors come from HBM whole, and the restriction's scattered pieces of
// q and r cost more than a pass of their own.  With the update in the restriction and the
// prolongation, and apart, us per multilevel iteration of n^2 quads: mixed 724 108.7 116.0,
// 1024 199.1 202.6, 1200 226.6 227.8, 1300 274.3 269.2, 1600 409.4 408.0, 2048 662.7 657.4;
// FP64 512 68.1 72.0, 1024 255.7 253.5, 1200 334.8 335.0, 1600 579.8 566.7.
constexpr int kApartN = 1572864;
static bool ml_update_apart(const eolc_ctx *c) { return c->topo.N > kApartN; }

// The restriction (with or after the vector update when there is one) and the coarse levels, with
// the linear fields when the last ml_setup formed them; fused: without the coarse levels,
// which the prolongation forms.
template <class T>
static void ml_coarse_chain(eolc_ctx *c, T *r, int parity, const MLUpdate *u, bool fused = false)
{
    const MLState &m = c->ml;
    const MLLevels &lv = m.lv;
    RestrictArgs g{lv,    m.hord, m.ptr1, m.cptr, m.kptr2, m.R, m.C,     m.Dinv, m.feat2,
                   m.geo, m.R9p,  c->scal, c->partials, u ? u->k : 0, u ? u->Ga : 0, vec_grid(c->topo.N), parity,
                   u != nullptr};
    VecUpdate<T> up{u ? static_cast<const T *>(u->q) : nullptr, r, (T)0};
    const bool apart = u && ml_update_apart(c), with = u && !apart;
    if (apart)
        hipLaunchKernelGGL((k_ml_update<T>), dim3(pcg_grid(c->topo.N)), dim3(WG), 0, c->stream, g, up, 3 * c->topo.N,
                           static_cast<const T *>(u->p), u->x);
    const dim3 grid(ml_restrict_grid(c));
    if (ml_linear_on(c)) {
        if (with) hipLaunchKernelGGL((k_ml_restrict3<T, true>), grid, dim3(kRestrict3WG), 0, c->stream, g, up);
        else hipLaunchKernelGGL((k_ml_restrict3<T, false>), grid, dim3(kRestrict3WG), 0, c->stream, g, up);
        if (!fused)
            hipLaunchKernelGGL(k_ml_coarse9, dim3(blocks_for(lv.n[3], 64)), dim3(kCoarse9WG), 0, c->stream, lv, m.cptr, m.par, m.geo, m.D9,
                           m.R9p, m.C9, c->scal, u != nullptr);
        return;
    }
    if (with) hipLaunchKernelGGL((k_ml_restrict<T, true>), grid, dim3(kRestrictWG), 0, c->stream, g, up);
    else hipLaunchKernelGGL((k_ml_restrict<T, false>), grid, dim3(kRestrictWG), 0, c->stream, g, up);
    if (lv.L >= 3 && !fused)
        hipLaunchKernelGGL(k_ml_coarse, dim3(1), dim3(kCoarseWG), 0, c->stream, lv, m.cptr, m.par, m.Dinv, m.R, m.C,
                           c->scal, u != nullptr);
}

// The prolongation on the vector kernels' grid (vec_wg, vec_grid).
template <class T, bool FINE>
static void launch_prolong(eolc_ctx *c, int parity, const T *D, const T *r, T *z, const MLUpdate *u)
{
    const MLState &m = c->ml;
    const MLLevels &lv = m.lv;
    const int N = c->topo.N;
    const double *c9 = ml_linear_on(c) ? m.C9 : nullptr;
    const bool with = u && !ml_update_apart(c);   // x += alpha p here
    auto go = [&](auto w) {
        constexpr int W = decltype(w)::value;
        hipLaunchKernelGGL((k_ml_prolong<T, FINE, W>), dim3(vec_grid(N)), dim3(W), 0, c->stream, parity, N, lv, m.agg1,
                           m.anc3, m.Dinv, m.R, m.C, D, r, z, c->fixmask, c->scal, c->partials, u != nullptr, m.feat3, c9,
                           with ? static_cast<const T *>(u->p) : nullptr, with ? u->x : nullptr);
    };
    if (vec_wg(N) == kVecWG) go(std::integral_constant<int, kVecWG>());
    else go(std::integral_constant<int, WG>());
}

template <class T>
static void launch_prolong_coarse(eolc_ctx *c, int parity, const T *D, const T *r, T *z, const MLUpdate *u)
{
    const MLState &m = c->ml;
    const int N = c->topo.N;
    auto go = [&](auto lin) {
        hipLaunchKernelGGL((k_ml_prolong_coarse<T, decltype(lin)::value>), dim3(vec_grid(N)), dim3(kVecWG), 0, c->stream,
                           parity, N, m.lv, m.agg1, m.anc3, m.cptr, m.par, m.geo, m.D9, m.R9p, m.Dinv, m.R, m.C, D, r, z,
                           c->fixmask, c->scal, c->partials, u != nullptr, m.feat3,
                           u ? static_cast<const T *>(u->p) : nullptr, u ? u->x : nullptr);
    };
    if (ml_linear_on(c)) go(std::true_type());
    else go(std::false_type());
}

hipError_t ml_apply(eolc_ctx *c, bool mixed, int parity, const MLUpdate *u)
{
    const bool fused = ml_fused(c);
    auto apply = [&](const auto *D, auto *r, auto *z) {
        using T = std::remove_pointer_t<decltype(r)>;
        ml_coarse_chain<T>(c, r, parity, u, fused);
        if (fused) launch_prolong_coarse<T>(c, parity, D, r, z, u);
        else launch_prolong<T, true>(c, parity, D, r, z, u);
    };
    if (mixed) apply(c->D32, c->r32, c->z32);
    else apply(c->D64, c->r64, c->z64);
    return hipGetLastError();
}

// z64 = the coarse corrections of r64 alone (no fine blocks), FP64, fixed DOFs zero.
hipError_t ml_coarse64(eolc_ctx *c)
{
    if (c->ml.lv.L <= 0) return hipMemsetAsync(c->z64, 0, sizeof(double) * 3 * (size_t)c->topo.N, c->stream);
    ml_coarse_chain<double>(c, c->r64, 0, nullptr);
    launch_prolong<double, false>(c, 0, c->D64, c->r64, c->z64, nullptr);
    return hipGetLastError();
}

}  // namespace eolc
