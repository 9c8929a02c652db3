/*
 * fsx_kernels.hip -- gfx950 kernels of the FFT dimer SAXS scoring path and
 * the C-ABI launchers the host side calls (fsx_hip_*).
 *
 * Pipeline for one call (reference: src/fftsaxs.c:608-986):
 *   k_bessel      j_p(z q) by the reference's truncated series        (fftsaxs.c:110-121, sfbessel.c:40-60)
 *   k_tmat        translation operator T^{|m|}_{l l1}(q z)            (fftsaxs.c:182-243)
 *   k_rotate      receptor  R^X_lm(b1,g1,q) = sum_m1 e^{-i m1 g1} d^l_{m m1}(b1) A^X_{l m1}
 *                 ligand    B^Y_lm(b2,g2,q) = sum_m2 e^{-i m2 g2} d^l_{m m2}(b2) conj(B^Y_{l m2})
 *                 (the beta/gamma factors of compute_sum1/compute_sum2 and of the
 *                 3-D DFT, fftsaxs.c:251-333, 416-524, 680, folded per pose axis)
 *   k_count/k_units/k_scatter  bucket poses by z, beta2 and gamma2, units of buckets
 *   k_cross       per unit and q (fsx_cross.h): U^Y_lm = sum_l1 conj(T_{|m| l l1}) B^Y_{l1 m} in LDS,
 *                 then per pose 2 Re sum_lm e^{-i m a2} (R^X U^Y [+ R^Y U^X]) for the six
 *                 cross terms VV,VD,VW,DD,DW,WW (fill_var, fftsaxs.c:87-108)
 *   k_fit         constant terms + peak rescale + bounded L-BFGS-B chi^2 fit per pose
 *                 (fill_const fftsaxs.c:52-85, sxs_fit_params min_saxs.c:153-259)
 *
 * The Bessel series, the translation operator and the fit run with FP
 * contraction off (bit-level agreement with the reference's arithmetic);
 * the contraction kernels use FMA.
 */
#include <hip/hip_runtime.h>
#include <math.h>
#include <pthread.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <type_traits>

#include "../fsx_internal.h"
#include "../fsx_pose.h"
#include "../fsx_rules.h"
/* the fit kernels keep the L-BFGS-B blocks K11, K12, K22 and WN1 in LDS, one
 * column of 256 lanes (a fit block) per value */
#define FSX_LB_KSHARED
#define FSX_LB_KSTRIDE 256
#include "../fsx_lbfgsb.h"
#include "../fsx_lb2.h"

#define FSX_WAVE 64
/* counters of the fit kernel: evaluations, capped fits, loop iterations summed
 * over wavefronts, of those wavefront-wide ones, the longest wavefront's */
#define FSX_TALLY_N 5

struct cplx { double re, im; };
struct cplx32 { float re, im; };   /* element of the mixed-precision (FP32) tables */
typedef double fsx_v4d __attribute__((ext_vector_type(4)));   /* FP64 MFMA 16x16x4 result */
#include "fsx_cross.h"

/* ---------------------------------------------------------------------- */
/* device helpers */

__device__ __forceinline__ int lm_l(int lm)
{
    int l = (int)sqrt((double)lm);
    while (l * l > lm) l--;
    while ((l + 1) * (l + 1) <= lm) l++;
    return l;
}

__device__ __forceinline__ int pos_mod(long v, int n)
{
    long r = v % n;
    return (int)(r < 0 ? r + n : r);
}

/* x^n for x > 0, integer n >= 0, correctly rounded: binary exponentiation
 * in double-double (each product exact to ~2^-104 through fma), rounded
 * once at the end.  glibc's pow, which the reference calls, is correctly
 * rounded for these arguments in practice; the device pow is not. */
__device__ __forceinline__ void dd_mul(double ah, double al, double bh, double bl, double *rh,
                                       double *rl)
{
    double p = ah * bh;
    double e = fma(ah, bh, -p);
    e = e + (ah * bl + al * bh);
    double h = p + e;
    *rl = e - (h - p);
    *rh = h;
}

__device__ double pow_int_cr(double x, int n)
{
    double rh = 1.0, rl = 0.0, bh = x, bl = 0.0;
    while (n) {
        if (n & 1) dd_mul(rh, rl, bh, bl, &rh, &rl);
        n >>= 1;
        if (n) dd_mul(bh, bl, bh, bl, &bh, &bl);
    }
    return rh + rl;
}

/* j_l(x) exactly as sfbessel.c:40-60 (contraction off) */
__device__ double dev_sbessel(int l, double x)
{
#pragma clang fp contract(off)
    if (x > 0.0) {
        double tl1 = 2.0 * (double)l + 1.0;
        int n = (int)tl1;
        double f = 1.0;
        for (int i = 1; i <= n; i += 2) f *= (double)i;
        double term = 1.0 / f;
        double sum = term;
        for (int k = 1; fabs(term / sum) > 0.00001; k++) {
            double ratio = (-1.0) * x * x / (2.0 * (double)k * (2.0 * (double)k + tl1));
            term *= ratio;
            sum += term;
        }
        return sum * pow_int_cr(x, l);
    }
    return l == 0 ? 1.0 : 0.0;
}

__global__ void k_bessel(double *bes, const double *zvals, const double *qvals, int znum,
                         int Q, int P)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long tot = (long)znum * Q * P;
    if (i >= tot) return;
    int p = (int)(i % P);
    int q = (int)((i / P) % Q);
    int z = (int)(i / ((long)P * Q));
    bes[i] = dev_sbessel(p, zvals[z] * qvals[q]);
}

__global__ void k_sbessel_batch(const double *x, int n, int P, double *out)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)n * P) return;
    out[i] = dev_sbessel((int)(i % P), x[i / P]);
}

/* T^{|m|}_{l l1}(q z) (fftsaxs.c:182-243), computed from (min(l,l1), max(l,l1))
 * so the mirrored entries are bitwise equal, as in fftsaxs.c:213-238, in the
 * operand order of the cross-term kernel's matrix products: per block and tile
 * of FSX_CROSS_TILE l, steps of 4 l1, FP32 [l1][l], FP64 [l1][l % 4][l / 4] (what a
 * lane of four 4x4x4 products takes side by side; split: 4 even, then 4 odd
 * l1), with zeros where l
 * or l1 exceeds L.  tb: the number of blocks, then per block 2 |m| + split
 * and its first value, then the table size
 * Tn.  Only p of the parity of l + l1
 * contribute (the 3j symbol (l p l1; 0 0 0) vanishes exactly otherwise), so
 * T = i^(l1 - l) tau with tau real, and the sum runs over those p: stored is
 * tau = i^(l - l1) T.
 * One thread forms one table entry for FSX_TMAT_ZQ (z, q): its d-symbols, whose
 * addresses are scattered over the wavefront, are then read once for all of
 * them, not once for each. */
#define FSX_TMAT_ZQ 8
template <typename F>
__global__ void __launch_bounds__(256)
k_tmat(F *T, const double *bes, const double *ds, const int *tb, int nzq, int L, int Tn)
{
#pragma clang fp contract(off)
    const int K = L + 1, N = 2 * L + 1;
    const int nbx = (Tn + 255) / 256, by = blockIdx.x / nbx;
    const int r = (blockIdx.x - by * nbx) * 256 + threadIdx.x;
    if (r >= Tn) return;
    int k = 0;
    while (k + 1 < tb[0] && r >= tb[2 * k + 4]) k++;
    const int m = tb[2 * k + 1] >> 1, split = tb[2 * k + 1] & 1, Km = K - m;
    constexpr int TL = FSX_CROSS_TILE;
    const int nks = cross_steps(Km, split), sv = cross_tstep(split), o = r - tb[2 * k + 2];
    const int st = o / sv, i = o % sv, ks = st % nks;
    const int l = m + TL * (st / nks) + (sizeof(F) == 4 ? i & 15 : (i >> 2 & 3) + 4 * (i & 3));
    const int j = i / TL;   /* l1 of the step: four, or four even and four odd ones */
    const int l1 = m + (split ? 2 * (4 * ks + (j & 3)) + (j >> 2) : 4 * ks + j);
    const bool in = l <= L && l1 <= L;
    const int lo = in ? (l < l1 ? l : l1) : m, hi = in ? (l < l1 ? l1 : l) : m;
    const double *d = ds + ((long)(lo * (lo + 1) + m) * K + hi) * N;
    const double sg = (m % 2) ? -1.0 : 1.0;
    const int zq0 = by * FSX_TMAT_ZQ;
    double t[FSX_TMAT_ZQ];
#pragma unroll
    for (int k = 0; k < FSX_TMAT_ZQ; k++) t[k] = 0.0;
    if (in)
        for (int p = hi - lo; p <= lo + hi; p += 2) {
            const double dv = sg * d[p];
            const bool neg = (p & 2) != 0;
#pragma unroll
            for (int k = 0; k < FSX_TMAT_ZQ; k++) {
                const double v = dv * bes[(size_t)min(zq0 + k, nzq - 1) * N + p];
                t[k] += neg ? -v : v;
            }
        }
    /* the sum is T's real part for even l - l1, its imaginary part for odd */
    const int ph = ((l - l1) % 4 + 4) % 4;
#pragma unroll
    for (int k = 0; k < FSX_TMAT_ZQ; k++)
        if (zq0 + k < nzq) T[(size_t)(zq0 + k) * Tn + r] = (F)(ph == 1 || ph == 2 ? -t[k] : t[k]);
}

/* x mod n in [0, n) for |x| < 2^24, n >= 1: a float quotient estimate
 * (off by at most one) and one correction. */
__device__ __forceinline__ int mod_small(int x, int n, float inv_n)
{
    int k = x - n * (int)floorf((float)x * inv_n);
    if (k < 0) k += n;
    else if (k >= n) k -= n;
    return k;
}

/* ---- rotated receptor / ligand coefficients -------------------------------
 * k_twiddle: src~[q][X][lm][g] = e^{-i m1 g} src^X_{l m1}(q) (conjugated first
 * for the ligand), gamma innermost.
 * k_rotate: out^X_{lm}(beta, gamma, q) = sum_{m1} d^l_{m m1}(beta) src~[q][X][l m1][gamma]
 * with one wavefront per (beta, q, X, entry) and the lanes over gamma, so the
 * Wigner-d value of a term is the same for the whole wavefront and the
 * source loads are contiguous. */
__global__ void k_twiddle(cplx *dst, const double *src_re, const double *src_im,
                          const double *twg, int ng, int Q, int L, int conj_src)
{
    const int K2 = (L + 1) * (L + 1);
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)Q * 3 * K2 * ng) return;
    int g = (int)(i % ng);
    long r = i / ng;
    int lm = (int)(r % K2);
    long xq = r / K2;   /* q*3 + X */
    int X = (int)(xq % 3), q = (int)(xq / 3);
    int l = lm_l(lm), m1 = lm - l * (l + 1);
    int k = mod_small(m1 * g, ng, 1.0f / (float)ng);
    double wr = twg[2 * k], wi = twg[2 * k + 1];
    long so = ((long)X * Q + q) * K2 + lm;
    double sr = src_re[so], si = (conj_src ? -1.0 : 1.0) * src_im[so];
    cplx v;
    v.re = wr * sr - wi * si;
    v.im = wr * si + wi * sr;
    dst[i] = v;
}

/* Where a rotated value goes.  Per m-chunk a row of the table (one q, beta,
 * gamma) holds
 *   ligand:   [l1, in steps of 4 per m][re, im][V, D, W], the order in which a
 *             lane of the translation product reads its operands (a block that
 *             is summed in both orders of l1 is there twice);
 *   receptor: [V, D, W][slot][re, im], the slots across the lanes of the
 *             pairing.  The m = 0 entries l = 2i and 2i + 1 of
 *             conjugate-symmetric coefficients, whose turned values i^l R_l0
 *             are real, are the two halves of slot i. */
struct fsx_tabmap {
    /* per entry: l, chunk, offset in the row, zero entries to add (ligand), and
     * the two of a second place (offset -1: none); per chunk: row length */
    const int *l, *pass, *off, *pad, *off2, *pad2, *rs;
    const long *coff;                       /* per chunk: first value */
    int lig, npk;                           /* ligand table; entries packed in halves */
};

/* one entry's place in the rows of a table: its values of row qrow go to d + qrow
 * * rs */
template <typename F>
struct fsx_tabput {
    F *d, *d2;          /* first row's place, the second one (NULL: none) */
    size_t rs;
    int pad, pad2, lig, half;
    int ph;             /* power of i that turns the value */
    __device__ __forceinline__ fsx_tabput(F *out, const fsx_tabmap &M, int e, int X, int lsgn)
    {
        const int c = M.pass[e], r = M.rs[c], o2 = M.lig ? M.off2[e] : -1;
        F *b = out + M.coff[c] + (M.lig ? X : X * (r / 3));
        rs = r;
        d = b + M.off[e];
        d2 = o2 >= 0 ? b + o2 : NULL;
        pad = M.lig ? M.pad[e] : 0;
        pad2 = M.lig ? M.pad2[e] : 0;
        lig = M.lig;
        half = e < M.npk;
        ph = (lsgn > 0 ? M.l[e] : -M.l[e]) & 3;
    }
    __device__ __forceinline__ void put(size_t qrow, F x, F y) const
    {
        const F re = ph == 0 ? x : ph == 1 ? -y : ph == 2 ? -x : y;
        const F im = ph == 0 ? y : ph == 1 ? x : ph == 2 ? -y : -x;
        F *p = d + qrow * rs;
        if (lig) {
            p[0] = re;
            p[3] = im;
            for (int j = 1; j <= pad; j++) p[6 * j] = p[6 * j + 3] = 0;
            if (d2) {
                p = d2 + qrow * rs;
                p[0] = re;
                p[3] = im;
                for (int j = 1; j <= pad2; j++) p[6 * j] = p[6 * j + 3] = 0;
            }
        } else {
            /* a whole slot (at an even place) in one store */
            struct alignas(2 * sizeof(F)) slot { F re, im; };
            if (half) p[0] = re;
            else *reinterpret_cast<slot *>(p) = {re, im};
        }
    }
};

/* Wigner-d tables, per beta [l][16 rows][4 m1][64]: row r = l - m (so the rows m
 * >= 0 come first) and m1 + l in the order of a 16x16x4 product's first operand
 * (value 16 (m1 % 4) + r % 16), zeros past 2l + 1; dw_base(l): first value of l */
__host__ __device__ __forceinline__ int dw_steps(int l) { return (2 * l + 4) / 4; }
__host__ __device__ __forceinline__ int dw_size(int l) { return (2 * l + 16) / 16 * dw_steps(l) * 64; }

/* One block per (q, X, l, chunk of FSX_ROT_BC betas, gamma chunk of gc): the
 * 2l+1 source rows of l, gamma in the chunk, are staged in LDS
 * ([m1][gamma]) together with the blocks d^l_{m m1}(beta) of the chunk's
 * betas; the wavefronts then take (beta, pair of m) items and form
 * out^X_{lm}(beta, gamma) = sum_m1 d^l_{m m1}(beta) src_{l m1}(gamma), lanes
 * over gamma, m1 ascending.  The output goes to a staging table with rows
 * innermost, [q][X][entry][row] (lanes store consecutive rows);
 * k_tab_transpose then writes the table the cross-term kernel reads. */
#define FSX_ROT_BC 2
template <typename E>
__global__ void __launch_bounds__(256)
k_rotate(E *out, const cplx *srct, const double *dW, const int *mstart, int nbeta, int ng,
         int Q, int L, int gc, int mlo, int ne)
{
#pragma clang fp contract(fast)
    extern __shared__ cplx sR[];   /* [2l+1][gc], then FSX_ROT_BC blocks [2l+1][2l+1] of d */
    const int K = L + 1, K2 = K * K;
    const int nrows = nbeta * ng;
    const int lane = threadIdx.x % FSX_WAVE, wave = threadIdx.x / FSX_WAVE;
    const int nwave = blockDim.x / FSX_WAVE;
    const int nch = (ng + gc - 1) / gc, nbc = (nbeta + FSX_ROT_BC - 1) / FSX_ROT_BC;
    int r = blockIdx.x;
    const int ch = r % nch; r /= nch;
    const int bc = r % nbc; r /= nbc;
    const int l = r % K; r /= K;
    const int X = r % 3;
    const int q = r / 3;
    const int g0 = ch * gc, gn = (ng - g0) < gc ? (ng - g0) : gc;
    const int b0 = bc * FSX_ROT_BC, nbh = nbeta - b0 < FSX_ROT_BC ? nbeta - b0 : FSX_ROT_BC;
    /* output rows m = mb..l (all m, or m >= 0 for the half entry set) */
    const int w = 2 * l + 1, mb = mlo > -l ? mlo : -l, nm = l - mb + 1, ww = nm * w;
    double *sD = reinterpret_cast<double *>(sR + w * gc);
    int dbase = 0, dsz = 0;
    for (int k = 0; k <= L; k++) {
        if (k < l) dbase += dw_size(k);
        dsz += dw_size(k);
    }
    const cplx *src = srct + (((long)q * 3 + X) * K2 + l * (l + 1) - l) * ng + g0;
    for (int i = threadIdx.x; i < w * gc; i += blockDim.x) {
        int m1 = i / gc, g = i - m1 * gc;
        if (g < gn) sR[i] = src[(long)m1 * ng + g];
    }
    for (int i = threadIdx.x; i < nbh * ww; i += blockDim.x) {
        const int bb = i / ww, rem = i - bb * ww, mr = rem / w, k = rem - mr * w;
        const int row = l - mb - mr;
        sD[i] = dW[(size_t)(b0 + bb) * dsz + dbase + (row / 16 * dw_steps(l) + k / 4) * 64 + k % 4 * 16 +
                   row % 16];
    }
    __syncthreads();
    const int np = (nm + 1) / 2;   /* pairs of m */
    for (int it = wave; it < nbh * np; it += nwave) {
        const int bb = it / np, mi = 2 * (it - bb * np), b = b0 + bb;
        const bool two = mi + 1 < nm;
        const double *d0 = sD + bb * ww + mi * w, *d1 = two ? d0 + w : d0;
        E *o[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            /* entry (l, m) in m-major order */
            const int m = mb + (two ? mi + u : mi);
            const int e = mstart[m + L] + (l - (m < 0 ? -m : m));
            o[u] = out + ((long)(q * 3 + X) * ne + e) * nrows + (long)b * ng + g0;
        }
        for (int gw = 0; gw < gn; gw += FSX_WAVE) {
            const int g = gw + lane;
            if (g < gn) {
                double r0 = 0.0, i0 = 0.0, r1 = 0.0, i1 = 0.0;
#pragma unroll 4
                for (int k = 0; k < w; k++) {
                    const cplx v = sR[k * gc + g];
                    const double a0 = d0[k], a1 = d1[k];
                    r0 += a0 * v.re;
                    i0 += a0 * v.im;
                    r1 += a1 * v.re;
                    i1 += a1 * v.im;
                }
                E v0, v1;
                v0.re = r0;
                v0.im = i0;
                v1.re = r1;
                v1.im = i1;
                o[0][g] = v0;
                if (two) o[1][g] = v1;
            }
        }
    }
}

/* A rotated table from the staging layout [q][X][entry][row] to its final one,
 * each value turned by i^(lsgn l), through a 64-entry x TR-row LDS tile per
 * block: loads run along rows, stores along entries. */
template <typename E, int TR>
__global__ void __launch_bounds__(256)
k_tab_transpose(decltype(E::re) *out, const E *tmp, int ne, int nrows, int nte, int ntr,
                const fsx_tabmap M, int lsgn)
{
    __shared__ E tile[64][TR + 1];
    int bid = blockIdx.x;
    const int tr = bid % ntr;
    bid /= ntr;
    const int te = bid % nte;
    const int qx = bid / nte;   /* q * 3 + X */
    const int X = qx % 3, q = qx / 3;
    const int e0 = te * 64, r0 = tr * TR;
    const E *src = tmp + (long)qx * ne * nrows;
    for (int k = threadIdx.x; k < 64 * TR; k += 256) {
        const int i = k / TR, j = k - (k / TR) * TR;
        const int e = e0 + i, r = r0 + j;
        if (e < ne && r < nrows) tile[i][j] = src[(long)e * nrows + r];
    }
    __syncthreads();
    for (int k = threadIdx.x; k < 64 * TR; k += 256) {
        const int j = k >> 6, i = k & 63;
        const int e = e0 + i, r = r0 + j;
        if (e < ne && r < nrows) {
            const fsx_tabput<decltype(E::re)> P(out, M, e, X, lsgn);
            P.put((size_t)q * nrows + r, tile[i][j].re, tile[i][j].im);
        }
    }
}

/* Rotated table on FP64 MFMA, written in the cross-term kernel's layout in
 * one pass (no staging table, no transpose).  One block of four waves per
 * (q, X, beta, tile of GT gamma): for every l, the (m x m1) block of
 * d^l(beta) times the (m1 x gamma, re/im) block of twiddled source rows
 * src[q][X][l m1][gamma] (16x16x4 FP64 MFMA: lane i feeds A[i % 16][i / 16],
 * B[i / 16][i % 16]; result register j of lane i is D[i / 16 + 4j][i % 16]),
 * rows m = max(mlo, -l)..l, each block's m rows and 16 columns (8 gamma, real
 * and imaginary parts) a job of one wave.  The results go to an LDS tile of
 * the block's GT rows of the table, all entries; the tile is written out row
 * by row, turned by i^(lsgn l), exactly as k_tab_transpose writes it. */
template <typename E, int GT>
__global__ void __launch_bounds__(256)
k_rotate_mfma(decltype(E::re) *out, const cplx *srct, const double *dW, const int *mstart,
              const fsx_tabmap M, int nbeta, int ng, int Q, int L, int mlo, int ne, int lsgn)
{
    extern __shared__ double smem_raw[];
    E *tile = reinterpret_cast<E *>(smem_raw);   /* [GT][ne] */
    const int K = L + 1, K2 = K * K;
    const int nrows = nbeta * ng, ngt = (ng + GT - 1) / GT;
    /* the three X of a tile eight blocks apart, on the same XCD: the ligand table
     * has them side by side, and its L2 joins their parts of a line */
    int r = blockIdx.x / 24 * 8 + blockIdx.x % 8;
    const int X = blockIdx.x / 8 % 3;
    if (r >= Q * nbeta * ngt) return;
    const int gt = r % ngt; r /= ngt;
    const int b = r % nbeta;
    const int q = r / nbeta;
    const int g0 = gt * GT;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int NT = GT / 8;   /* 16-column tiles: 8 gamma x (re, im) each */
    constexpr int CH = 4;        /* steps of 4 m1 whose operands are loaded together */
    int dsz = 0;
    for (int l = 0; l <= L; l++) dsz += dw_size(l);
    const double *dWb = dW + (size_t)b * dsz + lane;
    const cplx *srcq = srct + (size_t)(q * 3 + X) * K2 * ng;
    const int i = lane & 15, k = lane >> 4;
    /* jobs (l, m-tile, column tile), dealt to the waves in turn, each in chunks
     * of CH steps; the operands of the next chunk (of this job or the next) are
     * in flight during the products of the current one.  The loads are
     * unconditional (past a job's end: values that meet a zero of the other
     * operand or are not stored), so that the wait before a chunk's products
     * leaves the next one's loads in flight. */
    struct { int l, mt, nt, k0, d0; } J = {0, 0, 0, 0, 0};   /* d0: first Wigner-d value of l */
    auto next_job = [&]() {
        if (++J.nt < NT) return;
        J.nt = 0;
        const int mb = mlo > -J.l ? mlo : -J.l;
        if (16 * ++J.mt < J.l - mb + 1) return;
        J.mt = 0;
        J.d0 += dw_size(J.l);
        J.l++;
    };
    auto next = [&]() {
        J.k0 += CH;
        if (J.k0 < dw_steps(J.l)) return;
        J.k0 = 0;
        for (int u = 0; u < 4; u++) next_job();
    };
    double av[2][CH], bv[2][CH];
    auto load = [&](double *a, double *bo) {
        if (J.l > L) return;
        const int g = min(g0 + J.nt * 8 + (i >> 1), ng - 1), nks = dw_steps(J.l);
        const double *drow = dWb + J.d0 + J.mt * nks * 64;
        const double *scol = reinterpret_cast<const double *>(srcq + (size_t)J.l * J.l * ng + g) + (i & 1);
#pragma unroll
        for (int st = 0; st < CH; st++) {
            a[st] = drow[64 * min(J.k0 + st, nks - 1)];
            bo[st] = scol[(size_t)min(4 * (J.k0 + st) + k, 2 * J.l) * ng * 2];
        }
    };
    for (int u = 0; u < w; u++) next_job();
    fsx_v4d acc = {0.0, 0.0, 0.0, 0.0};
    auto run = [&](const double *a, const double *bo, int l, int mt, int nt, int k0) {
        const int nks = dw_steps(l);
        if (k0 == 0) acc = (fsx_v4d){0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int st = 0; st < CH; st++)
            if (k0 + st < nks) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[st], bo[st], acc, 0, 0, 0);
        if (k0 + CH < nks) return;
        const int mb = mlo > -l ? mlo : -l, gl = nt * 8 + (i >> 1), part = i & 1;
#pragma unroll
        for (int rr = 0; rr < 4; rr++) {
            const int m = l - mt * 16 - k - 4 * rr;   /* rows by falling m */
            if (m >= mb) {
                const int e = mstart[m + L] + (l - (m < 0 ? -m : m));
                reinterpret_cast<decltype(E::re) *>(&tile[gl * ne + e])[part] = (decltype(E::re))acc[rr];
            }
        }
    };
    load(av[0], bv[0]);
    while (J.l <= L) {
        auto P = J;
        next();
        load(av[1], bv[1]);
        run(av[0], bv[0], P.l, P.mt, P.nt, P.k0);
        if (J.l > L) break;
        P = J;
        next();
        load(av[0], bv[0]);
        run(av[1], bv[1], P.l, P.mt, P.nt, P.k0);
    }
    __syncthreads();
    /* a thread takes an entry of all rows: its place is looked up once */
    const int gn = ng - g0 < GT ? ng - g0 : GT;
    for (int e = threadIdx.x; e < ne; e += blockDim.x) {
        const fsx_tabput<decltype(E::re)> P(out, M, e, X, lsgn);
        const size_t row = (size_t)q * nrows + b * ng + g0;
#pragma unroll 4
        for (int gl = 0; gl < gn; gl++) P.put(row + gl, tile[gl * ne + e].re, tile[gl * ne + e].im);
    }
}

/* ---- pose bucketing --------------------------------------------------- */
/* The counters of a call in one launch: bucket counts and fills (nc values)
 * and the record, bucket and unit counters zero, the fit queue at next0, the
 * fit tallies zero. */
__global__ void k_init(int *counts, long nc, int *tail, int *next, int next0,
                       unsigned long long *tally)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nc) counts[i] = 0;
    if (i < 3) tail[i] = 0;
    if (i < FSX_TALLY_N) tally[i] = 0;
    if (i == 0) *next = next0;
}

/* The mirror image of a rotated table row.  With d^l_{m,m1}(pi - beta) =
 * (-1)^(l+m) d^l_{m,-m1}(beta) and coefficients with A_{l,-m} = (-1)^(l+m)
 * conj(A_lm), the row of (pi - beta, gamma) is, in both tables and after their
 * turns by i^l and i^-l,
 *   R_lm(pi - beta, gamma) = (-1)^(l+m) conj(R_lm(beta, gamma + pi)),
 * so that with an even gamma grid the tables need only beta <= pi / 2: half
 * the rotations, and half the receptor rows of a q for an XCD's L2 to hold.
 * A ligand row is mirrored as the translation reads it (cross_body).  A pose
 * with a mirrored receptor row takes alpha2 negated (Re(w conj(R) U) = Re(conj(w)
 * R conj(U))), the slots' signs (-1)^(l+m) with its twiddles (row 2 alpha2 + 1),
 * and the products of the imaginary parts with the other sign. */
__device__ __forceinline__ void fsx_mirror(int nbeta, int na, int ng, int *b1, int *g1, int *alpha)
{
    const int hb = (nbeta - 1) / 2, hg = ng / 2;
    const bool m1 = *b1 > hb;
    if (m1) {
        *b1 = nbeta - 1 - *b1;
        *g1 = *g1 >= hg ? *g1 - hg : *g1 + hg;
        if (*alpha > 0) *alpha = na - *alpha;
    }
    *alpha = 2 * *alpha + m1;
}

/* bucket of each pose, (z, beta2, gamma2) or, zmajor 0, (beta2, z, gamma2), its
 * receptor row and twiddle row */
__global__ void k_count(const long long *poses, int n, int znum, int nbeta, int na, int ng,
                        int mirror, int zmajor, int *keys, int2 *info, int *counts)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int row, alpha;
    int key = fsx_pose_key(poses[i], znum, nbeta, na, ng, &row, &alpha);
    if (key >= 0) {
        if (!zmajor) {
            const int zb = key / ng, z = zb / nbeta;
            key += ((zb - z * nbeta) * znum + z - zb) * ng;
        }
        int b1 = row / ng, g1 = row - b1 * ng;
        if (mirror) fsx_mirror(nbeta, na, ng, &b1, &g1, &alpha);
        row = b1 * ng + g1;
        atomicAdd(&counts[key], 1);
    }
    keys[i] = key;
    info[i] = make_int2(row, alpha);
}

/* First record of every bucket and the cross-term units, one wavefront per
 * (z, beta2).  Units are cut greedily along gamma2: up to urows rows, in even
 * shares, and cap poses; a bucket of more poses takes several.  Blocks take units
 * at a fixed stride, so that one small unit per group (the last of 25 rows cut by
 * eights) left every fourth block with small ones only: cross terms FP32, L = 12,
 * 25-point grids, 70,000 poses 0.86 against 0.80 ms, L = 20, 41-point grids, 400,000
 * poses 6.10 against 5.67.  PASS 0 counts every
 * group's records and units (grp), PASS 1 adds those of the groups before and
 * writes; tail: records, non-empty buckets, units.
 * The records, and with them the fits, are in the order of the groups.  Lists of more
 * fits than start at once have them by (z, beta2) (zmajor): the poses of one z take
 * about the same number of evaluations, and the long ones don't come last (by (beta2,
 * z) the fits of 210,000 poses, L = 10, 41 q took 1.05 against 0.67 ms in the mixed form
 * and 1.53 against 1.27 in FP64, L = 12 1.13 against 0.73 and 1.69 against 1.35).
 * Shorter ones by (beta2, z), which spreads the long fits over the wavefronts (2,000
 * poses, L = 10, 31 q 0.35 against 0.38 ms mixed, 0.31 against 0.32 FP64).
 * The units are in the order of (beta2, z): by (z, beta2), or with ranges
 * reserved by atomics, an XCD's blocks work on all beta2 at a time and its L2 loses
 * the ligand rows (cross terms FP64 L = 15, 210,000 poses 9.76 against 9.27 ms; L =
 * 25, 200,000 poses 156 against 146, FP32 300,000 poses 65.5 against 61.7).
 * scanned: grp holds the sums already (k_unit_scan), for many groups; summing them in
 * every wavefront costs the square of their number. */
template <int PASS>
__global__ void __launch_bounds__(256)
k_units(const int *counts, int nzb, int nb, int zn, int ng, int urows, int cap, int *offs,
        fsx_unit *units, int *tail, int2 *grp, int scanned, int zmajor)
{
    const int zb = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (zb >= nzb) return;
    const int *c = counts + (size_t)zb * ng;
    const int z = zmajor ? zb / nb : zb % zn, b2 = zmajor ? zb % nb : zb / zn;
    int total = 0, first = 0;
    if (PASS) {
        /* records in the order of the buckets, units by (beta2, z) */
        const int ub = b2 * zn + z;
        if (scanned) {
            total = grp[zb].x;
            first = grp[ub].y;
        } else {
            for (int k = lane; k < zb; k += 64) total += grp[k].x;
            for (int k = lane; k < ub; k += 64) first += grp[k].y;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                total += __shfl_xor(total, o);
                first += __shfl_xor(first, o);
            }
        }
        total = __builtin_amdgcn_readfirstlane(total);
        first = __builtin_amdgcn_readfirstlane(first);
    }
    int p = 0, nz = 0, un = 0, ur = 0, uc = 0;   /* records so far, buckets; open unit's poses and rows; units */
    fsx_unit u;
    u.b2 = b2;
    u.z = z;
    u.pad = 0;
    /* non-empty buckets left, and rows of the open unit at most: the same number of
     * units in even shares (25 rows as 7, 6, 6, 6, not 8, 8, 8, 1) */
    const int v0 = lane < ng ? c[lane] : 0;
    int rem = __popcll(__ballot(v0 > 0)), lim = 0;
    for (int g0 = 64; g0 < ng; g0 += 64) rem += __popcll(__ballot(g0 + lane < ng && c[g0 + lane] > 0));
    for (int g0 = 0; g0 < ng; g0 += 64) {
        const int v = g0 == 0 ? v0 : g0 + lane < ng ? c[g0 + lane] : 0;
        if (PASS) {
            /* exclusive scan over the 64 buckets */
            int x = v;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(x, o);
                if (lane >= o) x += y;
            }
            if (g0 + lane < ng) offs[(size_t)zb * ng + g0 + lane] = total + p + x - v;
        }
        unsigned long long mask = __ballot(v > 0);
        nz += __popcll(mask);
        while (mask) {
            const int b = __builtin_ctzll(mask);
            mask &= mask - 1;
            int left = __builtin_amdgcn_readlane(v, b);
            while (left > 0) {
                /* close the open unit where the row does not fit in it */
                if (un > 0 && (ur == lim || un + left > cap)) {
                    if (PASS && lane == 0) {
                        u.n = un;
                        u.nrow = ur;
                        units[first + uc] = u;
                    }
                    uc++;
                    un = ur = 0;
                }
                if (un == 0) lim = (int)ceilf((float)rem / ceilf((float)rem / (float)urows));
                const int k = left < cap - un ? left : cap - un;
                if (PASS) {
                    if (un == 0) u.p0 = total + p;
#pragma unroll
                    for (int r = 0; r < FSX_UROWS; r++)
                        if (r == ur) {
                            u.g2[r] = g0 + b;
                            if (r % 4 == 0) u.cum[r / 4] = 0;
                            u.cum[r / 4] |= (unsigned)un << r % 4 * 8;
                        } else if (r > ur) {
                            u.g2[r] = u.g2[0];
                        }
                }
                ur++;
                un += k;
                p += k;
                left -= k;
            }
            rem--;
        }
    }
    if (un > 0) {
        if (PASS && lane == 0) {
            u.n = un;
            u.nrow = ur;
            units[first + uc] = u;
        }
        uc++;
    }
    if (!PASS && lane == 0) {
        grp[zb].x = p;
        grp[b2 * zn + z].y = uc;
        if (p > 0) {
            atomicAdd(&tail[0], p);
            atomicAdd(&tail[1], nz);
            atomicAdd(&tail[2], uc);
        }
    }
}

/* The groups' counts (grp of k_units<0>) to the sums of those before, in place, by
 * one block, four groups per thread and step. */
__global__ void __launch_bounds__(1024)
k_unit_scan(int2 *grp, int nzb)
{
    __shared__ int2 part[16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int2 base = make_int2(0, 0);
    for (long g0 = 0; g0 < nzb; g0 += 4096) {
        const long i0 = g0 + 4 * threadIdx.x;
        int2 v[4], s = make_int2(0, 0);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int2 c = i0 + k < nzb ? grp[i0 + k] : make_int2(0, 0);
            v[k] = s;
            s.x += c.x;
            s.y += c.y;
        }
        /* over the wavefront, then over the wavefronts */
        int2 x = s;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int a = __shfl_up(x.x, o), b = __shfl_up(x.y, o);
            if (lane >= o) {
                x.x += a;
                x.y += b;
            }
        }
        if (lane == 63) part[w] = x;
        __syncthreads();
        int2 all = base;
        for (int k = 0; k < 16; k++) {
            if (k == w) {
                x.x += all.x - s.x;
                x.y += all.y - s.y;
            }
            all.x += part[k].x;
            all.y += part[k].y;
        }
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (i0 + k < nzb) grp[i0 + k] = make_int2(x.x + v[k].x, x.y + v[k].y);
        base = all;
        __syncthreads();
    }
}

/* sorted pose records: x = input position, y = receptor row, z = alpha index,
 * w = gamma2 */
__global__ void k_scatter(const int *keys, const int2 *info, int n, int ng, const int *offs,
                          int *fill, int4 *recs)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int k = keys[i];
    if (k < 0) return;
    int p = offs[k] + atomicAdd(&fill[k], 1);
    int2 inf = info[i];
    recs[p] = make_int4(i, inf.x, inf.y, k % ng);
}

/* ---- per-pose fit, lockstep over a pose queue ------------------------------
 * Each lane owns one fit at a time.  All busy lanes of a wavefront evaluate
 * chi^2 and its gradient together (the same instruction stream over q), then
 * each advances its own L-BFGS-B state to the next point it needs; a lane
 * whose fit ended stores the result and takes the next pose from the queue.
 * Profiles: pose-major acc[(s*Q + q)*6 + k] plus the constant parts cint[k*Q
 * + q], rescaled by peak / I(q0) (min_saxs.c:170-179). */
/* Scale of each pose's profile, peak / I(q0) with I(q0) the six terms at
 * q index 0 summed as min_saxs.c:170-179 (one thread per pose slot). */
__global__ void k_fit_scale(const double *acc, const double *cint, const int *nvalid_p, int Q,
                            double peak, double *scale)
{
#pragma clang fp contract(off)
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= *nvalid_p) return;
    const double *v = acc + (long)s * Q * 6;
    double g[6];
    for (int k = 0; k < 6; k++) {
        double x = cint[k * Q];
        x = x + v[k];
        g[k] = x * 1.0;
    }
    const double sc = g[0] + g[3] + g[5] + g[2] - g[1] - g[4];
    scale[s] = peak / sc;
}

/* The fit's profiles, (constant part + pose part) * scale, in place of the
 * pose part, and the unscaled profiles to cross_out when asked; one thread
 * per (pose slot, q): its six terms, contiguous and 16-byte aligned, are read
 * and written as three pairs. */
/* accf (the mixed form's lane-group fit): the rescaled profiles in FP32 to
 * accf [pose][q][6] instead of in place */
__global__ void k_fit_prep(double *acc, const double *cint, const int4 *recs,
                           const int *nvalid_p, int Q, const double *scale, double *cross_out,
                           float *accf)
{
#pragma clang fp contract(off)
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)*nvalid_p * Q) return;
    const int s = (int)(i / Q), q = (int)(i - (long)s * Q);
    double2 *a2 = reinterpret_cast<double2 *>(acc + i * 6);
    double x[6];
#pragma unroll
    for (int h = 0; h < 3; h++) {
        const double2 p = a2[h];
        x[2 * h] = p.x;
        x[2 * h + 1] = p.y;
    }
#pragma unroll
    for (int k = 0; k < 6; k++) {
        double y = cint[k * Q + q];
        y = y + x[k];
        x[k] = y;
    }
    if (cross_out) {
        const long o = (long)recs[s].x * 6 * Q + q;
#pragma unroll
        for (int k = 0; k < 6; k++) cross_out[o + (long)k * Q] = x[k] * 1.0;
    }
    const double sc = scale[s];
    if (accf) {
        float2 *f2 = reinterpret_cast<float2 *>(accf + i * 6);
#pragma unroll
        for (int h = 0; h < 3; h++) f2[h] = make_float2((float)(x[2 * h] * sc), (float)(x[2 * h + 1] * sc));
        return;
    }
#pragma unroll
    for (int h = 0; h < 3; h++) a2[h] = make_double2(x[2 * h] * sc, x[2 * h + 1] * sc);
}

__device__ __forceinline__ void fit_begin(fsx_ct *t, fsx_lbrc *S, const fsx_fitpar *fp,
                                          const double *acc, int s, int Q)
{
    t->v = acc + (long)s * Q * 6;
    fsx_lb_start(S, fp, 1.0, 0.0);
}

/* LDS of one fit block (256 lanes): the L-BFGS-B K blocks, the sums of the
 * wavefront-wide evaluation (FSX_WIDE_SUMS x 64 per wavefront), then (when
 * they fit, aq_lds) the moments, the q grid and the reciprocals
 * 1/(q_i - q_{i-1}) */
#define FSX_FIT_LDS (160 * 1024)
#define FSX_WIDE_SUMS 3
static inline size_t fit_lds_k(void)
{
    return (size_t)(FSX_LB_KN * FSX_LB_KSTRIDE + 4 * FSX_WIDE_SUMS * 64) * sizeof(double);
}
static inline int fit_aq_lds(int Q) { return fit_lds_k() + 8 * (size_t)Q * sizeof(double) <= FSX_FIT_LDS; }
static inline size_t fit_lds(int Q) { return fit_lds_k() + (fit_aq_lds(Q) ? 8 * (size_t)Q * sizeof(double) : 0); }

/* lane l's value of v, l the same in every lane */
__device__ __forceinline__ double lane_d(double v, int l)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

/* LDS written by some lanes of this wavefront, read by others */
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

/* sums[c] += row c of sW (nq values, in order) in lane c < nc: the q-ordered
 * sums of the wide evaluation */
__device__ __forceinline__ void wide_sum(const double *sW, int nq, int nc, double *sum)
{
    const int lane = threadIdx.x & 63;
    if (lane < nc) {
        const double *row = sW + lane * 64;
        double c = *sum;
        int i = 0;
        for (; i + 8 <= nq; i += 8) {
            double t[8];
#pragma unroll
            for (int u = 0; u < 8; u++) t[u] = row[i + u];
#pragma unroll
            for (int u = 0; u < 8; u++) c = c + t[u];
        }
        for (; i < nq; i++) c = c + row[i];
        *sum = c;
    }
}

/* The six one-pass sums of the wide evaluation, two rows of three at a
 * time: terms tt[0..5] of this lane's q (rows 0..nq-1 used), added in q
 * order into sa (sums 0..2, lanes 0..2) and sb (sums 3..5, lanes 0..2). */
__device__ __forceinline__ void wide_sum6(double *sW, const double *tt, int nq, double *sa,
                                          double *sb)
{
    const int lane = threadIdx.x & 63;
    sW[lane] = tt[0];
    sW[64 + lane] = tt[1];
    sW[128 + lane] = tt[2];
    wave_lds_sync();
    wide_sum(sW, nq, 3, sa);
    wave_lds_sync();
    sW[lane] = tt[3];
    sW[64 + lane] = tt[4];
    sW[128 + lane] = tt[5];
    wave_lds_sync();
    wide_sum(sW, nq, 3, sb);
    wave_lds_sync();
}

/* The wide evaluation of the mixed-precision form's one-pass objective
 * (FSX_1P_TERMS): the profile of a fit is read once per evaluation and each
 * q's G is formed once.  Lane i holds q = 64 r + i in round r; the sums add
 * the terms in q order, as fsx_eval_1p_blk does, so the results are
 * bit-identical to the lane-per-fit evaluation's. */
__device__ __forceinline__ void fit_eval_wide_1p(unsigned long long amask, const double *acc,
                                                 int slot, const fsx_fitpar *fp, const double *x,
                                                 double *f, double *g, double *sW)
{
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63, Q = fp->qnum;
    const double *qv = fp->q, *av = fp->a, *rdq = fp->rdq;
    const double mult = fp->mult;
    if (Q <= 64) {
        const int qs = lane < Q ? lane : 0;
        const double qc = qv[qs], qp = qs > 0 ? qv[qs - 1] : -1.0;
        const double rq = rdq ? rdq[qs] : 1.0 / (qc - qp);
        const double *ai = av + qs * 6;
        double vn[6];
        auto load = [&](int jj) {
            const double2 *v2 = reinterpret_cast<const double2 *>(
                acc + ((long)__builtin_amdgcn_readlane(slot, jj) * Q + qs) * 6);
#pragma unroll
            for (int h = 0; h < 3; h++) {
                const double2 p = v2[h];
                vn[2 * h] = p.x;
                vn[2 * h + 1] = p.y;
            }
        };
        load(__builtin_ctzll(amask));
        while (amask) {
            const int j = __builtin_ctzll(amask);
            amask &= amask - 1;
            double v[6];
#pragma unroll
            for (int h = 0; h < 6; h++) v[h] = vn[h];
            if (amask) load(__builtin_ctzll(amask));
            const double c1 = lane_d(x[0], j), c2 = lane_d(x[1], j);
            const double corr = -mult * (c1 * c1 - 1.0), c1c = c1 * c1 * c1;
            const double r3c1 = 3.0 / c1, c1m2 = 2.0 * c1 * mult;
            const double G = c1c * exp(corr * qc * qc);
            const double Gd = G * (r3c1 - c1m2 * qc * qc);
            double in, d1, d2;
            FSX_OBJ_VALS(v, G, Gd, c2, in, d1, d2);
            double inp = __shfl_up(in, 1), d1p = __shfl_up(d1, 1), d2p = __shfl_up(d2, 1);
            if (lane == 0) {
                inp = in;
                d1p = d1;
                d2p = d2;
            }
            double tt[6];
            FSX_1P_TERMS(in, d1, d2, inp, d1p, d2p, rq, qc, ai, tt);
            double sa = 0.0, sb = 0.0;
            wide_sum6(sW, tt, Q, &sa, &sb);
            const double sm[6] = {lane_d(sa, 0), lane_d(sa, 1), lane_d(sa, 2),
                                  lane_d(sb, 0), lane_d(sb, 1), lane_d(sb, 2)};
            if (lane == j) fsx_1p_finish(sm, fp->a0sum, f, g);
        }
        return;
    }
    while (amask) {
        const int j = __builtin_ctzll(amask);
        amask &= amask - 1;
        const double c1 = lane_d(x[0], j), c2 = lane_d(x[1], j);
        const double *vp = acc + (long)__builtin_amdgcn_readlane(slot, j) * Q * 6;
        const double corr = -mult * (c1 * c1 - 1.0), c1c = c1 * c1 * c1;
        const double r3c1 = 3.0 / c1, c1m2 = 2.0 * c1 * mult;
        double in_l = 0.0, d1_l = 0.0, d2_l = 0.0, sa = 0.0, sb = 0.0;
        for (int r0 = 0; r0 < Q; r0 += 64) {
            const int nq = Q - r0 < 64 ? Q - r0 : 64, q = r0 + lane, ok = lane < nq;
            const int qs = ok ? q : r0;    /* a valid q for the unused lanes */
            const double2 *v2 = reinterpret_cast<const double2 *>(vp + (long)qs * 6);
            double v[6];
#pragma unroll
            for (int h = 0; h < 3; h++) {
                const double2 p = v2[h];
                v[2 * h] = p.x;
                v[2 * h + 1] = p.y;
            }
            const double qc = qv[qs], qp = qs > 0 ? qv[qs - 1] : -1.0;
            const double G = c1c * exp(corr * qc * qc);
            const double Gd = G * (r3c1 - c1m2 * qc * qc);
            double in, d1, d2;
            FSX_OBJ_VALS(v, G, Gd, c2, in, d1, d2);
            double inp = __shfl_up(in, 1), d1p = __shfl_up(d1, 1), d2p = __shfl_up(d2, 1);
            if (lane == 0) {
                inp = r0 == 0 ? in : in_l;
                d1p = r0 == 0 ? d1 : d1_l;
                d2p = r0 == 0 ? d2 : d2_l;
            }
            const double rq = rdq ? rdq[qs] : 1.0 / (qc - qp);
            double tt[6];
            FSX_1P_TERMS(in, d1, d2, inp, d1p, d2p, rq, qc, av + qs * 6, tt);
            wide_sum6(sW, tt, nq, &sa, &sb);
            in_l = lane_d(in, 63);
            d1_l = lane_d(d1, 63);
            d2_l = lane_d(d2, 63);
        }
        const double sm[6] = {lane_d(sa, 0), lane_d(sa, 1), lane_d(sa, 2),
                              lane_d(sb, 0), lane_d(sb, 1), lane_d(sb, 2)};
        if (lane == j) fsx_1p_finish(sm, fp->a0sum, f, g);
    }
}

/* Evaluation of the fits of the lanes in amask (all of this wavefront) by
 * the whole wavefront, one fit at a time: lane i holds q = 64 r + i in
 * round r, forms that q's terms (FSX_BS_TERMS, FSX_OBJ_VALS, FSX_OBJ_TERMS,
 * with the previous q's values from its neighbour lane) and writes them to
 * sW; lane c then adds row c to its running sum in q order.  Every value is
 * therefore formed by the operations of the sequential loop and every sum
 * adds the same terms in the same order: the results are bit-identical to
 * lb_eval's.  x, slot: each lane's point and profile slot; f, g: the results
 * of lane j land in lane j. */
template <int ONEP>
__device__ __forceinline__ void fit_eval_wide(unsigned long long amask, const double *acc, int slot,
                              const fsx_fitpar *fp, const double *x, double *f, double *g,
                              double *sW)
{
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63, Q = fp->qnum;
    const double *qv = fp->q, *av = fp->a, *rdq = fp->rdq;
    const double mult = fp->mult;
    if (ONEP) {
        fit_eval_wide_1p(amask, acc, slot, fp, x, f, g, sW);
        return;
    }
    if (Q <= 64) {
        /* one round: each lane's q, its neighbour and 1/(q - q_prev) once;
         * the profile of a fit read once for both passes (the next fit's
         * read issued before this one's sums); G and I of the scale pass
         * reused by the objective */
        const int qs = lane < Q ? lane : 0;
        const double qc = qv[qs], qp = qs > 0 ? qv[qs - 1] : -1.0;
        const double rq = rdq ? rdq[qs] : 1.0 / (qc - qp);
        const double *ai = av + qs * 6;
        double vn[6];
        auto load = [&](int jj) {
            const double2 *v2 = reinterpret_cast<const double2 *>(
                acc + ((long)__builtin_amdgcn_readlane(slot, jj) * Q + qs) * 6);
#pragma unroll
            for (int h = 0; h < 3; h++) {
                const double2 p = v2[h];
                vn[2 * h] = p.x;
                vn[2 * h + 1] = p.y;
            }
        };
        load(__builtin_ctzll(amask));
        while (amask) {
            const int j = __builtin_ctzll(amask);
            amask &= amask - 1;
            double v[6];
#pragma unroll
            for (int h = 0; h < 6; h++) v[h] = vn[h];
            if (amask) load(__builtin_ctzll(amask));
            const double c1 = lane_d(x[0], j), c2 = lane_d(x[1], j);
            const double corr = -mult * (c1 * c1 - 1.0), c1c = c1 * c1 * c1;
            const double G = c1c * exp(corr * qc * qc);
            const double in = FSX_IN(v, G, c2);
            double inp = __shfl_up(in, 1);
            if (lane == 0) inp = in;
            double ut, dt;
            FSX_BS_TERMS(in, inp, qc, qp, ai, ut, dt);
            sW[lane] = ut;
            sW[64 + lane] = dt;
            wave_lds_sync();
            double sum = 0.0;
            wide_sum(sW, Q, 2, &sum);
            wave_lds_sync();
            const double k = lane_d(sum, 0) / lane_d(sum, 1);
            const double r3c1 = 3.0 / c1, c1m2 = 2.0 * c1 * mult;
            const double Gd = G * (r3c1 - c1m2 * qc * qc);
            double in2, d1, d2;
            FSX_OBJ_VALS(v, G, Gd, c2, in2, d1, d2);
            double d1p = __shfl_up(d1, 1), d2p = __shfl_up(d2, 1);
            inp = __shfl_up(in2, 1);
            if (lane == 0) {
                /* the values before the loop (min_saxs.c:28-41) */
                inp = FSX_IN(v, G, c2);
                d1p = -Gd * v[1] + 2.0 * G * Gd * v[3] - Gd * c2 * v[4];
                d2p = v[2] - G * v[4] + 2.0 * c2 * v[5];
            }
            double tg0, tg1, tsc;
            FSX_OBJ_TERMS(in2, d1, d2, inp, d1p, d2p, rq, qc, ai, k, tg0, tg1, tsc);
            sW[lane] = tg0;
            sW[64 + lane] = tg1;
            sW[128 + lane] = tsc;
            wave_lds_sync();
            sum = 0.0;
            wide_sum(sW, Q, 3, &sum);
            wave_lds_sync();
            const double g0 = lane_d(sum, 0), g1 = lane_d(sum, 1), sc = lane_d(sum, 2);
            if (lane == j) {
                g[0] = g0;
                g[1] = g1;
                *f = sc;
            }
        }
        return;
    }
    while (amask) {
        const int j = __builtin_ctzll(amask);
        amask &= amask - 1;
        const double c1 = lane_d(x[0], j), c2 = lane_d(x[1], j);
        const double *vp = acc + (long)__builtin_amdgcn_readlane(slot, j) * Q * 6;
        const double corr = -mult * (c1 * c1 - 1.0), c1c = c1 * c1 * c1;
        /* scale pass (min_saxs.c:261-319): up, down in lanes 0, 1 */
        double sum = 0.0, in_last = 0.0;
        for (int r0 = 0; r0 < Q; r0 += 64) {
            const int nq = Q - r0 < 64 ? Q - r0 : 64, q = r0 + lane, ok = lane < nq;
            const int qs = ok ? q : r0;    /* a valid q for the unused lanes */
            const double2 *v2 = reinterpret_cast<const double2 *>(vp + (long)qs * 6);
            double v[6];
#pragma unroll
            for (int h = 0; h < 3; h++) {
                const double2 p = v2[h];
                v[2 * h] = p.x;
                v[2 * h + 1] = p.y;
            }
            const double qc = qv[qs], qp = qs > 0 ? qv[qs - 1] : -1.0;
            const double G = c1c * exp(corr * qc * qc);
            const double in = FSX_IN(v, G, c2);
            double inp = __shfl_up(in, 1);
            if (lane == 0) inp = r0 == 0 ? in : in_last;
            double ut, dt;
            FSX_BS_TERMS(in, inp, qc, qp, av + qs * 6, ut, dt);
            sW[lane] = ut;
            sW[64 + lane] = dt;
            wave_lds_sync();
            wide_sum(sW, nq, 2, &sum);
            wave_lds_sync();
            in_last = lane_d(in, 63);
        }
        const double up = lane_d(sum, 0), down = lane_d(sum, 1);
        const double k = up / down;
        /* objective (min_saxs.c:3-105): g0, g1, score in lanes 0, 1, 2 */
        const double r3c1 = 3.0 / c1, c1m2 = 2.0 * c1 * mult;
        double in_l = 0.0, d1_l = 0.0, d2_l = 0.0;
        sum = 0.0;
        for (int r0 = 0; r0 < Q; r0 += 64) {
            const int nq = Q - r0 < 64 ? Q - r0 : 64, q = r0 + lane, ok = lane < nq;
            const int qs = ok ? q : r0;
            const double2 *v2 = reinterpret_cast<const double2 *>(vp + (long)qs * 6);
            double v[6];
#pragma unroll
            for (int h = 0; h < 3; h++) {
                const double2 p = v2[h];
                v[2 * h] = p.x;
                v[2 * h + 1] = p.y;
            }
            const double qc = qv[qs], qp = qs > 0 ? qv[qs - 1] : -1.0;
            const double G = c1c * exp(corr * qc * qc);
            const double Gd = G * (r3c1 - c1m2 * qc * qc);
            double in, d1, d2;
            FSX_OBJ_VALS(v, G, Gd, c2, in, d1, d2);
            double inp = __shfl_up(in, 1), d1p = __shfl_up(d1, 1), d2p = __shfl_up(d2, 1);
            if (lane == 0) {
                if (r0 == 0) {
                    /* the values before the loop (min_saxs.c:28-41) */
                    inp = FSX_IN(v, G, c2);
                    d1p = -Gd * v[1] + 2.0 * G * Gd * v[3] - Gd * c2 * v[4];
                    d2p = v[2] - G * v[4] + 2.0 * c2 * v[5];
                } else {
                    inp = in_l;
                    d1p = d1_l;
                    d2p = d2_l;
                }
            }
            const double rq = rdq ? rdq[qs] : 1.0 / (qc - qp);
            double tg0, tg1, tsc;
            FSX_OBJ_TERMS(in, d1, d2, inp, d1p, d2p, rq, qc, av + qs * 6, k, tg0, tg1, tsc);
            sW[lane] = tg0;
            sW[64 + lane] = tg1;
            sW[128 + lane] = tsc;
            wave_lds_sync();
            wide_sum(sW, nq, 3, &sum);
            wave_lds_sync();
            in_l = lane_d(in, 63);
            d1_l = lane_d(d1, 63);
            d2_l = lane_d(d2, 63);
        }
        const double g0 = lane_d(sum, 0), g1 = lane_d(sum, 1), sc = lane_d(sum, 2);
        if (lane == j) {
            g[0] = g0;
            g[1] = g1;
            *f = sc;
        }
    }
}

template <int AQ_LDS, int ONEP>
__global__ void __launch_bounds__(256)
k_fit(const double *acc, const int4 *recs, const int *nvalid_p, int Q, const double *qvals,
      const double *a, double mult, double c1_lo, double c1_hi, double c2_lo, double c2_hi,
      double *score, double *c1o, double *c2o, int *next, unsigned long long *tally,
      int wide_max, int fpw)
{
#pragma clang fp contract(off)
    /* LDS: the K blocks [FSX_LB_KN][256], the wide evaluation's sums
     * [4 wavefronts][FSX_WIDE_SUMS][64], then a [6][Q], q [Q] and
     * 1/(q_i - q_{i-1}) [Q] when aq_lds (read by every lane at the same
     * address); otherwise a and q are read from global memory and the
     * reciprocals formed per step */
    extern __shared__ double sKf[];
    double *sW = sKf + FSX_LB_KN * FSX_LB_KSTRIDE + (threadIdx.x >> 6) * FSX_WIDE_SUMS * 64;
    const int nvalid = *nvalid_p;
    /* each wavefront starts with fpw fits in its first lanes */
    const int lane0 = threadIdx.x & 63;
    int s = lane0 < fpw ? (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6) * fpw + lane0 : nvalid;
    fsx_fitpar fp;
    if (AQ_LDS) {
        double *sA = sKf + FSX_LB_KN * FSX_LB_KSTRIDE + 4 * FSX_WIDE_SUMS * 64;
        double *sQ = sA + 6 * Q, *sR = sQ + Q;
        for (int i = threadIdx.x; i < 6 * Q; i += blockDim.x) sA[i] = a[i];
        for (int i = threadIdx.x; i < Q; i += blockDim.x) {
            const double qc = qvals[i];
            sQ[i] = qc;
            sR[i] = 1.0 / (qc - (i > 0 ? qvals[i - 1] : -1.0));
        }
        __syncthreads();
        fp.a = sA; fp.q = sQ; fp.rdq = sR;
    } else {
        fp.a = a; fp.q = qvals; fp.rdq = NULL;
    }
    fp.qnum = Q; fp.mult = mult;
    fp.lo0 = c1_lo; fp.hi0 = c1_hi; fp.lo1 = c2_lo; fp.hi1 = c2_hi;
    fp.factr = 1e+7; fp.pgtol = 1e-5;
    fp.onepass = ONEP;
    fp.a0sum = ONEP ? fsx_a0sum(fp.a, Q) : 0.0;
    /* profiles already rescaled in place (k_fit_prep) */
    fsx_ct t;
    t.c = NULL; t.cks = 0; t.cqs = 0;
    t.v = acc; t.vks = 1; t.vqs = 6;
    t.scale = 1.0;
    fsx_lbrc S;
    S.w.kb = sKf + threadIdx.x;
    unsigned long long nev = 0, ncap = 0, steps = 0, wsteps = 0;
    int act = s < nvalid;
    int pose = act ? recs[s].x : 0;
    if (act) fit_begin(&t, &S, &fp, acc, s, Q);
    while (__any(act)) {
        /* once the queue is empty and at most wide_max lanes of the
         * wavefront still fit, the wavefront evaluates their fits together
         * (q across the lanes) instead of each lane running its whole q loop */
        const unsigned long long amask = __ballot(act);
        steps++;
        if (__popcll(amask) <= wide_max) {
            wsteps++;
            fit_eval_wide<ONEP>(amask, acc, s, &fp, S.x, &S.f, S.g, sW);
        } else if (act) {
            if (ONEP) {
                lb_eval_1p(&t, &fp, S.x, &S.f, S.g);
            } else {
                double k;
                lb_eval(&t, &fp, S.x, &S.f, S.g, &k);
            }
        }
        if (act && !fsx_lb_resume(&S)) {
            score[pose] = sqrt(S.f);
            c1o[pose] = S.x[0];
            c2o[pose] = S.x[1];
            nev += S.nev;
            ncap += S.task == FSX_T_STOP_ITER;
            s = atomicAdd(next, 1);
            act = s < nvalid;
            if (act) {
                pose = recs[s].x;
                fit_begin(&t, &S, &fp, acc, s, Q);
            }
        }
    }
    if (nev) atomicAdd(&tally[0], nev);
    if (ncap) atomicAdd(&tally[1], ncap);
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&tally[2], steps);
        atomicAdd(&tally[3], wsteps);
        atomicMax(&tally[4], steps);
    }
}

/* ---------------------------------------------------------------------- */
/* The mixed-precision form's fit: the two-variable L-BFGS-B of fsx_lb2.h
 * (the reference's steps with the 2 x 2 L-BFGS matrix held explicitly),
 * one pose per group of fpl lanes (a power of two).  Lane j of a group
 * evaluates the q range [j qpl, (j + 1) qpl), qpl = ceil(Q / fpl), reading
 * the pose's profile at each evaluation (one-pass form, fsx_lbfgsb.h
 * FSX_1P_TERMS): its six sums run in q order from its second q on, its
 * first q pairs with the previous lane's last (a lane shift), and the sums
 * meet by an xor butterfly, after which every lane of the group holds the
 * same value and gradient and runs the same solver step.  Between steps the
 * solver state lives in LDS, one copy per group (every lane of the group
 * writes the same values), so that the kernel fits in 128 registers with
 * 144 bytes of spills (reloaded once per evaluation or per fit, none in the
 * loop over q): four wavefronts per SIMD, against one for the
 * compact form's state (on the 210,000-pose L = 15 workload 1.50 ms,
 * against 1.60 ms at three wavefronts in 168 registers without spills).
 * With eight lanes per fit (33 to 64 q, fsx_fit_lanes) a wavefront runs 8 fits, so
 * the solver's divergent code is shared by several fits while the evaluation of
 * each, whose chain bounds all but the longest lists, is split eight ways.  The
 * moments, q and the step reciprocals sit in LDS, slot
 * ii * fpl + j for q = j qpl + ii, so the lanes of a group read consecutive
 * doubles.  Groups take poses from a queue (next) until none is left. */
#define FSX_FG_ARR 8     /* LDS arrays: a0..a5, q, 1 / (q_i - q_{i-1}) */
#ifndef FSX_FG_WAVES
#define FSX_FG_WAVES 4   /* wavefronts per SIMD (the register budget of the launch bounds) */
#endif

__device__ __forceinline__ void fitg_eval(const float *pr, const double *sNt, int ns, int qpl,
                                          int fpl, int j, int Q, double mult, double a0sum,
                                          const double *x, double *fv, double *g)
{
#pragma clang fp contract(fast)
    const double c1 = x[0], c2 = x[1];
    const double corr = -mult * (c1 * c1 - 1.0), c1c = c1 * c1 * c1;
    const int q0 = j * qpl, nq = Q - q0 < qpl ? Q - q0 : qpl;
    double s[6];
#pragma unroll
    for (int k = 0; k < 6; k++) s[k] = 0.0;
    double vf[3] = {0.0, 0.0, 0.0}, vp[3] = {0.0, 0.0, 0.0};
    /* the sums' terms of step ii from I and its derivatives there (vv) and
     * at the previous q (pp) */
    auto terms_at = [&](const double *vv, const double *pp, int ii) {
        const int slot = ii * fpl + j;
        double ai[6], tt[6];
#pragma unroll
        for (int k = 0; k < 6; k++) ai[k] = sNt[k * ns + slot];
        FSX_1P_TERMS(vv[0], vv[1], vv[2], pp[0], pp[1], pp[2], sNt[7 * ns + slot],
                     sNt[6 * ns + slot], ai, tt);
#pragma unroll
        for (int k = 0; k < 6; k++) s[k] += tt[k];
    };
    for (int ii = 0; ii < nq; ii++) {
        const float2 *p2 = reinterpret_cast<const float2 *>(pr + 6 * (q0 + ii));
        const float2 a = p2[0], b = p2[1], c = p2[2];
        const double cur[6] = {a.x, a.y, b.x, b.y, c.x, c.y};
        /* I and its derivatives in c1, c2 (min_saxs.c:52-68) */
        const double qc = sNt[6 * ns + ii * fpl + j];
        const double G = c1c * exp(corr * qc * qc);
        const double Gd = G * (3.0 / c1 - 2.0 * c1 * mult * qc * qc);
        double vv[3];
        FSX_OBJ_VALS(cur, G, Gd, c2, vv[0], vv[1], vv[2]);
        if (ii == 0) {
#pragma unroll
            for (int k = 0; k < 3; k++) vf[k] = vv[k];
        } else {
            terms_at(vv, vp, ii);
        }
#pragma unroll
        for (int k = 0; k < 3; k++) vp[k] = vv[k];
    }
    /* the first q of a lane pairs with the previous lane's last (lane 0:
     * q = 0 with itself, slope 0, as min_saxs.c:30-35 starts) */
    double pl[3];
#pragma unroll
    for (int k = 0; k < 3; k++) pl[k] = __shfl_up(vp[k], 1, fpl);
    if (nq > 0) terms_at(vf, j == 0 ? vf : pl, 0);
    for (int o = 1; o < fpl; o <<= 1) {
#pragma unroll
        for (int k = 0; k < 6; k++) s[k] += __shfl_xor(s[k], o, fpl);
    }
    fsx_1p_finish(s, a0sum, fv, g);
}

__device__ __forceinline__ void
fitg_body(const float *acc, const int4 *recs, const int *nvalid_p, int Q, const double *qvals,
          const double *a, double mult, double c1_lo, double c1_hi, double c2_lo, double c2_hi,
          double *score, double *c1o, double *c2o, int *next, unsigned long long *tally, int fpl)
{
    extern __shared__ double sNt[];
    const int qpl = (Q + fpl - 1) / fpl;
    const int ns = qpl * fpl;
    fsx_lb2 *sSt = reinterpret_cast<fsx_lb2 *>(sNt + FSX_FG_ARR * ns);
    for (int i = threadIdx.x; i < ns; i += blockDim.x) {
        const int q = (i % fpl) * qpl + i / fpl;
        const bool ok = q < Q;
#pragma unroll
        for (int k = 0; k < 6; k++) sNt[k * ns + i] = ok ? a[6 * q + k] : 0.0;
        sNt[6 * ns + i] = ok ? qvals[q] : 0.0;
        /* min_saxs.c:60: 1 / (q_i - q_{i-1}) with q_{-1} = -1 */
        sNt[7 * ns + i] = ok ? 1.0 / (qvals[q] - (q > 0 ? qvals[q - 1] : -1.0)) : 0.0;
    }
    __syncthreads();
    fsx_fitpar fp;
    fp.lo0 = c1_lo; fp.hi0 = c1_hi; fp.lo1 = c2_lo; fp.hi1 = c2_hi;
    fp.factr = 1e+7; fp.pgtol = 1e-5;
    const double a0sum = fsx_a0sum(a, Q);
    const int nvalid = *nvalid_p;
    const int lane = threadIdx.x & (FSX_WAVE - 1), j = lane & (fpl - 1);
    const int leader = lane & ~(fpl - 1);
    int s = (int)(((long)blockIdx.x * blockDim.x + threadIdx.x) / fpl);
    unsigned long long nev = 0, ncap = 0, nmax = 0;
    fsx_lb2 *S = sSt + threadIdx.x / fpl;
    while (s < nvalid) {
        const float *pr = acc + (long)s * 6 * Q;
        fsx_lb2_start(S, &fp, 1.0, 0.0);   /* define.h:33-34 */
        int more;
        do {
            double xt[2] = {S->x[0], S->x[1]}, fv, gv[2];
            /* the state is read back from LDS after the evaluation rather
             * than kept in registers across it */
            asm volatile("" ::: "memory");
            fitg_eval(pr, sNt, ns, qpl, fpl, j, Q, mult, a0sum, xt, &fv, gv);
            asm volatile("" ::: "memory");
            S->f = fv;
            S->g[0] = gv[0];
            S->g[1] = gv[1];
            more = fsx_lb2_resume(S, &fp);
        } while (more);
        if (j == 0) {
            const int o = recs ? recs[s].x : s;
            score[o] = sqrt(S->f);
            c1o[o] = S->x[0];
            c2o[o] = S->x[1];
        }
        nev += S->nev;
        ncap += S->task == FSX_T_STOP_ITER;
        nmax = nmax > (unsigned long long)S->nev ? nmax : (unsigned long long)S->nev;
        int sn = 0;
        if (j == 0) sn = atomicAdd(next, 1);
        s = __shfl(sn, leader, FSX_WAVE);
    }
    if (j == 0) {
        /* evaluations; fits stopped at the evaluation cap; evaluations again
         * as the loop count of the lane groups; none wavefront-wide; the
         * longest fit's evaluations */
        if (nev) {
            atomicAdd(&tally[0], nev);
            atomicAdd(&tally[2], nev);
        }
        if (ncap) atomicAdd(&tally[1], ncap);
        if (nmax) atomicMax(&tally[4], nmax);
    }
}

__global__ void __launch_bounds__(256, FSX_FG_WAVES)
k_fitg(const float *acc, const int4 *recs, const int *nvalid_p, int Q, const double *qvals,
       const double *a, double mult, double c1_lo, double c1_hi, double c2_lo, double c2_hi,
       double *score, double *c1o, double *c2o, int *next, unsigned long long *tally, int fpl)
{
    fitg_body(acc, recs, nvalid_p, Q, qvals, a, mult, c1_lo, c1_hi, c2_lo, c2_hi, score, c1o,
              c2o, next, tally, fpl);
}

/* The fits of several complexes in one persistent launch (the batched
 * form): every block runs the lane groups of job 0 until its pose queue is
 * empty, then those of job 1, and so on (each job with its own queue, q
 * grid, moments, bounds and lanes per fit). */
struct fsx_fit_job {
    const float *acc;
    const double *qvals, *a;
    const int4 *recs;
    const int *nvalid_p;
    double mult, c1_lo, c1_hi, c2_lo, c2_hi;
    double *score, *c1o, *c2o;
    int *next;
    unsigned long long *tally;
    int Q, fpl;
};

__global__ void __launch_bounds__(256, FSX_FG_WAVES)
k_fitg_jobs(const fsx_fit_job *jobs, int njobs)
{
    for (int k = 0; k < njobs; k++) {
        const fsx_fit_job &jb = jobs[k];
        fitg_body(jb.acc, jb.recs, jb.nvalid_p, jb.Q, jb.qvals, jb.a, jb.mult, jb.c1_lo,
                  jb.c1_hi, jb.c2_lo, jb.c2_hi, jb.score, jb.c1o, jb.c2o, jb.next, jb.tally,
                  jb.fpl);
        /* the next job refills the LDS arrays */
        __syncthreads();
    }
}

/* LDS of a k_fitg block: the moment arrays and one solver state per group */
static inline size_t fitg_lds(int Q, int fpl)
{
    const size_t qpl = ((size_t)Q + fpl - 1) / fpl;
    return (size_t)FSX_FG_ARR * qpl * fpl * sizeof(double) + (size_t)(256 / fpl) * sizeof(fsx_lb2);
}

/* fits of caller-supplied (rescaled) profiles ct[n][6][Q] */
__global__ void __launch_bounds__(256)
k_fit_batch(const double *ct, int n, const double *qvals, int Q, const double *a, double mult,
            double c1_lo, double c1_hi, double c2_lo, double c2_hi, double *out)
{
#pragma clang fp contract(off)
    extern __shared__ double sKb[];   /* K blocks [FSX_LB_KN][256] */
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    fsx_ct t;
    t.c = ct + (long)s * 6 * Q; t.cks = Q; t.cqs = 1;
    t.v = NULL; t.vks = 0; t.vqs = 0; t.scale = 1.0;
    fsx_fitpar fp;
    fp.a = a; fp.q = qvals; fp.rdq = NULL; fp.qnum = Q; fp.mult = mult;
    fp.lo0 = c1_lo; fp.hi0 = c1_hi; fp.lo1 = c2_lo; fp.hi1 = c2_hi;
    fp.factr = 1e+7; fp.pgtol = 1e-5;
    fp.onepass = 0; fp.a0sum = 0.0;
    double x[2] = {1.0, 0.0}, f;
    int nev;
    fsx_lbfgsb_fit(&t, &fp, x, &f, &nev, sKb + threadIdx.x);
    out[4L * s] = sqrt(f);
    out[4L * s + 1] = x[0];
    out[4L * s + 2] = x[1];
    out[4L * s + 3] = nev;
}

/* ---- atom expansion (pdb2spf.c:24-152) ------------------------------------
 * A^X_lm(q) = 4 pi i^l sum_a f^X_a j_l(q r_a) conj(Y_lm(theta_a, phi_a)) for
 * X = V, D, W (f^V, f^D the scalar form factors, f^W = zero_ff(OH2) * SASA).
 * With real f, conj(Y_{l,-m}) = (-1)^m Y_lm, so the sums are formed for
 * m >= 0 only and A_{l,-m} = (-1)^m 4 pi i^l conj(S_lm), S_lm the m >= 0 sum.
 * Stages, per pass over a range of atoms:
 *   k_atom_geom   r, f^X and conj(Y_lm) (m >= 0) per atom, the reference's
 *                 angles (cart2sph), norms and Legendre recurrence
 *                 (borrowed.c:19-65), contraction off
 *   k_atom_bes    J[l][q][atom] = j_l(q r) by the reference's series
 *   k_atom_mfma   per (chunk of 1024 atoms, l, up to 4 column and 3 q tiles of
 *                 16): the sums over the chunk's
 *                 atoms as FP64 MFMA products of the (q x atoms) Bessel tile and
 *                 the (atoms x (X, m, re/im)) tile f^X conj(Y_lm); four waves
 *                 take 256 atoms each and are summed in LDS in a fixed order;
 *                 one partial per chunk
 * then k_atom_finish sums the chunks in order and applies 4 pi i^l. */
#define FSX_AT_CHUNK 1024   /* atoms per k_atom_mfma block (4 waves x 256) */
#define FSX_AT_MAXT 16      /* most column tiles of an l: 3 * 2 (L + 1) <= 16 * 16 for L <= 41 */

/* A thread per (atom, m), the m of an atom side by side so that the entries of
 * an l go out together (a thread per atom filled 39 CUs with 10,000 atoms: 176 us
 * at L = 25, 52 now). */
__global__ void __launch_bounds__(256)
k_atom_geom(const double *xyz, const double *vac, const double *dum, const double *sa, double h2o_ff,
            int na, int L, double pi_ref, double *r_out, double *f_out, double *Y)
{
#pragma clang fp contract(off)
    const int N = L + 1, Kh = N * (N + 1) / 2;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int a = (int)(i / N), m = (int)(i - (long)a * N);
    if (a >= na) return;
    /* cart2sph (pdb2spf.c:9-22) */
    const double x = xyz[3 * (size_t)a], y = xyz[3 * (size_t)a + 1], z = xyz[3 * (size_t)a + 2];
    const double rr = sqrt(x * x + y * y + z * z);
    const double th = acos(z / rr);
    double fi;
    if (y > 0.0) fi = acos(x / sqrt(x * x + y * y));
    else fi = -acos(x / sqrt(x * x + y * y)) + 2.0 * pi_ref;
    if (m == 0) {
        r_out[a] = rr;
        f_out[a] = vac[a];
        f_out[na + a] = dum[a];
        f_out[2 * na + a] = sa ? h2o_ff * sa[a] : 0.0;
    }
    /* associated Legendre values (borrowed.c:40-65), written as conj(Y_lm)
     * = yn(l, m) P_l^m (cos m phi, sin(-m phi)) as soon as each is formed;
     * yn(l, m) = sqrt((2l + 1) / (4 pi) / prod_{k=1..m} (l - k + 1)(l + k))
     * (borrowed.c:19-38) */
    double *Ya = Y + (size_t)a * Kh * 2;
    const double xc = cos(th), yc = sqrt(1. - xc * xc);
    const double cm = cos(fi * m), sm = sin(-fi * m);
    /* the diagonal, then upwards in l */
    double pmm = 1.0;
    for (int k = 1; k <= m; k++) pmm = -1. * (2. * k - 1.) * yc * pmm;
    double q2 = 0.0, q1 = 0.0;
    for (int l = 0; l < N; l++) {
        if (l < m) continue;
        const double p = l == m ? pmm
                       : l == m + 1 ? (2. * m + 1.) * xc * q1
                                    : (2. * l - 1.) / (l - m) * xc * q1 - (l + m - 1.) / (l - m) * q2;
        q2 = q1;
        q1 = p;
        double f = 1.;
        const double base = (2 * l + 1.) / (4. * pi_ref);
        for (int k = 1; k <= m; k++) f *= (l - k + 1) * (l + k);
        const double h = sqrt(base / f) * p;
        const int e = l * (l + 1) / 2 + m;
        Ya[2 * e] = h * cm;
        Ya[2 * e + 1] = h * sm;
    }
}

/* The series of dev_sbessel for the threads of a block that share l, bit for bit
 * and without its divisions: begin() tabulates the denominators d = 2k (2k + 2l +
 * 1) and their rounded reciprocals y for k <= FSX_SB_TAB and 1 / (2l + 1)!!.
 * - The quotient n / d: q = n y, and twice q += (n - d q) y with fused
 *   multiply-adds.  The first leaves q within one unit in the last place, and
 *   from such a q and a correctly rounded y the second gives the correctly
 *   rounded quotient (Markstein 1990), 5 operations for the division's dozen.
 *   A residual that underflows belongs to a ratio far below the sum's last bit.
 * - The test |term / sum| > 1e-5: by products with margins a million times the
 *   rounding error; the division decides only in between.
 * Bound by the FP64 instructions of the terms (about 15 for each, up to 40 terms)
 * and of x^l: 10,000 atoms, L = 25, 81 q 737 us with the divisions and q across the
 * lanes, 350 now (60 G values/s). */
#define FSX_SB_TAB 64
struct sbessel_block {
    double d[FSX_SB_TAB + 1], y[FSX_SB_TAB + 1], t0;
    __device__ __forceinline__ void begin(int l)
    {
#pragma clang fp contract(off)
        const int k = threadIdx.x;
        const double tl1 = 2.0 * (double)l + 1.0;
        if (k >= 1 && k <= FSX_SB_TAB) {
            d[k] = 2.0 * (double)k * (2.0 * (double)k + tl1);
            y[k] = 1.0 / d[k];
        }
        if (k == 0) {
            double f = 1.0;
            for (int i = 1; i <= (int)tl1; i += 2) f *= (double)i;
            t0 = 1.0 / f;
        }
        __syncthreads();
    }
    __device__ __forceinline__ double value(int l, double x) const
    {
#pragma clang fp contract(off)
        if (!(x > 0.0)) return l == 0 ? 1.0 : 0.0;
        const double tl1 = 2.0 * (double)l + 1.0, n = (-1.0) * x * x;
        double term = t0, sum = t0;
        for (int k = 1;; k++) {
            const double at = fabs(term), as = fabs(sum);
            if (!(at > fma(as, 0.00001 * (1.0 + 1e-9), 1e-290))) {
                if (as > 1e-270 && at < as * (0.00001 * (1.0 - 1e-9))) break;
                if (!(fabs(term / sum) > 0.00001)) break;
            }
            double ratio;
            if (k <= FSX_SB_TAB) {
                ratio = n * y[k];
                ratio = fma(fma(-d[k], ratio, n), y[k], ratio);
                ratio = fma(fma(-d[k], ratio, n), y[k], ratio);
            } else {
                ratio = n / (2.0 * (double)k * (2.0 * (double)k + tl1));
            }
            term *= ratio;
            sum += term;
        }
        return sum * pow_int_cr(x, l);
    }
};

/* J[l][q][a] = j_l(q r_a); nbl blocks per l.  A wavefront takes atoms of one q,
 * whose series have about the same length (with q across the lanes all of them
 * waited for the largest q: 532 against 350 us at 10,000 atoms, L = 25, 81 q). */
__global__ void __launch_bounds__(256)
k_atom_bes(double *J, const double *r, const double *qvals, int na, int Q, unsigned nbl)
{
    __shared__ sbessel_block S;
    const int l = (int)(blockIdx.x / nbl);
    S.begin(l);
    const long i = (long)(blockIdx.x % nbl) * blockDim.x + threadIdx.x, n = (long)na * Q;
    if (i >= n) return;
    const int q = (int)(i / na), a = (int)(i - (long)q * na);
    J[l * n + i] = S.value(l, qvals[q] * r[a]);
}

/* One block of four waves per (chunk, l, up to FSX_AT_CT column tiles, up to
 * FSX_AT_QT q tiles), tiles of 16.  Rows are q, columns
 * c = X * 2(l+1) + 2m + part (part 0: real, 1: imaginary) of f^X conj(Y_lm).
 * FP64 MFMA 16x16x4 operand layout on gfx950: lane i feeds A[i % 16][i / 16]
 * and B[i / 16][i % 16]; result register j of lane i is D[i / 16 + 4j][i % 16].
 * A step's QT + 2 CT loads feed QT CT products, with the next step's in flight
 * (with one q tile and every column tile in a block, f and Y were read for each
 * q tile and waited for at each step: 539 us for 10,000 atoms, L = 25, 81 q,
 * against 133 to 157; the products alone take 96 at their measured rate).
 * Writes the chunk's partial sums P[chunk][X][Qp][Kh][2]. */
#define FSX_AT_QT 3
#define FSX_AT_CT 4
__host__ __device__ static inline int at_colgroups(int l)
{
    return (6 * (l + 1) + 16 * FSX_AT_CT - 1) / (16 * FSX_AT_CT);
}
__global__ void __launch_bounds__(256, 2)
k_atom_mfma(const double *J, const double *f, const double *Y, double *P, int na, int Q, int Qp, int L,
            int chunk0)
{
    __shared__ fsx_v4d red[3][64];
    const int K = L + 1, Kh = K * (K + 1) / 2, nqt = Qp / 16;
    const int nqg = (nqt + FSX_AT_QT - 1) / FSX_AT_QT;
    int bid = blockIdx.x, ncg = 0;
    for (int l = 0; l <= L; l++) ncg += at_colgroups(l);
    const int qt0 = bid % nqg * FSX_AT_QT;
    bid /= nqg;
    const int ch = bid / ncg;
    /* the orders with the most columns first */
    int cg = bid - ch * ncg, l = L;
    while (cg >= at_colgroups(l)) cg -= at_colgroups(l--);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int ncol = 3 * 2 * (l + 1);
    const int nq = min(FSX_AT_QT, nqt - qt0);
    const int nc = min(FSX_AT_CT, (ncol + 15) / 16 - cg * FSX_AT_CT);
    /* this lane's column of each tile: X (-1: none), entry offset and part */
    int cx[FSX_AT_CT], coff[FSX_AT_CT];
#pragma unroll
    for (int t = 0; t < FSX_AT_CT; t++) {
        const int c = (cg * FSX_AT_CT + t) * 16 + (lane & 15);
        const int X = c / (2 * (l + 1)), rem = c - X * 2 * (l + 1);
        cx[t] = c < ncol ? X : -1;
        coff[t] = c < ncol ? l * (l + 1) / 2 * 2 + rem : 0;   /* (entry, part) as a double index */
    }
    fsx_v4d acc[FSX_AT_QT][FSX_AT_CT];
#pragma unroll
    for (int u = 0; u < FSX_AT_QT; u++)
#pragma unroll
        for (int t = 0; t < FSX_AT_CT; t++) acc[u][t] = (fsx_v4d){0.0, 0.0, 0.0, 0.0};
    const int abeg = ch * FSX_AT_CHUNK + w * (FSX_AT_CHUNK / 4);
    const int aend = min(abeg + FSX_AT_CHUNK / 4, na);
    /* rows past the last q repeat it; nothing reads their sums */
    const double *Jl[FSX_AT_QT];
#pragma unroll
    for (int u = 0; u < FSX_AT_QT; u++)
        Jl[u] = J + ((size_t)l * Q + min((qt0 + u) * 16 + (lane & 15), Q - 1)) * na;
    struct ops {
        double j[FSX_AT_QT], f[FSX_AT_CT], y[FSX_AT_CT];
    } A, B;
    /* unconditional, so that a wait for one step leaves the next one's loads in
     * flight; what is read in place of no atom, tile or column is not used */
    auto load = [&](ops &o, int a0) {
        const int a = min(a0 + (lane >> 4), na - 1);
        const double *Ya = Y + (size_t)a * Kh * 2;
#pragma unroll
        for (int u = 0; u < FSX_AT_QT; u++) o.j[u] = Jl[u][a];
#pragma unroll
        for (int t = 0; t < FSX_AT_CT; t++) {
            o.f[t] = f[(size_t)max(cx[t], 0) * na + a];
            o.y[t] = Ya[coff[t]];
        }
    };
    auto run = [&](const ops &o, int a0) {
        const bool ok = a0 + (lane >> 4) < aend;
        double bv[FSX_AT_CT];
#pragma unroll
        for (int t = 0; t < FSX_AT_CT; t++) bv[t] = ok && cx[t] >= 0 ? o.f[t] * o.y[t] : 0.0;
#pragma unroll
        for (int u = 0; u < FSX_AT_QT; u++)
            if (u < nq) {
                const double av = ok ? o.j[u] : 0.0;
#pragma unroll
                for (int t = 0; t < FSX_AT_CT; t++)
                    if (t < nc) acc[u][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv[t], acc[u][t], 0, 0, 0);
            }
    };
    if (abeg < aend) {
        load(A, abeg);
        for (int a0 = abeg;; a0 += 8) {
            load(B, a0 + 4);
            run(A, a0);
            if (a0 + 4 >= aend) break;
            load(A, a0 + 8);
            run(B, a0 + 4);
            if (a0 + 8 >= aend) break;
        }
    }
    /* wave 0 + wave 1 + wave 2 + wave 3, in that order, per tile */
    double *Pc = P + (size_t)(chunk0 + ch) * 3 * Qp * Kh * 2;
#pragma unroll
    for (int u = 0; u < FSX_AT_QT; u++)
#pragma unroll
        for (int t = 0; t < FSX_AT_CT; t++) {
            if (u >= nq || t >= nc) continue;
            if (w > 0) red[w - 1][lane] = acc[u][t];
            __syncthreads();
            if (w == 0) {
                fsx_v4d v = acc[u][t];
                v += red[0][lane];
                v += red[1][lane];
                v += red[2][lane];
                if (cx[t] >= 0) {
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const int q = (qt0 + u) * 16 + (lane >> 4) + 4 * j;
                        Pc[((size_t)cx[t] * Qp + q) * Kh * 2 + coff[t]] = v[j];
                    }
                }
            }
            __syncthreads();
        }
}

/* ---- the atom expansion in split BF16 on MFMA (the mixed form) ----------
 * The same sums over atoms as k_atom_mfma, each FP64 operand x written as
 * three BF16 parts x = h + m + l + O(2^-24 x) (h = bf16(x), m = bf16(x - h),
 * l = bf16(x - h - m)), and every product as the six part products of at
 * least that order (hh, hm, mh, hl, lh, mm) on v_mfma_f32_16x16x32_bf16 with
 * FP32 accumulation; the chunk partials go to FP64 and k_atom_finish sums
 * them in order.  The parts are formed once per value by k_atom_bes_split
 * (j_l(q r), [part][l][q][atom]) and k_atom_bsplit (f^X conj(Y_lm),
 * [part][column][atom]), atoms innermost so that a lane's 8 atoms of a step
 * are one 16-byte load; atoms are padded to whole chunks with zeros. */
typedef __bf16 fsx_bf16x8 __attribute__((ext_vector_type(8)));
typedef float fsx_v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void split3(double x, __bf16 &h, __bf16 &m, __bf16 &l)
{
    h = (__bf16)(float)x;
    const double r1 = x - (double)(float)h;
    m = (__bf16)(float)r1;
    const double r2 = r1 - (double)(float)m;
    l = (__bf16)(float)r2;
}

/* Js[part][l][q][a] = parts of j_l(q r_a), 0 for q >= Q or a >= na */
__global__ void k_atom_bes_split(__bf16 *Js, const double *r, const double *qvals, int na, int nap,
                                 int Q, int Qp, int K)
{
    /* nap is a multiple of the block size, so a block has one (l, q) */
    __shared__ sbessel_block S;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long tot = (long)K * Qp * nap;
    const int a = (int)(i % nap);
    const long lq = i / nap;
    const int q = (int)(lq % Qp), l = (int)(lq / Qp);
    S.begin(l);
    if (i >= tot) return;
    const double v = q < Q && a < na ? S.value(l, qvals[q] * r[a]) : 0.0;
    __bf16 h, m, lo;
    split3(v, h, m, lo);
    Js[i] = h;
    Js[tot + i] = m;
    Js[2 * tot + i] = lo;
}

/* Bs[part][3 l (l+1) + c][a] = parts of f^X_a conj(Y_lm)(a) for column c =
 * X * 2 (l+1) + 2 m + (0 real, 1 imaginary) of order l */
__global__ void k_atom_bsplit(__bf16 *Bs, const double *f, const double *Y, int na, int nap, int L)
{
    const int K = L + 1, Kh = K * (K + 1) / 2, ncolt = 6 * Kh;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long tot = (long)ncolt * nap;
    if (i >= tot) return;
    const int a = (int)(i % nap), cg = (int)(i / nap);
    int l = 0;
    while (3 * (l + 1) * (l + 2) <= cg) l++;
    const int c = cg - 3 * l * (l + 1);
    const int X = c / (2 * (l + 1)), rem = c - X * 2 * (l + 1);
    const double v = a < na ? f[(size_t)X * na + a] * Y[(size_t)a * Kh * 2 + l * (l + 1) / 2 * 2 + rem]
                            : 0.0;
    __bf16 h, m, lo;
    split3(v, h, m, lo);
    Bs[i] = h;
    Bs[tot + i] = m;
    Bs[2 * tot + i] = lo;
}

/* One block of four waves per (chunk, l, 16-q tile), as k_atom_mfma.  BF16
 * MFMA 16x16x32 operand layout on gfx950: lane i feeds A[i % 16][8 (i / 16)
 * + e] and B[8 (i / 16) + e][i % 16], e = 0..7; result register j of lane i
 * is D[4 (i / 16) + j][i % 16].  Writes the chunk's partial sums
 * P[chunk][X][Qp][Kh][2] in FP64. */
__global__ void __launch_bounds__(256)
k_atom_bf16(const __bf16 *Js, const __bf16 *Bs, double *P, int nap, int Qp, int L, int chunk0)
{
    __shared__ fsx_v4f red[3][64];
    const int K = L + 1, Kh = K * (K + 1) / 2, nqt = Qp / 16;
    int bid = blockIdx.x;
    const int qt = bid % nqt;
    bid /= nqt;
    const int l = bid % K;
    const int ch = bid / K;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int ncol = 3 * 2 * (l + 1), nct = (ncol + 15) / 16;
    const long jtot = (long)K * Qp * nap, btot = (long)6 * Kh * nap;
    fsx_v4f acc[FSX_AT_MAXT];
#pragma unroll
    for (int t = 0; t < FSX_AT_MAXT; t++) acc[t] = (fsx_v4f){0.f, 0.f, 0.f, 0.f};
    const int abeg = ch * FSX_AT_CHUNK + w * (FSX_AT_CHUNK / 4);
    const __bf16 *Ja = Js + ((long)l * Qp + qt * 16 + (lane & 15)) * nap + 8 * (lane >> 4);
    const __bf16 *Bl = Bs + (long)3 * l * (l + 1) * nap + 8 * (lane >> 4);
    for (int a0 = abeg; a0 < abeg + FSX_AT_CHUNK / 4; a0 += 32) {
        const fsx_bf16x8 ah = *reinterpret_cast<const fsx_bf16x8 *>(Ja + a0);
        const fsx_bf16x8 am = *reinterpret_cast<const fsx_bf16x8 *>(Ja + jtot + a0);
        const fsx_bf16x8 al = *reinterpret_cast<const fsx_bf16x8 *>(Ja + 2 * jtot + a0);
#pragma unroll
        for (int t = 0; t < FSX_AT_MAXT; t++) {
            if (t < nct) {
                const int c = t * 16 + (lane & 15);
                fsx_bf16x8 bh = {}, bm = {}, bl = {};
                if (c < ncol) {
                    const __bf16 *Bc = Bl + (long)c * nap + a0;
                    bh = *reinterpret_cast<const fsx_bf16x8 *>(Bc);
                    bm = *reinterpret_cast<const fsx_bf16x8 *>(Bc + btot);
                    bl = *reinterpret_cast<const fsx_bf16x8 *>(Bc + 2 * btot);
                }
                fsx_v4f v = acc[t];
                v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, v, 0, 0, 0);
                v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bm, v, 0, 0, 0);
                v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am, bh, v, 0, 0, 0);
                v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, v, 0, 0, 0);
                v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, v, 0, 0, 0);
                v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am, bm, v, 0, 0, 0);
                acc[t] = v;
            }
        }
    }
    /* wave 0 + wave 1 + wave 2 + wave 3, in that order, per tile */
    const int q0 = qt * 16;
    double *Pc = P + (size_t)(chunk0 + ch) * 3 * Qp * Kh * 2;
#pragma unroll
    for (int t = 0; t < FSX_AT_MAXT; t++) {
        if (t < nct) {
            if (w > 0) red[w - 1][lane] = acc[t];
            __syncthreads();
            if (w == 0) {
                const int c = t * 16 + (lane & 15);
                const int X = c / (2 * (l + 1)), rem = c - X * 2 * (l + 1);
                double v[4];
#pragma unroll
                for (int j = 0; j < 4; j++)
                    v[j] = (double)acc[t][j] + (double)red[0][lane][j] + (double)red[1][lane][j] +
                           (double)red[2][lane][j];
                if (c < ncol) {
                    const int coff = l * (l + 1) / 2 * 2 + rem;
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const int q = q0 + 4 * (lane >> 4) + j;
                        Pc[((size_t)X * Qp + q) * Kh * 2 + coff] = v[j];
                    }
                }
            }
            __syncthreads();
        }
    }
}

/* A^X_lm = 4 pi i^l S_lm and A^X_{l,-m} = (-1)^m 4 pi i^l conj(S_lm), S the
 * sum of the nch chunk partials in chunk order; one thread per (X, q, l, m >= 0) */
__global__ void k_atom_finish(const double *P, int nch, double *re, double *im, int Q, int Qp,
                              int L, double four_pi)
{
#pragma clang fp contract(off)
    const int K = L + 1, Kh = K * (K + 1) / 2, K2 = K * K;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 3L * Q * Kh) return;
    const int e = (int)(i % Kh);
    const int xq = (int)(i / Kh), q = xq % Q, X = xq / Q;
    int l = 0;
    while ((l + 1) * (l + 2) / 2 <= e) l++;
    const int m = e - l * (l + 1) / 2;
    double sr = 0.0, si = 0.0;
    const size_t off = (((size_t)X * Qp + q) * Kh + e) * 2, stride = (size_t)3 * Qp * Kh * 2;
    for (int c = 0; c < nch; c++) {
        sr += P[c * stride + off];
        si += P[c * stride + off + 1];
    }
    const double cr[4] = {four_pi, 0.0, -four_pi, 0.0}, ci[4] = {0.0, four_pi, 0.0, -four_pi};
    const double c_r = cr[l % 4], c_i = ci[l % 4];
    const size_t o = ((size_t)X * Q + q) * K2;
    re[o + l * (l + 1) + m] = c_r * sr - c_i * si;
    im[o + l * (l + 1) + m] = c_r * si + c_i * sr;
    if (m > 0) {
        const double sg = (m & 1) ? -1.0 : 1.0, mr = sg * sr, mi = -sg * si;
        re[o + l * (l + 1) - m] = c_r * mr - c_i * mi;
        im[o + l * (l + 1) - m] = c_r * mi + c_i * mr;
    }
}

/* ---------------------------------------------------------------------- */
/* host side: device buffers, stream, launches */

static pthread_mutex_t g_mtx = PTHREAD_MUTEX_INITIALIZER;
static int g_init = 0;
static hipStream_t g_stream;

/* Working memory of the allocation-free atom expansion
 * (fsx_atoms2spf_noalloc): a fixed device array, one copy per GPU, held until
 * the process ends.  In host code the name scratch is only a host-side
 * stand-in for the symbol: kernels and copies get g_scratch, its device
 * address on the library's device, taken once by hipGetSymbolAddress in
 * init_once. */
#define FSX_NOALLOC_SCRATCH_BYTES ((size_t)64 << 20)
static __device__ __align__(256) unsigned char scratch[FSX_NOALLOC_SCRATCH_BYTES];
static void *g_scratch = NULL;
enum {
    B_BES, B_T, B_RT, B_BT, B_A, B_B, B_DW, B_DS, B_TWA, B_TWG, B_Q, B_Z, B_AM, B_CINT,
    B_POSES, B_KEYS, B_COUNTS, B_OFFS, B_UNITS, B_RECS, B_INFO, B_ACC, B_SCORE, B_C1, B_C2,
    B_CROSSOUT, B_ENT, B_COFF, B_NEXT, B_TALLY, B_SRCT, B_TW2, B_FITCT, B_FITOUT, B_BX, B_BOUT, B_AXYZ,
    B_AFF, B_AWS, B_AQ, B_ARE, B_AIM, B_RTMP, B_FITSC, B_ACCF, B_IN, B_NBUF
};
static void *g_buf[B_NBUF];
static size_t g_cap[B_NBUF];
/* content key of what a buffer holds (fsx_hip_args dw_key / ds_key); 0 =
 * unknown.  Reset whenever the buffer is (re)allocated or released. */
static unsigned long long g_key[B_NBUF];

#define HIPCHK(x)                                                                     \
    do {                                                                              \
        hipError_t e_ = (x);                                                          \
        if (e_ != hipSuccess) {                                                       \
            fprintf(stderr, "[fsx] %s failed: %s (%s:%d)\n", #x, hipGetErrorString(e_), \
                    __FILE__, __LINE__);                                              \
            return FSX_ERR_HIP;                                                       \
        }                                                                             \
    } while (0)

static int ensure(int slot, size_t bytes)
{
    if (bytes == 0) bytes = 256;
    if (g_cap[slot] >= bytes) return FSX_OK;
    if (g_buf[slot]) HIPCHK(hipFree(g_buf[slot]));
    g_buf[slot] = NULL;
    g_cap[slot] = 0;
    g_key[slot] = 0;
    size_t cap = bytes + bytes / 8;
    if (hipMalloc(&g_buf[slot], cap) != hipSuccess) {
        g_buf[slot] = NULL;
        return FSX_ERR_NOMEM;
    }
    g_cap[slot] = cap;
    return FSX_OK;
}

static int g_ncu = 256;
static int g_nxcd = 1;   /* XCDs (accelerator complex dies): workgroups go round-robin */

/* launch-shape knobs: environment override for tuning, defaults otherwise */
static int env_int(const char *name, int dflt, int lo, int hi)
{
    const char *v = getenv(name);
    if (!v || !*v) return dflt;
    int x = atoi(v);
    return x < lo ? lo : (x > hi ? hi : x);
}

static int init_once(void)
{
    if (g_init) return FSX_OK;
    int nd = 0;
    if (hipGetDeviceCount(&nd) != hipSuccess || nd < 1) return FSX_ERR_NODEV;
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    HIPCHK(hipDeviceGetAttribute(&g_ncu, hipDeviceAttributeMultiprocessorCount, dev));
    if (g_ncu < 1) g_ncu = 1;
    if (hipDeviceGetAttribute(&g_nxcd, hipDeviceAttributeNumberOfXccs, dev) != hipSuccess ||
        g_nxcd < 1)
        g_nxcd = 1;
    HIPCHK(hipStreamCreateWithFlags(&g_stream, hipStreamNonBlocking));
    HIPCHK(hipGetSymbolAddress(&g_scratch, HIP_SYMBOL(scratch)));
    g_init = 1;
    return FSX_OK;
}

extern "C" int fsx_hip_device_count(void)
{
    int nd = 0;
    if (hipGetDeviceCount(&nd) != hipSuccess) return 0;
    return nd;
}

static void batch_release(void);
static void stage_release(void);
extern "C" void fsx_hip_release(void)
{
    pthread_mutex_lock(&g_mtx);
    batch_release();
    stage_release();
    for (int i = 0; i < B_NBUF; i++) {
        if (g_buf[i]) (void)hipFree(g_buf[i]);
        g_buf[i] = NULL;
        g_cap[i] = 0;
        g_key[i] = 0;
    }
    pthread_mutex_unlock(&g_mtx);
}

static inline unsigned nblk(long n, int t) { return (unsigned)((n + t - 1) / t); }

#define RC(x)                          \
    do {                               \
        int r_ = (x);                  \
        if (r_ != FSX_OK) return r_;   \
    } while (0)

/* kernel of a cross-term launch with jn slots per lane and pw poses per wavefront */
template <typename E, int PW>
static const void *cross_kernel(int jn, int jobs)
{
    if (jobs)
        return jn <= 1 ? (const void *)k_cross_jobs<1, E, PW> : jn <= 2 ? (const void *)k_cross_jobs<2, E, PW>
             : jn <= 3 ? (const void *)k_cross_jobs<3, E, PW> : (const void *)k_cross_jobs<4, E, PW>;
    return jn <= 1 ? (const void *)k_cross<1, E, PW> : jn <= 2 ? (const void *)k_cross<2, E, PW>
         : jn <= 3 ? (const void *)k_cross<3, E, PW> : (const void *)k_cross<4, E, PW>;
}
static const void *cross_kernel_of(int mixed, int jn, int pw, int jobs)
{
    return pw == 2 ? (mixed ? cross_kernel<cplx32, 2>(jn, jobs) : cross_kernel<cplx, 2>(jn, jobs))
                   : (mixed ? cross_kernel<cplx32, 1>(jn, jobs) : cross_kernel<cplx, 1>(jn, jobs));
}
/* poses per wavefront (FSX_CROSS_PW overrides where two fit, four slots per lane) */
static int cross_pw(int mixed, int ns)
{
    return ns <= 4 * (FSX_WAVE / 2) && env_int("FSX_CROSS_PW", fsx_cross_pw(mixed, ns), 1, 2) == 2 ? 2 : 1;
}
static int cross_jn(int ns, int pw) { return (pw * ns + FSX_WAVE - 1) / FSX_WAVE; }
static size_t cross_lds_of(int mixed, int ns, int urows)
{
    return mixed ? cross_lds<float>(ns, urows) : cross_lds<double>(ns, urows);
}
/* blocks of a cross-term launch: those resident at once, up to most per CU
 * (fsx_cross_blocks; FSX_CROSS_BLOCKS_PER_CU overrides the per-CU count) */
static long cross_grid(const void *kern, size_t lds, int most)
{
    int per = env_int("FSX_CROSS_BLOCKS_PER_CU", 0, 0, 16);
    if (per == 0) {
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kern, FSX_CROSS_BLOCK, lds) != hipSuccess ||
            per < 1)
            per = 1;
        per = per > most ? most : per;
    }
    return (long)g_ncu * per;
}
/* ranges of the (q, unit) order: one per XCD when the grid divides evenly
 * (FSX_CROSS_XCD=0 turns them off) */
static int cross_nx(long grid)
{
    return env_int("FSX_CROSS_XCD", 1, 0, 1) && grid % g_nxcd == 0 ? g_nxcd : 1;
}

/* The persistent form of the cross-term stage (fsx_score_batch): each
 * complex's m-chunks become jobs, grouped into launches of k_cross_jobs by
 * chunk index and kernel shape. */
struct fsx_cross_group {
    int mixed, jn, pw, chunk;   /* the kernel and the m-chunk index */
    size_t lds;                 /* the largest job's LDS */
    int njobs, cap;
    int most;                   /* most blocks per CU any job takes */
    long grid;                  /* blocks of the launch */
    fsx_cross_job *jobs;
};

/* Entry tables of the m-major coefficient order used by the rotated tables
 * and the cross-term kernel: e runs over m = mlo..L, then l = |m|..L (mlo =
 * -L for the full set, 0 for the half set of conjugate-symmetric inputs).
 * The entries are cut into C chunks of whole m values with about ne/C
 * entries each; chunk[m - mlo] is the chunk of m. */
static int entry_chunks(int L, int C, int mlo, int *chunk)
{
    const int K = L + 1, ne = mlo == 0 ? K * (K + 1) / 2 : K * K;
    int e = 0, c = 0, cfirst = 0;
    for (int m = mlo; m <= L; m++) {
        /* close the chunk once it holds its share of the entries */
        if (e > cfirst && c < C - 1 && (long)e * C >= (long)(c + 1) * ne) {
            c++;
            cfirst = e;
        }
        chunk[m - mlo] = c;
        e += K - (m < 0 ? -m : m);
    }
    return ne;
}

/* A^X_{l,-m}(q) = (-1)^(l+m) conj(A^X_{lm}(q)) for m >= 0, to 1e-13 of the
 * largest coefficient of each (X, q): the amplitude of a real density.
 * Then the terms of m and -m of every cross-term sum are complex
 * conjugates of each other, and the sums run over m >= 0 with the m > 0
 * terms counted twice. */
static int spf_conj_symmetric(const double *re, const double *im, int Q, int L)
{
    const int K2 = (L + 1) * (L + 1);
    for (long xq = 0; xq < 3L * Q; xq++) {
        const double *r = re + xq * K2, *i = im + xq * K2;
        double mx = 0.0;
        for (int e = 0; e < K2; e++) {
            const double a = fabs(r[e]), b = fabs(i[e]);
            mx = a > mx ? a : mx;
            mx = b > mx ? b : mx;
        }
        const double tol = 1e-13 * mx;
        /* m = 0: A_l0 = (-1)^l conj(A_l0), i.e. real for even l and imaginary
         * for odd l (the packed m = 0 slots keep only that part of i^l A_l0) */
        for (int l = 0; l <= L; l++) {
            const int e0 = l * l + l;
            if (!(fabs((l & 1) ? r[e0] : i[e0]) <= tol)) return 0;
        }
        for (int l = 1; l <= L; l++)
            for (int m = 1; m <= l; m++) {
                const int ep = l * l + l + m, en = l * l + l - m;
                const double sg = ((l + m) & 1) ? -1.0 : 1.0;
                if (!(fabs(r[en] - sg * r[ep]) <= tol) || !(fabs(i[en] + sg * i[ep]) <= tol)) return 0;
            }
    }
    return 1;
}

/* ---- one complex's pipeline: plan, buffers, uploads, launches ---------------
 * plan_init derives sizes and the host tables of a call; plan_bind gets its
 * device buffers (the process-wide slots for single calls, per-complex sets
 * for batches); plan_upload copies the inputs and tables; plan_enqueue
 * launches every stage on one stream without waiting; plan_finish fills the
 * statistics once the stream has drained. */
enum {
    P_BES, P_T, P_RT, P_BT, P_RTMP, P_A, P_B, P_DW, P_DS, P_TWA, P_TWG, P_Q, P_Z, P_AM, P_CINT,
    P_KEYS, P_INFO, P_COUNTS, P_OFFS, P_UNITS, P_RECS, P_ACC, P_FITSC, P_ENT, P_TW2, P_COFF,
    P_NEXT, P_TALLY, P_SRCT, P_POSES, P_SCORE, P_C1, P_C2, P_CROSSOUT, P_ACCF, P_IN, P_NBUF
};
/* the process-wide slot of each plan buffer (single calls) */
static const int k_plan_slot[P_NBUF] = {
    B_BES, B_T, B_RT, B_BT, B_RTMP, B_A, B_B, B_DW, B_DS, B_TWA, B_TWG, B_Q, B_Z, B_AM, B_CINT,
    B_KEYS, B_INFO, B_COUNTS, B_OFFS, B_UNITS, B_RECS, B_ACC, B_FITSC, B_ENT, B_TW2, B_COFF,
    B_NEXT, B_TALLY, B_SRCT, B_POSES, B_SCORE, B_C1, B_C2, B_CROSSOUT, B_ACCF, B_IN};
/* The inputs and host tables of a call, packed into one device buffer
 * (P_IN, each at a 256-byte aligned offset) and uploaded by one copy from
 * pinned memory: separate copies from pageable memory cost 10 to 40 us of
 * host time each. */
static const int k_packed[] = {P_A, P_B, P_TWA, P_TWG, P_Q, P_Z, P_AM, P_CINT, P_TW2, P_ENT, P_COFF};
static inline bool plan_packed(int i)
{
    for (int k = 0; k < (int)(sizeof(k_packed) / sizeof(k_packed[0])); k++)
        if (k_packed[k] == i) return true;
    return false;
}

typedef void (*fit_kernel_t)(const double *, const int4 *, const int *, int, const double *,
                             const double *, double, double, double, double, double, double *,
                             double *, double *, int *, unsigned long long *, int, int);

struct fsx_plan {
    fsx_hip_args A;
    int L, K, K2, N, Q, n, nb, na, ng, zn, nrows, mixed, half, mlo, npk, C, Tn, ne, dev_out;
    int urows;           /* gamma2 rows per cross-term unit */
    int xblocks;         /* most cross-term blocks per CU */
    int zmajor;          /* more fits than start at once: records sorted by (z, beta2),
                            else by (beta2, z) (k_units) */
    int mirror, nbr;     /* tables of beta <= pi / 2 only (fsx_mirror); their betas */
    long nkeys;
    size_t dsz, spf, es, nent;
    int *ent;     /* host tables (malloc); ent: FSX_E_* parts */
    long *coff;   /* first table value of each chunk: receptor [C], ligand [C] */
    int *pm;      /* first tile, tiles, first entry, entries of each chunk [C][4] */
    double *tw2;
    size_t sz[P_NBUF];   /* bytes of each device buffer (0: not used) */
    size_t inoff[P_NBUF];   /* offset of a packed input within P_IN */
    void *d[P_NBUF];     /* device buffers */
    const long long *dposes;
    double *dscore, *dc1, *dc2, *dcross;
    int aq_lds;
    size_t lds_fit;
    long lanes;
    fit_kernel_t kfit;   /* the compact-form fit (grp = 0) */
    int grp;             /* the lane-group fit k_fitg (mixed form) */
    int fit_wide;        /* lanes with a fit at or below which a fit wavefront
                            evaluates them together (L-BFGS-B fits); lanes per
                            fit (lane groups) */
    int fit_fpw;         /* fits a wavefront starts with (L-BFGS-B fits) */
    long fit_next0;      /* first queue entry not taken at launch */
    int tile_rows;       /* pairs of gamma2 rows per unit (0: as many as fit) */
    int rot_gt;          /* gamma per block of the MFMA rotation (16 or 8), 0: the
                            rotation-then-transpose kernels */
};

/* parts of the entry table (ints), from K2 = (L + 1)^2, K = L + 1, N = 2 L + 1:
 * per entry l, m, chunk, row offset in the receptor table, row offset and
 * padding of its places in the ligand table; first entry of each m; the blocks
 * of the translation table (k_tmat); per chunk the row lengths of the two
 * tables; the translation's tiles */
#define FSX_E_L(p) 0
#define FSX_E_M(p) ((p)->K2)
#define FSX_E_PASS(p) (2 * (p)->K2)
#define FSX_E_OFFR(p) (3 * (p)->K2)
#define FSX_E_OFFB(p) (4 * (p)->K2)
#define FSX_E_PADB(p) (5 * (p)->K2)
#define FSX_E_OFFB2(p) (6 * (p)->K2)
#define FSX_E_PADB2(p) (7 * (p)->K2)
#define FSX_E_MST(p) (8 * (p)->K2)
#define FSX_E_TB(p) (FSX_E_MST(p) + (p)->N)
#define FSX_E_RSR(p) (FSX_E_TB(p) + 4 * (p)->K + 3)
#define FSX_E_RSB(p) (FSX_E_RSR(p) + (p)->N)
#define FSX_E_TILES(p) ((FSX_E_RSB(p) + (p)->N + 7) / 8 * 8)
#define FSX_E_SIZE(p) ((size_t)FSX_E_TILES(p) + 8 * 6 * (size_t)(p)->N)   /* up to 3 tiles in 2 orders per m */

static void plan_free_host(fsx_plan *p)
{
    free(p->ent);
    free(p->coff);
    free(p->pm);
    free(p->tw2);
    p->pm = NULL;
    p->ent = NULL;
    p->coff = NULL;
    p->tw2 = NULL;
}

/* Entry tables, translation tiles and table offsets of the chunks (chunk[m -
 * mlo]) */
static void plan_entries(fsx_plan *p, const int *chunk)
{
    const int L = p->L, K = p->K, TL = FSX_CROSS_TILE;
    int *t = p->ent, *tb = t + FSX_E_TB(p), e = 0, c, nt = 0, tn = 0;
    fsx_tile *tiles = (fsx_tile *)(t + FSX_E_TILES(p));
    for (int m = -L; m <= L; m++) t[FSX_E_MST(p) + m + L] = 0;
    tb[0] = 0;
    /* block of |m| in the given order of l1: its first value in the table */
    auto tblock = [&](int am, int split) {
        for (int k = 0; k < tb[0]; k++)
            if (tb[2 * k + 1] == 2 * am + split) return tb[2 * k + 2];
        const int k = tb[0]++, Km = K - am;
        tb[2 * k + 1] = 2 * am + split;
        tb[2 * k + 2] = tn;
        tn += cross_steps(Km, split) * ((Km + TL - 1) / TL) * cross_tstep(split);
        tb[2 * k + 3] = 0;
        tb[2 * k + 4] = tn;
        return tb[2 * k + 2];
    };
    for (c = 0; c < p->C; c++) {
        const int npk = c == 0 ? p->npk : 0, e0 = e;
        int nc = 0, m0 = L + 1, m1 = -L - 1;
        for (int m = p->mlo; m <= L; m++)
            if (chunk[m - p->mlo] == c) {
                nc += K - (m < 0 ? -m : m);
                m0 = m < m0 ? m : m0;
                m1 = m;
            }
        /* FP64: the entries whose l1 are summed by parity, then added: the
         * first nsplit of the chunk by increasing |m| (as many as made up 256
         * lanes of one entry, or half an entry, each; single terms are not
         * split) */
        int nsplit = 0;
        if (!p->mixed && nc < 256) {
            int one = 0;
            for (int m = m0; m <= m1; m++) one += m == L || m == -L;
            nsplit = 256 - nc < nc - one ? 256 - nc : nc - one;
        }
        p->pm[4 * c] = nt;
        p->pm[4 * c + 2] = e0;
        p->pm[4 * c + 3] = nc;
        int b = 0;
        for (int m = m0; m <= m1; m++) {
            const int am = m < 0 ? -m : m, Km = K - am;
            /* entries before this m by increasing |m| (m = -|m| before |m|) */
            int before = 0;
            for (int k = m0; k <= m1; k++) {
                const int ak = k < 0 ? -k : k;
                if (ak < am || (ak == am && k < m)) before += K - ak;
            }
            int nsp = nsplit - before;
            nsp = nsp < 0 ? 0 : nsp > Km ? Km : nsp;
            t[FSX_E_MST(p) + m + L] = e;
            for (int i = 0; i < Km; i++) {
                const int ec = e + i - e0;
                t[FSX_E_L(p) + e + i] = am + i;
                t[FSX_E_M(p) + e + i] = m;
                t[FSX_E_PASS(p) + e + i] = c;
                t[FSX_E_OFFR(p) + e + i] = ec < 2 * npk ? ec : 2 * (ec - npk);
                t[FSX_E_OFFB2(p) + e + i] = -1;
                t[FSX_E_PADB2(p) + e + i] = 0;
            }
            /* split order (the first nsp l), natural order (the others) */
            for (int split = 1, place = 0; split >= 0; split--) {
                const int lo = split ? 0 : nsp, hi = split ? nsp : Km;
                if (lo >= hi) continue;
                const int nks = cross_steps(Km, split), to = tblock(am, split);
                int *off = t + (place ? FSX_E_OFFB2(p) : FSX_E_OFFB(p)) + e;
                int *pad = t + (place ? FSX_E_PADB2(p) : FSX_E_PADB(p)) + e;
                for (int i = 0; i < Km; i++) {
                    /* split: the even ones' steps, then the odd ones' */
                    const int pos = !split ? i : i % 2 ? 4 * nks + i / 2 : i / 2;
                    const int end = !split || i % 2 == 0 ? 4 * nks : 8 * nks;
                    const int last = split ? i + 2 >= Km : i + 1 == Km;
                    off[i] = b + 6 * pos;
                    pad[i] = last ? end - 1 - pos : 0;
                }
                for (int t0 = 0; t0 < Km; t0 += TL) {
                    const int l = lo > t0 ? lo - t0 : 0, h = hi - t0 < TL ? hi - t0 : TL;
                    if (l >= h) continue;
                    fsx_tile *x = &tiles[nt++];
                    x->bo = b;
                    x->to = to + t0 / TL * nks * cross_tstep(split);
                    x->e = e - e0 + t0;
                    x->nks = nks;
                    x->odd = split ? 24 * nks : 0;
                    x->lo = l;
                    x->hi = h;
                    x->packed = m == 0 && npk > 0;
                }
                b += 24 * nks << split;
                place++;
            }
            e += Km;
        }
        p->pm[4 * c + 1] = nt - p->pm[4 * c];
        t[FSX_E_RSR(p) + c] = 6 * (nc - npk);
        t[FSX_E_RSB(p) + c] = b;
    }
    p->Tn = tn;
    long cr = 0, cb = 0;
    for (c = 0; c < p->C; c++) {
        p->coff[c] = cr;
        p->coff[p->C + c] = cb;
        cr += (long)p->Q * p->nrows * t[FSX_E_RSR(p) + c];
        cb += (long)p->Q * p->nrows * t[FSX_E_RSB(p) + c];
    }
    p->sz[P_RT] = (size_t)cr * (p->es / 2);
    p->sz[P_BT] = (size_t)(cb + FSX_TAB_PAD) * (p->es / 2);
}

/* tile_rows, slot_cap: the cross-term tile shape (pairs of gamma2 rows per unit,
 * pairing slots per m-chunk); 0 takes the defaults (environment knobs, then
 * the form's defaults) */
static int plan_init(fsx_plan *p, const fsx_hip_args *A, int tile_rows, int slot_cap)
{
    memset(p, 0, sizeof(*p));
    p->A = *A;
    p->tile_rows = tile_rows;
    const int L = A->L, K = L + 1, K2 = K * K, N = 2 * L + 1, Q = A->qnum, n = A->n;
    const int nb = A->nbeta, na = A->nalpha, ng = A->ngamma, zn = A->znum;
    p->L = L; p->K = K; p->K2 = K2; p->N = N; p->Q = Q; p->n = n;
    p->nb = nb; p->na = na; p->ng = ng; p->zn = zn;
    p->nrows = nb * ng;
    p->nkeys = (long)zn * nb * ng;
    if (p->nkeys > 0x3fffffffL || (long)p->nrows * Q > 0x7fffffffL) return FSX_ERR_ARG;
    if ((long)L * na >= (1L << 24) || (long)L * ng >= (1L << 24)) return FSX_ERR_ARG;
    p->dsz = 0;
    for (int l = 0; l <= L; l++) p->dsz += dw_size(l);
    p->spf = (size_t)3 * Q * K2;
    p->mixed = (A->flags & FSX_MIXED_FP32) != 0;
    p->dev_out = (A->flags & FSX_DEVICE_OUTPUT) != 0;
    /* half entry set (m >= 0) when both molecules' coefficients are
     * conjugate symmetric; FSX_CROSS_HALF=0 forces the full set */
    p->half = env_int("FSX_CROSS_HALF", 1, 0, 1) && spf_conj_symmetric(A->A_re, A->A_im, Q, L) &&
              spf_conj_symmetric(A->B_re, A->B_im, Q, L);
    p->mlo = p->half ? 0 : -L;
    /* half set: the m = 0 entries of the receptor table and of U share
     * pairing slots two by two (FSX_CROSS_PACK=0 keeps one slot each) */
    p->npk = p->half && env_int("FSX_CROSS_PACK", 1, 0, 1) ? K / 2 : 0;
    p->es = p->mixed ? sizeof(cplx32) : sizeof(cplx);   /* table element size */
    /* half the betas by the mirror image of rows: FP32 tables, whose rounding
     * is far above the 1e-11 by which a truncated pi makes the grid's mirror
     * image miss the grid (the FP64 form keeps every beta) */
    p->mirror = p->mixed && p->half && ng % 2 == 0 && na < (1 << 22) &&
                fabs(A->pi - 3.14159265358979323846) < 1e-10 && env_int("FSX_MIRROR", 1, 0, 1);
    p->nbr = p->mirror ? (nb + 1) / 2 : nb;
    /* m-chunks: one launch per chunk of entries, starting from one chunk
     * (FSX_CROSS_CHUNKS: the smallest count to try); more below while a chunk
     * is too large */
    int C = env_int("FSX_CROSS_CHUNKS", 1, 1, N);
    p->nent = FSX_E_SIZE(p);
    p->ent = (int *)malloc(sizeof(int) * p->nent);
    p->coff = (long *)malloc(sizeof(long) * 2 * (N + 1));
    p->pm = (int *)malloc(sizeof(int) * 4 * (N + 1));
    const int twk = p->mirror ? 2 : 1;   /* x and (l + m) mod 2 of a mirrored form's rows */
    p->tw2 = (double *)calloc(2 * (size_t)na * (N + 1) * twk * twk, sizeof(double));
    int *chunk = (int *)malloc(sizeof(int) * N);
    if (!p->ent || !p->coff || !p->pm || !p->tw2 || !chunk) {
        free(chunk);
        plan_free_host(p);
        return FSX_ERR_NOMEM;
    }
    /* more chunks until the largest fits: at most 256 entries, and for FP32
     * tables at most 128 pairing slots (the order of the FP32 sums across
     * chunks); FSX_CROSS_CHUNK overrides the slot limit */
    const int cmax = slot_cap > 0 ? slot_cap
                                  : env_int("FSX_CROSS_CHUNK", p->mixed ? 2 * FSX_WAVE : 4 * FSX_WAVE,
                                            64, 4 * FSX_WAVE);
    int ncmax, nsmax, ne;
    for (;;) {
        ne = entry_chunks(L, C, p->mlo, chunk);
        ncmax = nsmax = 0;
        for (int c = 0; c < C; c++) {
            int nc = 0;
            for (int m = p->mlo; m <= L; m++)
                if (chunk[m - p->mlo] == c) nc += K - (m < 0 ? -m : m);
            const int ns = nc - (c == 0 ? p->npk : 0);
            if (nc > ncmax) ncmax = nc;
            if (ns > nsmax) nsmax = ns;
        }
        if ((ncmax <= 4 * FSX_WAVE && nsmax <= cmax) || C == N) break;
        C++;
    }
    /* the cross-term kernel addresses a q's receptor rows and a row of the
     * twiddle table by 32-bit byte offsets */
    if (ncmax > 4 * FSX_WAVE || (size_t)p->nrows * 3 * ncmax * p->es >= ((size_t)1 << 32) ||
        p->nrows >= (1 << 24) || na >= (1 << 24) ||
        (size_t)na * (2 * L + 2) * p->es >= ((size_t)1 << 32)) {
        free(chunk);
        plan_free_host(p);
        return FSX_ERR_ARG;
    }
    const long rows_all = p->nrows;
    p->nrows = p->nbr * ng;
    p->C = C;
    p->ne = ne;
    plan_entries(p, chunk);
    free(chunk);
    /* rows per unit: as many as the LDS leaves room for with three blocks to a CU,
     * or two where more are not wanted: a unit's fixed cost is shared by more poses,
     * but a CU needs its blocks to cover the receptor rows' latency */
    auto rows_of = [&](int blocks) {
        int r = FSX_UROWS;
        while (r > 2 && blocks * ((cross_lds_of(p->mixed, nsmax, r) + 2047) / 2048) > 80) r -= 2;
        return r;
    };
    p->xblocks = fsx_cross_blocks(p->mixed, rows_of(3), nsmax, cross_pw(p->mixed, nsmax), rows_all,
                                  (double)n / (double)p->nkeys);
    p->urows = 2 * (tile_rows > 0 ? tile_rows : env_int("FSX_CROSS_ROWS", 0, 0, 4));
    if (p->urows == 0) p->urows = rows_of(p->xblocks < 3 ? p->xblocks : 3);
    /* twiddle e^{-i m a2 2pi/na} per (a2, m): the same table entries the
     * reference's exact transform uses, gathered by (m a2) mod na */
    for (int a2 = 0; a2 < na; a2++)
        for (int m = -L; m <= L; m++) {
            long k = ((long)m * a2) % na;
            if (k < 0) k += na;
            /* half set: the m > 0 terms stand for m and -m (an exact
             * factor 2) */
            const double f = p->half && m > 0 ? 2.0 : 1.0;
            for (int v = 0; v < twk * twk; v++) {
                /* v = 2 x + ((l + m) mod 2), fsx_mirror */
                const double sg = v == 3 ? -f : f;
                double *w = p->tw2 + 2 * (((long)a2 * twk + v / 2) * twk * (N + 1) +
                                          (long)(m + L) * twk + v % 2);
                w[0] = sg * A->tw_a[2 * k];
                w[1] = sg * A->tw_a[2 * k + 1];
            }
        }
    /* the mixed form reads them as FP32 pairs, in place */
    if (p->mixed) {
        float *f32 = (float *)p->tw2;
        for (long i = 0; i < 2L * na * (N + 1) * twk * twk; i++) f32[i] = (float)p->tw2[i];
    }
    /* buffer sizes */
    const size_t es = p->es, spfe = (size_t)3 * Q * ne;   /* rotated-table entries per row */
    size_t *z = p->sz;
    z[P_BES] = sizeof(double) * zn * Q * N;
    z[P_T] = es / 2 * (zn * Q * (size_t)p->Tn + FSX_TAB_PAD);
    z[P_RTMP] = es * (size_t)p->nrows * spfe;
    /* the MFMA rotation, 16 rows of the table to a tile where that takes up to
     * 32 KB of LDS (at 35 and 45 KB, FP64 L = 15 and FP32 L = 25, 0.72 and 6.3 ms
     * against 0.66 and 5.0 with 8 rows and twice the blocks; at 17 KB the same),
     * 8 rows up to 64 KB (FSX_ROT_MFMA=0: the rotation-then-transpose kernels) */
    p->rot_gt = 0;
    if (env_int("FSX_ROT_MFMA", 1, 0, 1)) {
        if ((size_t)16 * ne * es <= 32 * 1024) p->rot_gt = 16;
        else if ((size_t)8 * ne * es <= 64 * 1024) p->rot_gt = 8;
    }
    if (p->rot_gt) z[P_RTMP] = 0;
    z[P_A] = z[P_B] = sizeof(double) * 2 * p->spf;
    z[P_DW] = sizeof(double) * p->dsz * nb;
    z[P_DS] = sizeof(double) * (size_t)K * K2 * N;
    z[P_TWA] = sizeof(double) * 2 * na;
    z[P_TWG] = sizeof(double) * 2 * ng;
    z[P_Q] = sizeof(double) * Q;
    z[P_Z] = sizeof(double) * zn;
    z[P_AM] = z[P_CINT] = sizeof(double) * 6 * Q;
    z[P_KEYS] = sizeof(int) * n;
    z[P_INFO] = sizeof(int2) * n;
    z[P_COUNTS] = sizeof(int) * 2 * p->nkeys;   /* counts, then fills */
    /* then records, buckets, units; then records and units per (z, beta2) group */
    z[P_OFFS] = sizeof(int) * (p->nkeys + 4) + sizeof(int2) * (size_t)nb * zn;
    z[P_UNITS] = sizeof(fsx_unit) * (size_t)n;
    z[P_RECS] = sizeof(int4) * n;
    z[P_ACC] = sizeof(double) * 6 * Q * (size_t)n;
    z[P_FITSC] = sizeof(double) * (size_t)(n > 0 ? n : 1);
    z[P_ENT] = sizeof(int) * p->nent;
    /* rows of 2L + 2 entries (FP32 tables: the packed FP32 values) */
    z[P_TW2] = 2 * (size_t)na * (N + 1) * twk * twk * (p->mixed ? sizeof(float) : sizeof(double));
    z[P_COFF] = sizeof(long) * 2 * p->C;
    z[P_NEXT] = sizeof(int);
    z[P_TALLY] = FSX_TALLY_N * sizeof(unsigned long long);
    z[P_SRCT] = sizeof(cplx) * (size_t)Q * 3 * K2 * ng;
    z[P_POSES] = (A->flags & FSX_DEVICE_POSES) ? 0 : sizeof(long long) * n;
    z[P_SCORE] = z[P_C1] = z[P_C2] = p->dev_out ? 0 : sizeof(double) * n;
    z[P_CROSSOUT] = (!p->dev_out && A->cross) ? sizeof(double) * 6 * Q * (size_t)n : 0;
    size_t inb = 0;
    for (int k = 0; k < (int)(sizeof(k_packed) / sizeof(k_packed[0])); k++) {
        p->inoff[k_packed[k]] = inb;
        inb += (z[k_packed[k]] + 255) & ~(size_t)255;
    }
    z[P_IN] = inb;
    /* the fit launch: as many lanes as are resident at once (the fit
     * state lives in registers, one 256-thread block per CU) */
    p->aq_lds = fit_aq_lds(Q);
    p->lds_fit = fit_lds(Q);
    /* the mixed-precision form's fit: the two-variable L-BFGS-B on lane
     * groups (k_fitg), or with FSX_FIT_COMPACT (or a q grid whose arrays do
     * not fit the block's LDS) the compact-form L-BFGS-B lane per fit, both
     * evaluated in one pass over q; the FP64 form: the reference's
     * L-BFGS-B, lane per fit.  Lanes per fit of the group fit from the number
     * of q alone (fsx_fit_lanes; FSX_FIT_GROUP_LANES overrides), doubled until
     * the block's LDS fits: they set the order of the sums over q, and a pose's
     * result must not depend on the length of its list */
    int fpl = fsx_fit_lanes(Q);
    fpl = env_int("FSX_FIT_GROUP_LANES", fpl, 1, FSX_WAVE);
    while (fpl & (fpl - 1)) fpl &= fpl - 1;   /* a power of two */
    while (fpl < FSX_WAVE && fitg_lds(Q, fpl) > FSX_FIT_LDS) fpl *= 2;
    const int grp = p->mixed && !(A->flags & FSX_FIT_COMPACT) && fitg_lds(Q, fpl) <= FSX_FIT_LDS;
    p->kfit = p->aq_lds ? (p->mixed ? k_fit<1, 1> : k_fit<1, 0>)
                        : (p->mixed ? k_fit<0, 1> : k_fit<0, 0>);
    p->fit_wide = env_int("FSX_FIT_WIDE", 24, 0, 64);
    p->grp = grp;
    if (grp) {
        p->fit_wide = fpl;
        p->lds_fit = fitg_lds(Q, fpl);
        p->sz[P_ACCF] = sizeof(float) * 6 * Q * (size_t)n;
        int bpc = env_int("FSX_FIT_BLOCKS_PER_CU", 0, 0, 16);
        if (bpc == 0 && (hipOccupancyMaxActiveBlocksPerMultiprocessor(&bpc, k_fitg, 256,
                                                                      p->lds_fit) != hipSuccess ||
                         bpc < 1))
            bpc = 1;
        p->lanes = (long)g_ncu * 256 * bpc;
        if (p->lanes > (long)n * fpl) p->lanes = ((long)n * fpl + 255) / 256 * 256;
        p->fit_next0 = p->lanes / fpl;
        p->zmajor = n > p->fit_next0;
        return FSX_OK;
    }
    int fit_bpc = env_int("FSX_FIT_BLOCKS_PER_CU", 0, 0, 16);
    if (fit_bpc == 0 && (hipOccupancyMaxActiveBlocksPerMultiprocessor(&fit_bpc, p->kfit, 256,
                                                                      p->lds_fit) != hipSuccess ||
                         fit_bpc < 1))
        fit_bpc = 1;
    p->lanes = (long)g_ncu * 256 * fit_bpc;
    const int fit_blocks = env_int("FSX_FIT_BLOCKS", 0, 0, 1 << 20);
    if (fit_blocks > 0) p->lanes = 256L * fit_blocks;
    /* fewer fits than lanes are spread evenly over the wavefronts, for the wide
     * evaluation to take them from the start and the steps' divergent code to
     * run for few (52 fits 0.44 to 0.18 ms, 2,000 fits 0.67 to 0.31) */
    const long nw = p->lanes / FSX_WAVE;
    p->fit_fpw = n < p->lanes && p->fit_wide > 0 ? (int)((n + nw - 1) / nw) : FSX_WAVE;
    if (p->fit_fpw < 1) p->fit_fpw = 1;
    if (p->lanes > n) p->lanes = ((long)(n + p->fit_fpw - 1) / p->fit_fpw * FSX_WAVE + 255) / 256 * 256;
    p->fit_next0 = p->lanes / FSX_WAVE * p->fit_fpw;
    p->zmajor = n > p->fit_next0;
    return FSX_OK;
}

/* Device pointers of the plan from get(buffer index, bytes, ctx); the
 * device-resident inputs and outputs of the call are used in place. */
static int plan_bind(fsx_plan *p, int (*get)(int, size_t, void *, void **), void *ctx)
{
    for (int i = 0; i < P_NBUF; i++) {
        p->d[i] = NULL;
        if (p->sz[i] == 0 || plan_packed(i)) continue;
        RC(get(i, p->sz[i], ctx, &p->d[i]));
    }
    for (int i = 0; i < P_NBUF; i++)
        if (plan_packed(i)) p->d[i] = (char *)p->d[P_IN] + p->inoff[i];
    const fsx_hip_args *A = &p->A;
    p->dposes = (A->flags & FSX_DEVICE_POSES) ? (const long long *)A->poses
                                              : (const long long *)p->d[P_POSES];
    if (p->dev_out) {
        p->dscore = A->score; p->dc1 = A->c1; p->dc2 = A->c2; p->dcross = A->cross;
    } else {
        p->dscore = (double *)p->d[P_SCORE];
        p->dc1 = (double *)p->d[P_C1];
        p->dc2 = (double *)p->d[P_C2];
        p->dcross = (double *)p->d[P_CROSSOUT];
    }
    return FSX_OK;
}

#define HIPR(x)                                                                       \
    do {                                                                              \
        hipError_t e_ = (x);                                                          \
        if (e_ != hipSuccess) {                                                       \
            fprintf(stderr, "[fsx] %s failed: %s (%s:%d)\n", #x, hipGetErrorString(e_), \
                    __FILE__, __LINE__);                                              \
            return FSX_ERR_HIP;                                                       \
        }                                                                             \
    } while (0)

/* Pinned staging memory of the packed inputs: stage_begin(bytes) before a
 * call's uploads waits until the previous call's copies out of it are done
 * (an event recorded by stage_end) and grows it to bytes; stage_take hands
 * out 256-byte aligned pieces in order. */
static void *g_stage = NULL;
static size_t g_stage_cap = 0, g_stage_used = 0;
static hipEvent_t g_stage_ev = NULL;
static int g_stage_pending = 0;

static int stage_begin(size_t bytes)
{
    if (g_stage_pending) {
        HIPCHK(hipEventSynchronize(g_stage_ev));
        g_stage_pending = 0;
    }
    if (!g_stage_ev) HIPCHK(hipEventCreateWithFlags(&g_stage_ev, hipEventDisableTiming));
    g_stage_used = 0;
    if (g_stage_cap >= bytes) return FSX_OK;
    if (g_stage) HIPCHK(hipHostFree(g_stage));
    g_stage = NULL;
    g_stage_cap = 0;
    const size_t cap = bytes + bytes / 8 + 256;
    if (hipHostMalloc(&g_stage, cap, hipHostMallocDefault) != hipSuccess) {
        g_stage = NULL;
        return FSX_ERR_NOMEM;
    }
    g_stage_cap = cap;
    return FSX_OK;
}

static char *stage_take(size_t bytes)
{
    bytes = (bytes + 255) & ~(size_t)255;
    if (!g_stage || g_stage_used + bytes > g_stage_cap) return NULL;
    char *h = (char *)g_stage + g_stage_used;
    g_stage_used += bytes;
    return h;
}

static int stage_end(hipStream_t s)
{
    HIPCHK(hipEventRecord(g_stage_ev, s));
    g_stage_pending = 1;
    return FSX_OK;
}

static void stage_release(void)
{
    if (g_stage_pending) (void)hipEventSynchronize(g_stage_ev);
    g_stage_pending = 0;
    if (g_stage) (void)hipHostFree(g_stage);
    g_stage = NULL;
    g_stage_cap = g_stage_used = 0;
}

/* Inputs and tables to the plan's buffers: the packed ones through the
 * pinned staging memory (stage_begin must have made room for sz[P_IN]) in
 * one copy.  up_dw / up_ds: whether the Wigner-d and d-symbol tables must
 * be copied (the buffers may already hold them). */
static int plan_upload(fsx_plan *p, hipStream_t s, int up_dw, int up_ds)
{
    const fsx_hip_args *A = &p->A;
    const size_t spf = p->spf;
    const int Q = p->Q, n = p->n, K = p->K, K2 = p->K2, N = p->N;
    char *h = stage_take(p->sz[P_IN]);
    if (!h) return FSX_ERR_NOMEM;
    auto put = [&](int i, size_t at, const void *src, size_t bytes) {
        memcpy(h + p->inoff[i] + at, src, bytes);
    };
    put(P_A, 0, A->A_re, sizeof(double) * spf);
    put(P_A, sizeof(double) * spf, A->A_im, sizeof(double) * spf);
    put(P_B, 0, A->B_re, sizeof(double) * spf);
    put(P_B, sizeof(double) * spf, A->B_im, sizeof(double) * spf);
    put(P_TWA, 0, A->tw_a, p->sz[P_TWA]);
    put(P_TWG, 0, A->tw_g, p->sz[P_TWG]);
    put(P_Q, 0, A->qvals, sizeof(double) * Q);
    put(P_Z, 0, A->zvals, sizeof(double) * p->zn);
    put(P_AM, 0, A->a, sizeof(double) * 6 * Q);
    put(P_CINT, 0, A->cint, sizeof(double) * 6 * Q);
    put(P_ENT, 0, p->ent, sizeof(int) * p->nent);
    put(P_TW2, 0, p->tw2, p->sz[P_TW2]);
    put(P_COFF, 0, p->coff, p->sz[P_COFF]);
    HIPR(hipMemcpyAsync(p->d[P_IN], h, p->sz[P_IN], hipMemcpyHostToDevice, s));
    if (up_dw) HIPR(hipMemcpyAsync(p->d[P_DW], A->dW, p->sz[P_DW], hipMemcpyHostToDevice, s));
    if (up_ds)
        HIPR(hipMemcpyAsync(p->d[P_DS], A->dsymb, sizeof(double) * K * K2 * N, hipMemcpyHostToDevice, s));
    if (!(A->flags & FSX_DEVICE_POSES))
        HIPR(hipMemcpyAsync(p->d[P_POSES], A->poses, sizeof(long long) * n, hipMemcpyHostToDevice, s));
    if (!p->dev_out) {
        /* device mirrors start from the caller's values so that poses the
         * reference leaves untouched stay untouched */
        HIPR(hipMemcpyAsync(p->dscore, A->score, sizeof(double) * n, hipMemcpyHostToDevice, s));
        HIPR(hipMemcpyAsync(p->dc1, A->c1, sizeof(double) * n, hipMemcpyHostToDevice, s));
        HIPR(hipMemcpyAsync(p->dc2, A->c2, sizeof(double) * n, hipMemcpyHostToDevice, s));
        if (A->cross)
            HIPR(hipMemcpyAsync(p->dcross, A->cross, sizeof(double) * 6 * Q * (size_t)n,
                                hipMemcpyHostToDevice, s));
    }
    return FSX_OK;
}

/* Every stage of the plan on stream s, no waiting; ev (may be NULL): seven
 * events recorded at the stage boundaries (after the tables, rotations,
 * bucketing, cross terms, fit preparation and fit). */
/* stages of plan_enqueue */
#define FSX_ST_PREP 1      /* translation tables, rotated tables, pose buckets */
#define FSX_ST_CROSS 2     /* cross terms */
#define FSX_ST_FITPREP 4   /* fit queue and counters, profile rescale */
#define FSX_ST_FIT 8       /* the fit */
#define FSX_ST_ALL 15

/* chunk c of the plan as a cross-term job of a launch of grid blocks */
static fsx_cross_job cross_job(const fsx_plan *p, int c, long grid)
{
    void *const *g = p->d;
    fsx_cross_job jb;
    memset(&jb, 0, sizeof(jb));
    const size_t fs = p->es / 2;
    jb.acc = (double *)g[P_ACC];
    jb.R = (const char *)g[P_RT] + fs * p->coff[c];
    jb.B = (const char *)g[P_BT] + fs * p->coff[p->C + c];
    jb.T = g[P_T];
    jb.tw2 = g[P_TW2];
    jb.tiles = (const fsx_tile *)((const int *)g[P_ENT] + FSX_E_TILES(p)) + p->pm[4 * c];
    jb.ntiles = p->pm[4 * c + 1];
    jb.el = (const int *)g[P_ENT] + FSX_E_L(p);
    jb.em = (const int *)g[P_ENT] + FSX_E_M(p);
    jb.units = (const fsx_unit *)g[P_UNITS];
    jb.tail = (const int *)g[P_OFFS] + p->nkeys;
    jb.recs = (const int4 *)g[P_RECS];
    jb.Q = p->Q; jb.L = p->L; jb.nrows = p->nrows; jb.ng = p->ng; jb.zn = p->zn; jb.Tn = p->Tn;
    jb.cstart = p->pm[4 * c + 2];
    jb.nc = p->pm[4 * c + 3];
    jb.npk = c == 0 ? p->npk : 0;
    jb.rsB = p->ent[FSX_E_RSB(p) + c];
    jb.first = c == 0;
    jb.nx = cross_nx(grid);
    jb.urows = p->urows;
    jb.mirror = p->mirror;
    jb.nbeta = p->nb;
    return jb;
}

static int plan_enqueue(fsx_plan *p, hipStream_t s, hipEvent_t *ev, int stages = FSX_ST_ALL)
{
    const fsx_hip_args *A = &p->A;
    const int L = p->L, K = p->K, K2 = p->K2, N = p->N, Q = p->Q, n = p->n;
    const int nb = p->nbr, ng = p->ng, zn = p->zn, nrows = p->nrows;
    const long nkeys = p->nkeys;
    void **g = p->d;
    int *counts = (int *)g[P_COUNTS], *offs = (int *)g[P_OFFS], *tail = offs + nkeys;
    const int *ent = (const int *)g[P_ENT];
    if (stages & FSX_ST_PREP) {
    /* translation tables */
    const long nbes = (long)zn * Q * N;
    hipLaunchKernelGGL(k_bessel, dim3(nblk(nbes, 256)), dim3(256), 0, s, (double *)g[P_BES],
                       (const double *)g[P_Z], (const double *)g[P_Q], zn, Q, N);
    const int nzq = zn * Q;
    const dim3 gt(nblk(p->Tn, 256) * nblk(nzq, FSX_TMAT_ZQ));
    if (p->mixed)
        hipLaunchKernelGGL(k_tmat<float>, gt, dim3(256), 0, s, (float *)g[P_T], (const double *)g[P_BES],
                           (const double *)g[P_DS], ent + FSX_E_TB(p), nzq, L, p->Tn);
    else
        hipLaunchKernelGGL(k_tmat<double>, gt, dim3(256), 0, s, (double *)g[P_T], (const double *)g[P_BES],
                           (const double *)g[P_DS], ent + FSX_E_TB(p), nzq, L, p->Tn);
    HIPR(hipGetLastError());
    if (ev) HIPR(hipEventRecord(ev[1], s));
    /* rotated receptor and ligand coefficients, m-chunked */
    {
        const long ntw = (long)Q * 3 * K2 * ng;
        cplx *srct = (cplx *)g[P_SRCT];
        const double *dA = (const double *)g[P_A], *dB = (const double *)g[P_B];
        const size_t spf = p->spf;
        /* gamma chunk: the staged rows (2L+1) x gc complex stay within 48 KB */
        int gc = ng < FSX_WAVE ? ng : FSX_WAVE;
        while (gc > 1 && (size_t)N * gc * sizeof(cplx) > 48 * 1024) gc /= 2;
        const long nrot = (long)Q * 3 * K * ((nb + FSX_ROT_BC - 1) / FSX_ROT_BC) * ((ng + gc - 1) / gc);
        const size_t lds_rot = (size_t)N * gc * sizeof(cplx) + (size_t)FSX_ROT_BC * N * N * sizeof(double);
        for (int side = 0; side < 2; side++) {
            const double *src = side == 0 ? dA : dB;
            void *out = side == 0 ? g[P_RT] : g[P_BT];
            hipLaunchKernelGGL(k_twiddle, dim3(nblk(ntw, 256)), dim3(256), 0, s, srct, src,
                               src + spf, (const double *)g[P_TWG], ng, Q, L, side);
            const int lrot = side == 0 ? 1 : -1;
            fsx_tabmap M;
            M.l = ent + FSX_E_L(p);
            M.pass = ent + FSX_E_PASS(p);
            M.off = ent + (side == 0 ? FSX_E_OFFR(p) : FSX_E_OFFB(p));
            M.pad = ent + FSX_E_PADB(p);
            M.off2 = ent + FSX_E_OFFB2(p);
            M.pad2 = ent + FSX_E_PADB2(p);
            M.rs = ent + (side == 0 ? FSX_E_RSR(p) : FSX_E_RSB(p));
            M.coff = (const long *)g[P_COFF] + (side == 0 ? 0 : p->C);
            M.lig = side;
            M.npk = 2 * p->npk;
            const int *mst = ent + FSX_E_MST(p);
            const double *dw = (const double *)g[P_DW];
            if (p->rot_gt) {
                const int gt = p->rot_gt;
                const dim3 nbr((unsigned)(((long)Q * nb * ((ng + gt - 1) / gt) + 7) / 8 * 24));
                const size_t lds = (size_t)gt * p->ne * p->es;
#define FSX_ROT(E, F, GT)                                                                      \
    hipLaunchKernelGGL((k_rotate_mfma<E, GT>), nbr, dim3(256), lds, s, (F *)out,               \
                       (const cplx *)srct, dw, mst, M, nb, ng, Q, L, p->mlo, p->ne, lrot)
                if (p->mixed && gt == 16) FSX_ROT(cplx32, float, 16);
                else if (p->mixed) FSX_ROT(cplx32, float, 8);
                else if (gt == 16) FSX_ROT(cplx, double, 16);
                else FSX_ROT(cplx, double, 8);
#undef FSX_ROT
                continue;
            }
            /* 64-row tiles of FP32 tables, 32-row tiles of FP64 tables (33 KB of LDS) */
            const int nte = (p->ne + 63) / 64;
            if (p->mixed) {
                hipLaunchKernelGGL(k_rotate<cplx32>, dim3((unsigned)nrot), dim3(256), lds_rot, s,
                                   (cplx32 *)g[P_RTMP], (const cplx *)srct, dw, mst, nb, ng, Q, L, gc,
                                   p->mlo, p->ne);
                const int ntr = (nrows + 63) / 64;
                hipLaunchKernelGGL((k_tab_transpose<cplx32, 64>), dim3((unsigned)((long)Q * 3 * nte * ntr)),
                                   dim3(256), 0, s, (float *)out, (const cplx32 *)g[P_RTMP], p->ne, nrows,
                                   nte, ntr, M, lrot);
            } else {
                hipLaunchKernelGGL(k_rotate<cplx>, dim3((unsigned)nrot), dim3(256), lds_rot, s,
                                   (cplx *)g[P_RTMP], (const cplx *)srct, dw, mst, nb, ng, Q, L, gc,
                                   p->mlo, p->ne);
                const int ntr = (nrows + 31) / 32;
                hipLaunchKernelGGL((k_tab_transpose<cplx, 32>), dim3((unsigned)((long)Q * 3 * nte * ntr)),
                                   dim3(256), 0, s, (double *)out, (const cplx *)g[P_RTMP], p->ne, nrows,
                                   nte, ntr, M, lrot);
            }
        }
    }
    HIPR(hipGetLastError());
    if (ev) HIPR(hipEventRecord(ev[2], s));
    /* poses sorted by z, beta2 and gamma2, and the cross-term units */
    hipLaunchKernelGGL(k_init, dim3(nblk(2 * nkeys, 256)), dim3(256), 0, s, counts, 2 * nkeys, tail,
                       (int *)g[P_NEXT], (int)p->fit_next0, (unsigned long long *)g[P_TALLY]);
    hipLaunchKernelGGL(k_count, dim3(nblk(n, 256)), dim3(256), 0, s, p->dposes, n, zn, p->nb, p->na,
                       ng, p->mirror, p->zmajor, (int *)g[P_KEYS], (int2 *)g[P_INFO], counts);
    int2 *grp = (int2 *)(offs + ((nkeys + 4) & ~1L));
    /* most poses of a unit: where the buckets are crowded, 64 leave most of a unit's
     * rows unused (1,000,000 poses FP64 L = 15: cross terms 34.6 against 30.4 ms); fewer
     * only where the units would not fill the device four times */
    const long items = 4L * 5 * g_ncu;
    const int cap = (int)((long)n * Q / items > FSX_UPOSES ? FSX_UPOSES
                          : (long)n * Q / items < 64 ? 64 : (long)n * Q / items);
    const int nzb = p->nb * zn, scan = fsx_unit_scan(nzb);
    hipLaunchKernelGGL(k_units<0>, dim3(nblk(nzb, 4)), dim3(256), 0, s, (const int *)counts, nzb, p->nb, zn, ng,
                       p->urows, cap, offs, (fsx_unit *)g[P_UNITS], tail, grp, 0, p->zmajor);
    if (scan) hipLaunchKernelGGL(k_unit_scan, dim3(1), dim3(1024), 0, s, grp, nzb);
    hipLaunchKernelGGL(k_units<1>, dim3(nblk(nzb, 4)), dim3(256), 0, s, (const int *)counts, nzb, p->nb, zn, ng,
                       p->urows, cap, offs, (fsx_unit *)g[P_UNITS], tail, grp, scan, p->zmajor);
    hipLaunchKernelGGL(k_scatter, dim3(nblk(n, 256)), dim3(256), 0, s, (const int *)g[P_KEYS],
                       (const int2 *)g[P_INFO], n, ng, (const int *)offs, counts + nkeys,
                       (int4 *)g[P_RECS]);
    HIPR(hipGetLastError());
    if (ev) HIPR(hipEventRecord(ev[3], s));
    }
    /* per-pose cross terms, one launch per m-chunk, accumulated in order */
    if (stages & FSX_ST_CROSS) {
    for (int c = 0; c < p->C; c++) {
        const int ns = p->ent[FSX_E_RSR(p) + c] / 6;
        const int pw = cross_pw(p->mixed, ns);
        const void *kern = cross_kernel_of(p->mixed, cross_jn(ns, pw), pw, 0);
        const size_t lds = cross_lds_of(p->mixed, ns, p->urows);
        /* no more blocks than (q, unit) items can be */
        long grid = cross_grid(kern, lds, p->xblocks);
        if (grid > (long)n * Q) grid = ((long)n * Q + g_nxcd - 1) / g_nxcd * g_nxcd;
        fsx_cross_job jb = cross_job(p, c, grid);
        void *args[1] = {&jb};
        HIPR(hipLaunchKernel(kern, dim3((unsigned)grid), dim3(FSX_CROSS_BLOCK), args, lds, s));
    }
    if (ev) HIPR(hipEventRecord(ev[4], s));
    }
    if (stages & FSX_ST_FITPREP) {
    /* rescaled profiles in place of the pose parts (bounded by n slots;
     * the kernels read the number of valid slots on the device) */
    hipLaunchKernelGGL(k_fit_scale, dim3(nblk(n, 256)), dim3(256), 0, s, (const double *)g[P_ACC],
                       (const double *)g[P_CINT], (const int *)(offs + nkeys), Q, A->peak,
                       (double *)g[P_FITSC]);
    hipLaunchKernelGGL(k_fit_prep, dim3(nblk((long)n * Q, 256)), dim3(256), 0, s,
                       (double *)g[P_ACC], (const double *)g[P_CINT], (const int4 *)g[P_RECS],
                       (const int *)(offs + nkeys), Q, (const double *)g[P_FITSC], p->dcross,
                       p->grp ? (float *)g[P_ACCF] : (float *)NULL);
    HIPR(hipGetLastError());
    if (ev) HIPR(hipEventRecord(ev[5], s));   /* the fit kernel alone from here */
    }
    if (stages & FSX_ST_FIT) {
    if (p->grp)
        hipLaunchKernelGGL(k_fitg, dim3((unsigned)(p->lanes / 256)), dim3(256), p->lds_fit, s,
                           (const float *)g[P_ACCF], (const int4 *)g[P_RECS],
                           (const int *)(offs + nkeys), Q, (const double *)g[P_Q],
                           (const double *)g[P_AM], A->mult, A->c1_lo, A->c1_hi, A->c2_lo,
                           A->c2_hi, p->dscore, p->dc1, p->dc2, (int *)g[P_NEXT],
                           (unsigned long long *)g[P_TALLY], p->fit_wide);
    else
        hipLaunchKernelGGL(p->kfit, dim3((unsigned)(p->lanes / 256)), dim3(256), p->lds_fit, s,
                           (const double *)g[P_ACC], (const int4 *)g[P_RECS],
                           (const int *)(offs + nkeys), Q, (const double *)g[P_Q],
                           (const double *)g[P_AM], A->mult, A->c1_lo, A->c1_hi, A->c2_lo,
                           A->c2_hi, p->dscore, p->dc1, p->dc2, (int *)g[P_NEXT],
                           (unsigned long long *)g[P_TALLY], p->fit_wide, p->fit_fpw);
    HIPR(hipGetLastError());
    if (ev) HIPR(hipEventRecord(ev[6], s));
    }
    return FSX_OK;
}

/* Results to the host (host outputs) and the call's counters to tail /
 * tally, on stream s. */
static int plan_download(fsx_plan *p, hipStream_t s, int *tail, unsigned long long *tally)
{
    const fsx_hip_args *A = &p->A;
    const int n = p->n, Q = p->Q;
    if (!p->dev_out) {
        HIPR(hipMemcpyAsync(A->score, p->dscore, sizeof(double) * n, hipMemcpyDeviceToHost, s));
        HIPR(hipMemcpyAsync(A->c1, p->dc1, sizeof(double) * n, hipMemcpyDeviceToHost, s));
        HIPR(hipMemcpyAsync(A->c2, p->dc2, sizeof(double) * n, hipMemcpyDeviceToHost, s));
        if (A->cross)
            HIPR(hipMemcpyAsync(A->cross, p->dcross, sizeof(double) * 6 * Q * (size_t)n,
                                hipMemcpyDeviceToHost, s));
    }
    HIPR(hipMemcpyAsync(tail, (int *)p->d[P_OFFS] + p->nkeys, sizeof(int) * 2, hipMemcpyDeviceToHost, s));
    HIPR(hipMemcpyAsync(tally, p->d[P_TALLY], FSX_TALLY_N * sizeof(unsigned long long),
                        hipMemcpyDeviceToHost, s));
    return FSX_OK;
}

/* The statistics of a finished plan: counters, algorithmic work and (ms not
 * NULL) the six stage times. */
static void plan_stats(const fsx_plan *p, fsx_stats *st, const float *ms, const int *tail,
                       const unsigned long long *tally)
{
    const int K = p->K, Q = p->Q, ne = p->ne, npk = p->npk, C = p->C;
    const int nvalid = tail[0];
    const long items = (long)Q * tail[1];
    if (ms) {
        st->ms_bessel_t = ms[0];
        st->ms_rotate = ms[1];
        st->ms_group = ms[2];
        st->ms_cross = ms[3];
        st->ms_fit_prep = ms[4];
        st->ms_fit = ms[5];
    }
    st->n_scored = nvalid;
    st->fit_evals = (long)tally[0];
    st->n_capped = (int)tally[1];
    st->fit_steps = (long)tally[2];
    st->fit_wide_steps = (long)tally[3];
    st->fit_max_steps = (long)tally[4];
    st->cross_items = items;
    st->cross_chunks = C;
    /* useful FP64 flops of the cross-term launches: 8 per complex
     * multiply-add of the translated ligand (3 parts, sum_e (L+1-|m_e|)
     * terms per item) and 54 per (pose, q, pairing slot); the npk packed
     * slots carry two m = 0 entries whose other halves are zero */
    double tpair = 0.0;
    for (int m = p->mlo; m <= p->L; m++) {
        const double Km = K - (m < 0 ? -m : m);
        tpair += Km * Km;
    }
    const double nslot = (double)(ne - npk);
    st->cross_flops = (double)items * 3.0 * 8.0 * tpair + (double)nvalid * Q * nslot * 54.0;
    /* algorithmic bytes: per pose and q one receptor row (3 parts, one
     * value per slot) and the six-term accumulator (read and written by
     * every chunk after the first); per item one ligand row */
    st->cross_bytes = (double)nvalid * Q * (3.0 * nslot * (double)p->es + (2.0 * C - 1.0) * 48.0)
                    + (double)items * 3.0 * ne * (double)p->es;
    st->cross_entries = ne;
}

/* single calls: the process-wide buffer slots */
static int get_slot(int i, size_t bytes, void *ctx, void **out)
{
    (void)ctx;
    RC(ensure(k_plan_slot[i], bytes));
    *out = g_buf[k_plan_slot[i]];
    return FSX_OK;
}

static int run_locked(const fsx_hip_args *A, fsx_stats *st)
{
    RC(init_once());
    fsx_plan p;
    RC(plan_init(&p, A, 0, 0));
    hipStream_t s = g_stream;
    hipEvent_t ev[7];
    int nev_made = 0, rc = FSX_OK;
    int tail[2] = {0, 0};
    unsigned long long tally[FSX_TALLY_N] = {0};
    float ms[6];
    rc = plan_bind(&p, get_slot, NULL);
    if (rc == FSX_OK) {
        /* the Wigner-d and d-symbol tables are not copied again when the
         * buffer already holds the same table (content keys) */
        const int up_dw = !(A->dw_key && g_key[B_DW] == A->dw_key);
        const int up_ds = !(A->ds_key && g_key[B_DS] == A->ds_key);
        /* the staging event is recorded whatever the upload returns, so
         * that the next call waits for any copy it did enqueue */
        rc = stage_begin(p.sz[P_IN]);
        if (rc == FSX_OK) {
            rc = plan_upload(&p, s, up_dw, up_ds);
            const int r2 = stage_end(s);
            if (rc == FSX_OK) rc = r2;
        }
        if (rc == FSX_OK) {
            g_key[B_DW] = A->dw_key;
            g_key[B_DS] = A->ds_key;
        }
    }
    for (; rc == FSX_OK && nev_made < 7; nev_made++)
        if (hipEventCreate(&ev[nev_made]) != hipSuccess) rc = FSX_ERR_HIP;
    if (rc == FSX_OK && hipEventRecord(ev[0], s) != hipSuccess) rc = FSX_ERR_HIP;
    if (rc == FSX_OK) rc = plan_enqueue(&p, s, ev);
    if (rc == FSX_OK) rc = plan_download(&p, s, tail, tally);
    if (rc == FSX_OK && hipStreamSynchronize(s) != hipSuccess) rc = FSX_ERR_HIP;
    for (int i = 0; rc == FSX_OK && i < 6; i++)
        if (hipEventElapsedTime(&ms[i], ev[i], ev[i + 1]) != hipSuccess) rc = FSX_ERR_HIP;
    if (rc == FSX_OK) plan_stats(&p, st, ms, tail, tally);
    for (int i = 0; i < nev_made; i++) (void)hipEventDestroy(ev[i]);
    plan_free_host(&p);
    return rc;
}

extern "C" int fsx_hip_run(const fsx_hip_args *A, fsx_stats *st)
{
    pthread_mutex_lock(&g_mtx);
    int rc = run_locked(A, st);
    pthread_mutex_unlock(&g_mtx);
    return rc;
}

/* ---- batches: several complexes in one call --------------------------------
 * Each complex gets its own plan and buffer set.  The inputs are uploaded on
 * the library's stream; then every complex's stages are launched on one of
 * FSX_BSTREAMS streams (complex i on stream i mod FSX_BSTREAMS, forked from
 * and joined back into the library's stream), so that the stages of small
 * complexes run side by side.  That launch sequence is captured once into a
 * HIP graph and replayed by one graph launch on later calls whose launch
 * parameters (sizes, tile shapes, scalars, buffer addresses) are all the same.
 * The cross-term tile shape per expansion-order bucket and form comes from a
 * tuner that times the candidates once on the first complex of the bucket.
 * Two streams: one complex's tables and fits run beside another's cross terms.  With
 * four, several persistent cross-term grids share the CUs and their rows drive each
 * other out of the L2: FP64, 64 complexes of 215,000 poses on average 1,312 ms with
 * four streams, 1,221 with three, 1,188 with two, 1,103 with one; 7 of 14,000 to 71,000
 * 30.8, 30.0, 26.3 and 24.8, 8 of 4,000 to 21,000 14.7, 13.9, 13.7 and 14.1; FP32 508,
 * 498, 496 and 520 for the 64. */
#define FSX_BSTREAMS 2
struct fsx_bset {
    void *d[P_NBUF];
    size_t cap[P_NBUF];
    unsigned long long dw_key, ds_key;   /* tables held by d[P_DW], d[P_DS] */
};
static fsx_bset *g_bat = NULL;
static int g_nbat = 0;
/* intermediates (written and read by the stages of one complex only) are
 * shared by the complexes of one stream, which run one after another;
 * inputs uploaded before the stages run, outputs and the counters read
 * back afterwards are per complex */
static fsx_bset g_bstr[FSX_BSTREAMS];
/* persist: the persistent launches read the translation and rotated tables,
 * the buckets, the accumulators and the fit queue of every complex after all
 * complexes' table stages, so those are per complex */
static inline int per_stream_buffer(int i, int persist)
{
    switch (i) {
    case P_T: case P_RT: case P_BT: case P_UNITS: case P_RECS: case P_ACC: case P_NEXT:
    case P_ACCF:
        return !persist;
    case P_BES: case P_RTMP: case P_KEYS: case P_INFO: case P_COUNTS: case P_FITSC: case P_SRCT:
        return 1;
    default:
        return 0;
    }
}
struct fsx_bctx {
    fsx_bset *cplx, *strm;
    int persist;
};
static hipStream_t g_bs[FSX_BSTREAMS];
static hipEvent_t g_bfork, g_bjoin[FSX_BSTREAMS];
static int g_binit = 0;
static hipGraph_t g_graph = NULL;
static hipGraphExec_t g_gexec = NULL;
static void *g_gkey = NULL;
static size_t g_gkey_len = 0;

/* the launch parameters a captured graph depends on, per complex */
struct fsx_gkey {
    int L, nb, na, ng, Q, zn, n, flags, half, npk, C, urows, mirror, tile_rows, aq_lds,
        fit_wide, fit_fpw;
    long lanes;
    double mult, peak, c1_lo, c1_hi, c2_lo, c2_hi;
    void *d[P_NBUF];
    const void *dposes;
    void *dscore, *dc1, *dc2, *dcross;
};

static int batch_init(void)
{
    if (g_binit) return FSX_OK;
    for (int i = 0; i < FSX_BSTREAMS; i++) {
        HIPCHK(hipStreamCreateWithFlags(&g_bs[i], hipStreamNonBlocking));
        HIPCHK(hipEventCreateWithFlags(&g_bjoin[i], hipEventDisableTiming));
    }
    HIPCHK(hipEventCreateWithFlags(&g_bfork, hipEventDisableTiming));
    g_binit = 1;
    return FSX_OK;
}

static void graph_drop(void)
{
    if (g_gexec) (void)hipGraphExecDestroy(g_gexec);
    if (g_graph) (void)hipGraphDestroy(g_graph);
    g_gexec = NULL;
    g_graph = NULL;
    free(g_gkey);
    g_gkey = NULL;
    g_gkey_len = 0;
}

static int get_bat(int i, size_t bytes, void *ctx, void **out)
{
    const fsx_bctx *c = (const fsx_bctx *)ctx;
    fsx_bset *b = per_stream_buffer(i, c->persist) ? c->strm : c->cplx;
    if (b->cap[i] < bytes) {
        if (b->d[i]) HIPCHK(hipFree(b->d[i]));
        b->d[i] = NULL;
        b->cap[i] = 0;
        if (i == P_DW) b->dw_key = 0;
        if (i == P_DS) b->ds_key = 0;
        const size_t cap = bytes + bytes / 8;
        if (hipMalloc(&b->d[i], cap) != hipSuccess) {
            b->d[i] = NULL;
            return FSX_ERR_NOMEM;
        }
        b->cap[i] = cap;
    }
    *out = b->d[i];
    return FSX_OK;
}


/* ---- tile-shape tuner ----
 * Per expansion-order bucket (L <= 10, 15, 20, 25, 30, 40) and form, the
 * pairs of gamma2 rows per unit with the shortest cross-term stage on the first
 * complex of that bucket; FSX_TUNE_FILE names a text file the table is
 * read from and appended to ("bucket mixed rows slots ms pairs" lines, slots 0:
 * the form's default pairing-slot cap).  Lines without the last word are of
 * versions whose rows meant single rows of another kernel: they are passed over,
 * and their buckets tuned again. */
#define FSX_TUNE_BUCKETS 6
static int g_tune[FSX_TUNE_BUCKETS][2][2];   /* rows, slots; 0: not tuned */
static int g_tune_loaded = 0;
static fsx_cross_job *g_cjob_dev;
static size_t g_cjob_cap;
static fsx_fit_job *g_fjob_dev;
static size_t g_fjob_cap;
static void batch_release(void)
{
    graph_drop();
    if (g_cjob_dev) (void)hipFree(g_cjob_dev);
    if (g_fjob_dev) (void)hipFree(g_fjob_dev);
    g_cjob_dev = NULL;
    g_fjob_dev = NULL;
    g_cjob_cap = g_fjob_cap = 0;
    memset(g_tune, 0, sizeof(g_tune));
    g_tune_loaded = 0;
    for (int k = 0; k < g_nbat; k++)
        for (int i = 0; i < P_NBUF; i++)
            if (g_bat[k].d[i]) (void)hipFree(g_bat[k].d[i]);
    for (int k = 0; k < FSX_BSTREAMS; k++)
        for (int i = 0; i < P_NBUF; i++)
            if (g_bstr[k].d[i]) (void)hipFree(g_bstr[k].d[i]);
    memset(g_bstr, 0, sizeof(g_bstr));
    free(g_bat);
    g_bat = NULL;
    g_nbat = 0;
}

static inline int tune_bucket(int L)
{
    return L <= 10 ? 0 : L <= 15 ? 1 : L <= 20 ? 2 : L <= 25 ? 3 : L <= 30 ? 4 : 5;
}

static void tune_load(void)
{
    if (g_tune_loaded) return;
    g_tune_loaded = 1;
    const char *path = getenv("FSX_TUNE_FILE");
    if (!path || !*path) return;
    FILE *f = fopen(path, "r");
    if (!f) return;
    int b, m, r, c;
    double ms;
    char line[128], tag[8];
    while (fgets(line, sizeof(line), f))
        if (sscanf(line, "%d %d %d %d %lf %7s", &b, &m, &r, &c, &ms, tag) == 6 &&
            strcmp(tag, "pairs") == 0 && b >= 0 && b < FSX_TUNE_BUCKETS && m >= 0 && m <= 1 && r >= 1 && r <= 4 &&
            (c == 0 || (c >= 64 && c <= 4 * FSX_WAVE))) {
            g_tune[b][m][0] = r;
            g_tune[b][m][1] = c;
        }
    fclose(f);
}

static void tune_save(int b, int m, int r, int c, double ms)
{
    const char *path = getenv("FSX_TUNE_FILE");
    if (!path || !*path) return;
    FILE *f = fopen(path, "a");
    if (!f) return;
    fprintf(f, "%d %d %d %d %.4f pairs\n", b, m, r, c, ms);
    fclose(f);
}

/* Time the cross-term stage of complex A for each candidate shape in the
 * process-wide buffers and record the fastest for its bucket. */
static int tune_one(const fsx_hip_args *A)
{
    const int mixed = (A->flags & FSX_MIXED_FP32) != 0, b = tune_bucket(A->L);
    /* pairs of gamma2 rows per unit; the pairing-slot cap stays the form's default,
     * since it sets the m-chunks and with them the order of the FP32 sums
     * (rows change no arithmetic: a tuned batch scores every pose exactly as
     * a single call does) */
    static const int cand32[][2] = {{4, 0}, {2, 0}, {1, 0}};
    static const int cand64[][2] = {{2, 0}, {1, 0}, {4, 0}};
    const int nc = 3;
    hipEvent_t ev[7];
    int nev = 0, rc = FSX_OK, best = -1;
    float best_ms = 0.f;
    for (; nev < 7; nev++)
        if (hipEventCreate(&ev[nev]) != hipSuccess) {
            rc = FSX_ERR_HIP;
            break;
        }
    for (int k = 0; rc == FSX_OK && k < nc; k++) {
        const int rows = mixed ? cand32[k][0] : cand64[k][0];
        const int slots = mixed ? cand32[k][1] : cand64[k][1];
        fsx_plan p;
        rc = plan_init(&p, A, rows, slots);
        if (rc != FSX_OK) break;
        rc = plan_bind(&p, get_slot, NULL);
        if (rc == FSX_OK) {
            rc = stage_begin(p.sz[P_IN]);
            if (rc == FSX_OK) {
                rc = plan_upload(&p, g_stream, 1, 1);
                const int r2 = stage_end(g_stream);
                if (rc == FSX_OK) rc = r2;
            }
        }
        if (rc == FSX_OK) {
            g_key[B_DW] = 0;   /* the buffers now hold this complex's tables */
            g_key[B_DS] = 0;
        }
        /* twice: the first run warms the caches and code */
        float ms = 0.f;
        for (int rep = 0; rc == FSX_OK && rep < 2; rep++) {
            if (hipEventRecord(ev[0], g_stream) != hipSuccess) rc = FSX_ERR_HIP;
            if (rc == FSX_OK) rc = plan_enqueue(&p, g_stream, ev, FSX_ST_PREP | FSX_ST_CROSS);
            if (rc == FSX_OK && hipStreamSynchronize(g_stream) != hipSuccess) rc = FSX_ERR_HIP;
            if (rc == FSX_OK && hipEventElapsedTime(&ms, ev[3], ev[4]) != hipSuccess) rc = FSX_ERR_HIP;
        }
        plan_free_host(&p);
        if (rc == FSX_OK && (best < 0 || ms < best_ms)) {
            best = k;
            best_ms = ms;
        }
    }
    for (int i = 0; i < nev; i++) (void)hipEventDestroy(ev[i]);
    if (rc == FSX_OK && best >= 0) {
        g_tune[b][mixed][0] = mixed ? cand32[best][0] : cand64[best][0];
        g_tune[b][mixed][1] = mixed ? cand32[best][1] : cand64[best][1];
        tune_save(b, mixed, g_tune[b][mixed][0], g_tune[b][mixed][1], best_ms);
    }
    return rc;
}


/* the cross-term chunks of plan p appended to the groups (grown as needed);
 * nx is set at launch */
static int plan_cross_collect(const fsx_plan *p, fsx_cross_group **gr, int *ngr)
{
    for (int c = 0; c < p->C; c++) {
        const int ns = p->ent[FSX_E_RSR(p) + c] / 6;
        const size_t lds = cross_lds_of(p->mixed, ns, p->urows);
        const int pw = cross_pw(p->mixed, ns), jn = cross_jn(ns, pw);
        fsx_cross_group *t = NULL;
        for (int i = 0; i < *ngr; i++) {
            fsx_cross_group *u = &(*gr)[i];
            if (u->mixed == p->mixed && u->jn == jn && u->pw == pw && u->chunk == c) t = u;
        }
        if (!t) {
            fsx_cross_group *ng2 = (fsx_cross_group *)realloc(*gr, sizeof(fsx_cross_group) * (*ngr + 1));
            if (!ng2) return FSX_ERR_NOMEM;
            *gr = ng2;
            t = &(*gr)[(*ngr)++];
            memset(t, 0, sizeof(*t));
            t->mixed = p->mixed; t->jn = jn; t->pw = pw; t->chunk = c;
        }
        if (t->njobs == t->cap) {
            const int cap = t->cap ? 2 * t->cap : 8;
            fsx_cross_job *nj = (fsx_cross_job *)realloc(t->jobs, sizeof(fsx_cross_job) * cap);
            if (!nj) return FSX_ERR_NOMEM;
            t->jobs = nj;
            t->cap = cap;
        }
        if (lds > t->lds) t->lds = lds;
        if (p->xblocks > t->most) t->most = p->xblocks;
        t->jobs[t->njobs++] = cross_job(p, c, 1);
    }
    return FSX_OK;
}

static int grow_dev(void **buf, size_t *cap, size_t bytes)
{
    if (*cap >= bytes) return FSX_OK;
    if (*buf) HIPCHK(hipFree(*buf));
    *buf = NULL;
    *cap = 0;
    if (hipMalloc(buf, bytes) != hipSuccess) {
        *buf = NULL;
        return FSX_ERR_NOMEM;
    }
    *cap = bytes;
    return FSX_OK;
}

static int run_batch_locked(int nprob, const fsx_hip_args *args, fsx_stats *st)
{
    RC(init_once());
    RC(batch_init());
    tune_load();
    const int use_graph = env_int("FSX_BATCH_GRAPH", 1, 0, 1);
    const int tune = env_int("FSX_TUNE", 1, 0, 1);
    /* FSX_BATCH_PERSIST=1: the persistent form, one cross-term launch per
     * (m-chunk index, kernel shape) and one fit launch over all complexes,
     * after every complex's table stages.  Default: each complex's whole
     * pipeline on one of two streams, which on the 64-complex bench batch
     * is faster (496 against 706 ms per mixed step, 1,200 against 1,325 in
     * FP64): the streams overlap one complex's tables and fits with
     * another's cross terms, where the persistent form runs those stages one
     * after another, the fits with a block-level tail per complex */
    const int persist = env_int("FSX_BATCH_PERSIST", 0, 0, 1);
    /* the tuner first (it runs in the process-wide buffers) */
    for (int i = 0; tune && i < nprob; i++) {
        const int m = (args[i].flags & FSX_MIXED_FP32) != 0, b = tune_bucket(args[i].L);
        if (!g_tune[b][m][0] && args[i].n > 0) RC(tune_one(&args[i]));
    }
    if (g_nbat < nprob) {
        fsx_bset *nb = (fsx_bset *)realloc(g_bat, sizeof(fsx_bset) * nprob);
        if (!nb) return FSX_ERR_NOMEM;
        memset(nb + g_nbat, 0, sizeof(fsx_bset) * (nprob - g_nbat));
        g_bat = nb;
        g_nbat = nprob;
    }
    fsx_plan *pl = (fsx_plan *)calloc(nprob, sizeof(fsx_plan));
    int *tail = (int *)calloc(2 * (size_t)nprob, sizeof(int));
    unsigned long long *tally =
        (unsigned long long *)calloc(FSX_TALLY_N * (size_t)nprob, sizeof(unsigned long long));
    /* one key per complex and one for the batch's own launches */
    fsx_gkey *key = (fsx_gkey *)calloc((size_t)nprob + 1, sizeof(fsx_gkey));
    fsx_cross_group *cg = NULL;
    int ncg = 0, nfj = 0;
    fsx_fit_job *fj = NULL;
    size_t fj_lds = 0;
    long fj_lanes = 0;
    int rc = (pl && tail && tally && key) ? FSX_OK : FSX_ERR_NOMEM;
    int ninit = 0;
    for (; rc == FSX_OK && ninit < nprob; ninit++) {
        const fsx_hip_args *A = &args[ninit];
        const int m = (A->flags & FSX_MIXED_FP32) != 0, b = tune_bucket(A->L);
        rc = plan_init(&pl[ninit], A, g_tune[b][m][0], g_tune[b][m][1]);
        if (rc != FSX_OK) break;
    }
    /* the shared buffers of each stream at the size its largest complex
     * needs, before any plan takes their addresses */
    for (int j = 0; rc == FSX_OK && j < FSX_BSTREAMS; j++)
        for (int i = 0; rc == FSX_OK && i < P_NBUF; i++) {
            if (!per_stream_buffer(i, persist)) continue;
            size_t need = 0;
            for (int k = j; k < ninit; k += FSX_BSTREAMS)
                if (pl[k].sz[i] > need) need = pl[k].sz[i];
            if (need == 0) continue;
            fsx_bctx bc = {NULL, &g_bstr[j], persist};
            void *dummy;
            rc = get_bat(i, need, &bc, &dummy);
        }
    size_t stage_bytes = 0;
    for (int k = 0; k < ninit; k++) stage_bytes += (pl[k].sz[P_IN] + 255) & ~(size_t)255;
    const int staged = rc == FSX_OK;
    if (rc == FSX_OK) rc = stage_begin(stage_bytes);
    for (int k = 0; rc == FSX_OK && k < ninit; k++) {
        const fsx_hip_args *A = &args[k];
        fsx_bctx bc = {&g_bat[k], &g_bstr[k % FSX_BSTREAMS], persist};
        rc = plan_bind(&pl[k], get_bat, &bc);
        if (rc != FSX_OK) break;
        fsx_bset *bs = &g_bat[k];
        const int up_dw = !(A->dw_key && bs->dw_key == A->dw_key);
        const int up_ds = !(A->ds_key && bs->ds_key == A->ds_key);
        rc = plan_upload(&pl[k], g_stream, up_dw, up_ds);
        if (rc == FSX_OK) {
            bs->dw_key = A->dw_key;
            bs->ds_key = A->ds_key;
        }
    }
    if (staged && g_stage_ev) {
        const int r2 = stage_end(g_stream);
        if (rc == FSX_OK) rc = r2;
    }
    /* the persistent launches' jobs */
    int fitjobs = 0;
    if (rc == FSX_OK && persist && nprob > 0) {
        for (int k = 0; rc == FSX_OK && k < ninit; k++)
            if (pl[k].n > 0) rc = plan_cross_collect(&pl[k], &cg, &ncg);
        /* launches in m-chunk order, so that each complex's chunks add up in
         * order (one chunk of a complex per launch) */
        for (int i = 1; i < ncg; i++)
            for (int j = i; j > 0 && cg[j].chunk < cg[j - 1].chunk; j--) {
                const fsx_cross_group t = cg[j];
                cg[j] = cg[j - 1];
                cg[j - 1] = t;
            }
        size_t ntot = 0;
        for (int i = 0; i < ncg; i++) ntot += cg[i].njobs;
        for (int i = 0; rc == FSX_OK && i < ncg; i++) {
            cg[i].grid = cross_grid(cross_kernel_of(cg[i].mixed, cg[i].jn, cg[i].pw, 1), cg[i].lds, cg[i].most);
            for (int j = 0; j < cg[i].njobs; j++) cg[i].jobs[j].nx = cross_nx(cg[i].grid);
        }
        if (rc == FSX_OK) rc = grow_dev((void **)&g_cjob_dev, &g_cjob_cap,
                                        sizeof(fsx_cross_job) * (ntot > 0 ? ntot : 1));
        for (int i = 0, o = 0; rc == FSX_OK && i < ncg; o += cg[i].njobs, i++)
            if (hipMemcpy(g_cjob_dev + o, cg[i].jobs, sizeof(fsx_cross_job) * cg[i].njobs,
                          hipMemcpyHostToDevice) != hipSuccess)
                rc = FSX_ERR_HIP;
        /* one fit launch when every complex with poses takes the lane-group
         * fit */
        fitjobs = 1;
        for (int k = 0; k < ninit; k++)
            if (pl[k].n > 0 && !pl[k].grp) fitjobs = 0;
        if (fitjobs && rc == FSX_OK) {
            fj = (fsx_fit_job *)calloc((size_t)ninit, sizeof(fsx_fit_job));
            if (!fj) rc = FSX_ERR_NOMEM;
            for (int k = 0; rc == FSX_OK && k < ninit; k++) {
                if (pl[k].n == 0) continue;
                if (pl[k].lds_fit > fj_lds) fj_lds = pl[k].lds_fit;
            }
            int bpc = env_int("FSX_FIT_BLOCKS_PER_CU", 0, 0, 16);
            if (rc == FSX_OK && bpc == 0 &&
                (hipOccupancyMaxActiveBlocksPerMultiprocessor(&bpc, k_fitg_jobs, 256, fj_lds) !=
                     hipSuccess ||
                 bpc < 1))
                bpc = 1;
            fj_lanes = (long)g_ncu * 256 * bpc;
            for (int k = 0; rc == FSX_OK && k < ninit; k++) {
                fsx_plan *p = &pl[k];
                if (p->n == 0) continue;
                const fsx_hip_args *A = &p->A;
                void **g = p->d;
                fsx_fit_job *f = &fj[nfj++];
                f->acc = (const float *)g[P_ACCF];
                f->qvals = (const double *)g[P_Q];
                f->a = (const double *)g[P_AM];
                f->recs = (const int4 *)g[P_RECS];
                f->nvalid_p = (const int *)g[P_OFFS] + p->nkeys;
                f->mult = A->mult;
                f->c1_lo = A->c1_lo; f->c1_hi = A->c1_hi; f->c2_lo = A->c2_lo; f->c2_hi = A->c2_hi;
                f->score = p->dscore; f->c1o = p->dc1; f->c2o = p->dc2;
                f->next = (int *)g[P_NEXT];
                f->tally = (unsigned long long *)g[P_TALLY];
                f->Q = p->Q;
                f->fpl = p->fit_wide;
                /* each job's queue starts past the groups the launch holds */
                p->fit_next0 = fj_lanes / p->fit_wide;
            }
            if (rc == FSX_OK) rc = grow_dev((void **)&g_fjob_dev, &g_fjob_cap,
                                            sizeof(fsx_fit_job) * (nfj > 0 ? nfj : 1));
            if (rc == FSX_OK && nfj > 0 &&
                hipMemcpy(g_fjob_dev, fj, sizeof(fsx_fit_job) * nfj, hipMemcpyHostToDevice) !=
                    hipSuccess)
                rc = FSX_ERR_HIP;
        }
    }
    for (int k = 0; rc == FSX_OK && k < ninit; k++) {
        const fsx_hip_args *A = &args[k];
        fsx_gkey *ky = &key[k];
        const fsx_plan *p = &pl[k];
        ky->L = p->L; ky->nb = p->nb; ky->na = p->na; ky->ng = p->ng; ky->Q = p->Q; ky->zn = p->zn;
        ky->n = p->n; ky->flags = (int)A->flags; ky->half = p->half; ky->npk = p->npk; ky->C = p->C;
        ky->urows = p->urows; ky->mirror = p->mirror;
        ky->tile_rows = p->tile_rows; ky->aq_lds = p->aq_lds; ky->lanes = p->lanes;
        ky->fit_wide = p->fit_wide; ky->fit_fpw = p->fit_fpw;
        ky->mult = A->mult; ky->peak = A->peak; ky->c1_lo = A->c1_lo; ky->c1_hi = A->c1_hi;
        ky->c2_lo = A->c2_lo; ky->c2_hi = A->c2_hi;
        memcpy(ky->d, p->d, sizeof(ky->d));
        ky->dposes = p->dposes; ky->dscore = p->dscore; ky->dc1 = p->dc1; ky->dc2 = p->dc2;
        ky->dcross = p->dcross;
    }
    if (rc == FSX_OK) {
        /* the batch's own launches: the form, the job tables and their grids */
        fsx_gkey *ky = &key[nprob];
        ky->n = persist;
        ky->flags = fitjobs;
        ky->lanes = fj_lanes;
        ky->d[0] = g_cjob_dev;
        ky->d[1] = g_fjob_dev;
        ky->C = ncg;
        ky->Q = nfj;
    }
    /* the stages of every complex: one graph launch, or the launches */
    if (rc == FSX_OK && nprob > 0) {
        const size_t klen = sizeof(fsx_gkey) * ((size_t)nprob + 1);
        const int replay = use_graph && g_gexec && g_gkey_len == klen && memcmp(g_gkey, key, klen) == 0;
        if (!replay) {
            graph_drop();
            hipError_t e = use_graph ? hipStreamBeginCapture(g_stream, hipStreamCaptureModeRelaxed)
                                     : hipSuccess;
            /* fork to the streams, stages, join back on g_stream */
            auto fork = [&]() {
                hipError_t r = hipEventRecord(g_bfork, g_stream);
                for (int j = 0; r == hipSuccess && j < FSX_BSTREAMS; j++)
                    r = hipStreamWaitEvent(g_bs[j], g_bfork, 0);
                return r;
            };
            auto join = [&]() {
                hipError_t r = hipSuccess;
                for (int j = 0; r == hipSuccess && j < FSX_BSTREAMS; j++) {
                    r = hipEventRecord(g_bjoin[j], g_bs[j]);
                    if (r == hipSuccess) r = hipStreamWaitEvent(g_stream, g_bjoin[j], 0);
                }
                return r;
            };
            if (e == hipSuccess) e = fork();
            if (e != hipSuccess) rc = FSX_ERR_HIP;
            for (int i = 0; rc == FSX_OK && i < nprob; i++)
                rc = plan_enqueue(&pl[i], g_bs[i % FSX_BSTREAMS], NULL,
                                  persist ? FSX_ST_PREP : FSX_ST_ALL);
            if (rc == FSX_OK && join() != hipSuccess) rc = FSX_ERR_HIP;
            if (persist) {
                for (int i = 0, o = 0; rc == FSX_OK && i < ncg; o += cg[i].njobs, i++) {
                    const fsx_cross_job *jobs = g_cjob_dev + o;
                    int nj = cg[i].njobs;
                    void *kargs[2] = {(void *)&jobs, (void *)&nj};
                    if (hipLaunchKernel(cross_kernel_of(cg[i].mixed, cg[i].jn, cg[i].pw, 1),
                                        dim3((unsigned)cg[i].grid), dim3(FSX_CROSS_BLOCK), kargs,
                                        cg[i].lds, g_stream) !=
                        hipSuccess)
                        rc = FSX_ERR_HIP;
                }
                if (rc == FSX_OK && fork() != hipSuccess) rc = FSX_ERR_HIP;
                for (int i = 0; rc == FSX_OK && i < nprob; i++)
                    rc = plan_enqueue(&pl[i], g_bs[i % FSX_BSTREAMS], NULL,
                                      FSX_ST_FITPREP | (fitjobs ? 0 : FSX_ST_FIT));
                if (rc == FSX_OK && join() != hipSuccess) rc = FSX_ERR_HIP;
                if (rc == FSX_OK && fitjobs && nfj > 0) {
                    hipLaunchKernelGGL(k_fitg_jobs, dim3((unsigned)(fj_lanes / 256)), dim3(256),
                                       fj_lds, g_stream, (const fsx_fit_job *)g_fjob_dev, nfj);
                    if (hipGetLastError() != hipSuccess) rc = FSX_ERR_HIP;
                }
            }
            if (use_graph) {
                hipGraph_t gr = NULL;
                const hipError_t ee = hipStreamEndCapture(g_stream, &gr);
                if (rc == FSX_OK && ee != hipSuccess) rc = FSX_ERR_HIP;
                if (rc == FSX_OK && hipGraphInstantiate(&g_gexec, gr, NULL, NULL, 0) != hipSuccess) {
                    g_gexec = NULL;
                    rc = FSX_ERR_HIP;
                }
                if (rc == FSX_OK) {
                    g_graph = gr;
                    g_gkey = malloc(klen);
                    if (g_gkey) {
                        memcpy(g_gkey, key, klen);
                        g_gkey_len = klen;
                    }
                } else if (gr) {
                    (void)hipGraphDestroy(gr);
                }
            }
        }
        if (rc == FSX_OK && use_graph && hipGraphLaunch(g_gexec, g_stream) != hipSuccess)
            rc = FSX_ERR_HIP;
    }
    for (int i = 0; rc == FSX_OK && i < nprob; i++)
        rc = plan_download(&pl[i], g_stream, tail + 2 * i, tally + FSX_TALLY_N * i);
    if (hipStreamSynchronize(g_stream) != hipSuccess && rc == FSX_OK) rc = FSX_ERR_HIP;
    for (int i = 0; rc == FSX_OK && i < nprob; i++)
        plan_stats(&pl[i], &st[i], NULL, tail + 2 * i, tally + FSX_TALLY_N * i);
    if (rc != FSX_OK) graph_drop();
    for (int i = 0; i < ninit; i++) plan_free_host(&pl[i]);
    for (int i = 0; i < ncg; i++) free(cg[i].jobs);
    free(cg);
    free(fj);
    free(pl);
    free(tail);
    free(tally);
    free(key);
    return rc;
}

extern "C" int fsx_hip_run_batch(int nprob, const fsx_hip_args *args, fsx_stats *st)
{
    pthread_mutex_lock(&g_mtx);
    int rc = run_batch_locked(nprob, args, st);
    pthread_mutex_unlock(&g_mtx);
    return rc;
}

extern "C" int fsx_hip_fit_batch(const double *ct, int n, const double *qvals, int Q,
                                 const double *a, double mult, double c1_lo, double c1_hi,
                                 double c2_lo, double c2_hi, double *out)
{
    pthread_mutex_lock(&g_mtx);
    int rc = init_once();
    if (rc == FSX_OK) rc = ensure(B_FITCT, sizeof(double) * 6 * Q * (size_t)n);
    if (rc == FSX_OK) rc = ensure(B_FITOUT, sizeof(double) * 4 * (size_t)n);
    if (rc == FSX_OK) rc = ensure(B_Q, sizeof(double) * Q);
    if (rc == FSX_OK) rc = ensure(B_AM, sizeof(double) * 6 * Q);
    if (rc == FSX_OK) {
        hipStream_t s = g_stream;
        hipError_t e = hipMemcpyAsync(g_buf[B_FITCT], ct, sizeof(double) * 6 * Q * (size_t)n,
                                      hipMemcpyHostToDevice, s);
        if (e == hipSuccess) e = hipMemcpyAsync(g_buf[B_Q], qvals, sizeof(double) * Q, hipMemcpyHostToDevice, s);
        if (e == hipSuccess) e = hipMemcpyAsync(g_buf[B_AM], a, sizeof(double) * 6 * Q, hipMemcpyHostToDevice, s);
        if (e == hipSuccess) {
            hipLaunchKernelGGL(k_fit_batch, dim3(nblk(n, 256)), dim3(256),
                               (size_t)FSX_LB_KN * FSX_LB_KSTRIDE * sizeof(double), s,
                               (const double *)g_buf[B_FITCT], n, (const double *)g_buf[B_Q], Q,
                               (const double *)g_buf[B_AM], mult, c1_lo, c1_hi, c2_lo, c2_hi,
                               (double *)g_buf[B_FITOUT]);
            e = hipGetLastError();
        }
        if (e == hipSuccess) e = hipMemcpyAsync(out, g_buf[B_FITOUT], sizeof(double) * 4 * (size_t)n, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) {
            fprintf(stderr, "[fsx] fit batch: %s\n", hipGetErrorString(e));
            rc = FSX_ERR_HIP;
        }
    }
    pthread_mutex_unlock(&g_mtx);
    return rc;
}

extern "C" int fsx_hip_sbessel_batch(const double *x, int n, int pmax, double *out)
{
    pthread_mutex_lock(&g_mtx);
    int P = pmax + 1;
    int rc = init_once();
    if (rc == FSX_OK) rc = ensure(B_BX, sizeof(double) * n);
    if (rc == FSX_OK) rc = ensure(B_BOUT, sizeof(double) * (size_t)n * P);
    if (rc == FSX_OK) {
        hipStream_t s = g_stream;
        hipError_t e = hipMemcpyAsync(g_buf[B_BX], x, sizeof(double) * n, hipMemcpyHostToDevice, s);
        if (e == hipSuccess) {
            hipLaunchKernelGGL(k_sbessel_batch, dim3(nblk((long)n * P, 256)), dim3(256), 0, s,
                               (const double *)g_buf[B_BX], n, P, (double *)g_buf[B_BOUT]);
            e = hipGetLastError();
        }
        if (e == hipSuccess) e = hipMemcpyAsync(out, g_buf[B_BOUT], sizeof(double) * (size_t)n * P, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) {
            fprintf(stderr, "[fsx] sbessel batch: %s\n", hipGetErrorString(e));
            rc = FSX_ERR_HIP;
        }
    }
    pthread_mutex_unlock(&g_mtx);
    return rc;
}

/* Atom-expansion workspace: the per-chunk partial sums of all natoms atoms,
 * then the tables of one pass of atoms (Bessel table, f, r, conj(Y)). */
static inline int at_qp(int Q) { return (Q + 15) / 16 * 16; }
static inline size_t at_part_bytes(int natoms, int Q, int L)
{
    const size_t Kh = (size_t)(L + 1) * (L + 2) / 2, nch = ((size_t)natoms + FSX_AT_CHUNK - 1) / FSX_AT_CHUNK;
    return (nch * 3 * at_qp(Q) * Kh * 2 * sizeof(double) + 255) & ~(size_t)255;
}
static inline size_t at_atom_bytes(int Q, int L)
{
    const size_t K = L + 1, Kh = K * (K + 1) / 2;
    return sizeof(double) * (K * at_qp(Q) + 4 + 2 * Kh);
}

/* The expansion of natoms atoms (device inputs) into re/im [3][Q][(L+1)^2]
 * (device), on stream s, in ws (ws_bytes): passes of as many whole chunks of
 * atoms as the workspace holds. */
static int atoms_run(hipStream_t s, char *ws, size_t ws_bytes, int natoms, const double *xyz,
                     const double *vac, const double *dum, const double *sa, double h2o_ff,
                     const double *qv, int Q, int L, double *re, double *im)
{
    const int K = L + 1, Kh = K * (K + 1) / 2, Qp = at_qp(Q);
    const int nch = (natoms + FSX_AT_CHUNK - 1) / FSX_AT_CHUNK;
    const size_t pb = at_part_bytes(natoms, Q, L), per = at_atom_bytes(Q, L);
    if (ws_bytes < pb + per * FSX_AT_CHUNK && ws_bytes < pb + per * (size_t)natoms) return FSX_ERR_ARG;
    long npass = (long)((ws_bytes - pb) / per) / FSX_AT_CHUNK * FSX_AT_CHUNK;
    if (npass < 1) npass = natoms;   /* a single pass of fewer than one chunk of atoms */
    if (npass > natoms) npass = natoms;
    double *P = reinterpret_cast<double *>(ws);
    double *J = reinterpret_cast<double *>(ws + pb);
    double *f = J + (size_t)K * npass * Qp, *r = f + 3 * (size_t)npass, *Y = r + npass;
    for (long a0 = 0; a0 < natoms; a0 += npass) {
        const int na = (int)(natoms - a0 < npass ? natoms - a0 : npass);
        hipLaunchKernelGGL(k_atom_geom, dim3(nblk((long)na * K, 256)), dim3(256), 0, s, xyz + 3 * a0,
                           vac + a0, dum + a0, sa ? sa + a0 : (const double *)NULL, h2o_ff, na, L,
                           FSX_PI_REFERENCE, r, f, Y);
        const unsigned nbl = nblk((long)na * Q, 256);
        hipLaunchKernelGGL(k_atom_bes, dim3(nbl * K), dim3(256), 0, s, J, (const double *)r, qv, na, Q,
                           nbl);
        const int nchp = (na + FSX_AT_CHUNK - 1) / FSX_AT_CHUNK;
        int ncg = 0;
        for (int l = 0; l <= L; l++) ncg += at_colgroups(l);
        const int nqg = (Qp / 16 + FSX_AT_QT - 1) / FSX_AT_QT;
        hipLaunchKernelGGL(k_atom_mfma, dim3((unsigned)(nchp * ncg * nqg)), dim3(256), 0, s,
                           (const double *)J, (const double *)f, (const double *)Y, P, na, Q, Qp, L,
                           (int)(a0 / FSX_AT_CHUNK));
    }
    hipLaunchKernelGGL(k_atom_finish, dim3(nblk(3L * Q * Kh, 256)), dim3(256), 0, s,
                       (const double *)P, nch, re, im, Q, Qp, L, 4.0 * FSX_PI_REFERENCE);
    return hipGetLastError() == hipSuccess ? FSX_OK : FSX_ERR_HIP;
}

/* The mixed form of atoms_run in one pass over all atoms: the BF16 parts of
 * the Bessel values and of f conj(Y_lm), then the split products on BF16
 * MFMA.  Workspace: the chunk partials, then per atom (padded to whole
 * chunks) f, r, Y in FP64 and the parts. */
static inline size_t at_bf16_atom_bytes(int Q, int L)
{
    const size_t K = L + 1, Kh = K * (K + 1) / 2;
    return sizeof(double) * (4 + 2 * Kh) + 3 * sizeof(__bf16) * (K * at_qp(Q) + 6 * Kh);
}
static int atoms_run_bf16(hipStream_t s, char *ws, size_t ws_bytes, int natoms,
                          const double *xyz, const double *vac, const double *dum,
                          const double *sa, double h2o_ff, const double *qv, int Q, int L,
                          double *re, double *im)
{
    const int K = L + 1, Kh = K * (K + 1) / 2, Qp = at_qp(Q);
    const int nch = (natoms + FSX_AT_CHUNK - 1) / FSX_AT_CHUNK, nap = nch * FSX_AT_CHUNK;
    const size_t pb = at_part_bytes(natoms, Q, L);
    if (ws_bytes < pb + at_bf16_atom_bytes(Q, L) * (size_t)nap) return FSX_ERR_ARG;
    double *P = reinterpret_cast<double *>(ws);
    double *f = reinterpret_cast<double *>(ws + pb), *r = f + 3 * (size_t)natoms;
    double *Y = r + natoms;
    __bf16 *Js = reinterpret_cast<__bf16 *>(Y + (size_t)natoms * Kh * 2);
    __bf16 *Bs = Js + 3 * (size_t)K * Qp * nap;
    hipLaunchKernelGGL(k_atom_geom, dim3(nblk((long)natoms * K, 256)), dim3(256), 0, s, xyz, vac, dum, sa,
                       h2o_ff, natoms, L, FSX_PI_REFERENCE, r, f, Y);
    hipLaunchKernelGGL(k_atom_bes_split, dim3(nblk((long)K * Qp * nap, 256)), dim3(256), 0, s, Js,
                       (const double *)r, qv, natoms, nap, Q, Qp, K);
    hipLaunchKernelGGL(k_atom_bsplit, dim3(nblk(6L * Kh * nap, 256)), dim3(256), 0, s, Bs,
                       (const double *)f, (const double *)Y, natoms, nap, L);
    hipLaunchKernelGGL(k_atom_bf16, dim3((unsigned)(nch * K * (Qp / 16))), dim3(256), 0, s,
                       (const __bf16 *)Js, (const __bf16 *)Bs, P, nap, Qp, L, 0);
    hipLaunchKernelGGL(k_atom_finish, dim3(nblk(3L * Q * Kh, 256)), dim3(256), 0, s,
                       (const double *)P, nch, re, im, Q, Qp, L, 4.0 * FSX_PI_REFERENCE);
    return hipGetLastError() == hipSuccess ? FSX_OK : FSX_ERR_HIP;
}

extern "C" int fsx_hip_atoms2spf(int natoms, const double *xyz, const double *vac,
                                 const double *dum, const double *sa, double h2o_ff,
                                 const double *qvals, int Q, int L, double *re, double *im,
                                 int bf16)
{
    pthread_mutex_lock(&g_mtx);
    const int K = L + 1, K2 = K * K;
    const size_t nap = ((size_t)natoms + FSX_AT_CHUNK - 1) / FSX_AT_CHUNK * FSX_AT_CHUNK;
    const size_t wsb = at_part_bytes(natoms, Q, L) +
                       (bf16 ? at_bf16_atom_bytes(Q, L) * nap : at_atom_bytes(Q, L) * (size_t)natoms);
    int rc = init_once();
    if (rc == FSX_OK) rc = ensure(B_AXYZ, sizeof(double) * 3 * (size_t)natoms);
    if (rc == FSX_OK) rc = ensure(B_AFF, sizeof(double) * 3 * (size_t)natoms);
    if (rc == FSX_OK) rc = ensure(B_AWS, wsb);
    if (rc == FSX_OK) rc = ensure(B_AQ, sizeof(double) * Q);
    if (rc == FSX_OK) rc = ensure(B_ARE, sizeof(double) * 3 * (size_t)Q * K2);
    if (rc == FSX_OK) rc = ensure(B_AIM, sizeof(double) * 3 * (size_t)Q * K2);
    if (rc == FSX_OK) {
        hipStream_t s = g_stream;
        double *dff = (double *)g_buf[B_AFF];
        const size_t nb = sizeof(double) * (size_t)natoms;
        hipError_t e = hipMemcpyAsync(g_buf[B_AXYZ], xyz, 3 * nb, hipMemcpyHostToDevice, s);
        if (e == hipSuccess) e = hipMemcpyAsync(dff, vac, nb, hipMemcpyHostToDevice, s);
        if (e == hipSuccess) e = hipMemcpyAsync(dff + natoms, dum, nb, hipMemcpyHostToDevice, s);
        if (e == hipSuccess && sa) e = hipMemcpyAsync(dff + 2 * (size_t)natoms, sa, nb, hipMemcpyHostToDevice, s);
        if (e == hipSuccess) e = hipMemcpyAsync(g_buf[B_AQ], qvals, sizeof(double) * Q, hipMemcpyHostToDevice, s);
        if (e == hipSuccess) {
            rc = (bf16 ? atoms_run_bf16 : atoms_run)(
                s, (char *)g_buf[B_AWS], g_cap[B_AWS], natoms, (const double *)g_buf[B_AXYZ], dff,
                dff + natoms, sa ? dff + 2 * (size_t)natoms : NULL, h2o_ff,
                (const double *)g_buf[B_AQ], Q, L, (double *)g_buf[B_ARE], (double *)g_buf[B_AIM]);
            if (rc == FSX_ERR_HIP) e = hipErrorUnknown;
        }
        if (e == hipSuccess && rc == FSX_OK)
            e = hipMemcpyAsync(re, g_buf[B_ARE], sizeof(double) * 3 * (size_t)Q * K2, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess && rc == FSX_OK)
            e = hipMemcpyAsync(im, g_buf[B_AIM], sizeof(double) * 3 * (size_t)Q * K2, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) {
            fprintf(stderr, "[fsx] atoms2spf: %s\n", hipGetErrorString(e));
            rc = FSX_ERR_HIP;
        }
    }
    pthread_mutex_unlock(&g_mtx);
    return rc;
}

/* The atom expansion on caller-owned device arrays with no allocation: its
 * tables and chunk partials live in the fixed scratch array.  Nothing there
 * needs clearing first: every pass writes its tables whole, and every chunk
 * partial is written (all of (X, q, l, m, part)) before the final sum reads
 * it.  The library's lock orders calls from several threads of one process. */
extern "C" int fsx_atoms2spf_noalloc(int natoms, const double *coords, const double *vac,
                                     const double *dum, const double *sa, double h2o_ff,
                                     const double *qvals, int qnum, int L, double *re, double *im)
{
    if (natoms < 1 || !coords || !vac || !dum || !qvals || qnum < 1 || L < 0 || L > 40 || !re ||
        !im)
        return FSX_ERR_ARG;
    const size_t need = at_part_bytes(natoms, qnum, L) +
                        at_atom_bytes(qnum, L) * (size_t)(natoms < FSX_AT_CHUNK ? natoms : FSX_AT_CHUNK);
    if (need > FSX_NOALLOC_SCRATCH_BYTES) {
        fprintf(stderr, "[fsx] atoms2spf_noalloc: %d atoms at L = %d with %d q need %zu bytes of "
                "working memory, more than the %zu-byte scratch array\n", natoms, L, qnum, need,
                FSX_NOALLOC_SCRATCH_BYTES);
        return FSX_ERR_SCRATCH;
    }
    pthread_mutex_lock(&g_mtx);
    int rc = init_once();
    if (rc == FSX_OK) {
        rc = atoms_run(g_stream, (char *)g_scratch, FSX_NOALLOC_SCRATCH_BYTES, natoms, coords, vac,
                       dum, sa, sa ? h2o_ff : 0.0, qvals, qnum, L, re, im);
        const hipError_t e = hipStreamSynchronize(g_stream);
        if (rc == FSX_OK && e != hipSuccess) {
            fprintf(stderr, "[fsx] atoms2spf_noalloc: %s\n", hipGetErrorString(e));
            rc = FSX_ERR_HIP;
        }
    }
    pthread_mutex_unlock(&g_mtx);
    return rc;
}

