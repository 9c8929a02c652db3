/*
 * fsx_cross.h -- the per-pose cross terms (device code, included by
 * fsx_kernels.hip).
 *
 * Work item of one block: one q and one fsx_unit, a run of poses with the same
 * (z, beta2) on at most FSX_UROWS different gamma2 (the poses are sorted by z and
 * beta2, either of them first, and gamma2, so a unit is a range of the sorted
 * records).  The block
 *   1. translates the unit's ligand rows on the matrix cores,
 *        U^Y_lm(row) = sum_{l1 >= |m|} tau^{|m|}_{l l1}(q z) B^Y_{l1 m}(row),
 *      per m one matrix product with 16 rows (ligand row, re/im) for each of Y
 *      = V, D, W and l in the columns, the m values dealt to the wavefronts,
 *      and puts U into LDS;
 *   2. pairs U with the receptor row of each pose (one or two poses per wavefront,
 *      the coefficient slots across its lanes),
 *        2 Re sum_e e^{-i m a2} (R^X_e U^Y_e [+ R^Y_e U^X_e]),
 *      and writes the six sums, or adds them to those of earlier m-chunks.
 * The products take 16 rows whether the unit has them or not (rows past nrow repeat
 * row 0).  What bounds it depends on the poses per unit: with many (210,000 poses at
 * L = 15: 38 to a unit) the receptor rows, 6 KB (FP64) or 3 KB per pose and q, most
 * of which an XCD's 4 MB L2 does not hold in FP64; with few (200,000 to 300,000 on a
 * 37 x 128 grid of 0.5 A steps at L = 25: about 10) the loads and waits of an item's
 * chain, unit, operands, products, rows.  The form before it, tiles of adjacent
 * gamma2 with all z inside and the translation on the vector units, translated every
 * row of a tile for every z in use and read 100 bytes of LDS per lane for 24
 * multiply-adds.  Cross terms of that form and of this one: L = 25, 81 q, 300,000
 * poses FP32 224 and 64 ms, 200,000 poses FP64 219 and 143; L = 15, 51 q, 210,000
 * poses FP32 4.7 and 4.4, FP64 9.65 and 9.15; crowded buckets FP64, 1,000,000 poses
 * at L = 15 28.7 and 28.7, 2,500,000 at L = 25 645 and 657.
 */
#ifndef FSX_CROSS_H
#define FSX_CROSS_H

#define FSX_UROWS 8           /* most gamma2 rows of a unit */
#define FSX_UPOSES 256        /* most poses of a unit: one per thread */
#define FSX_UBATCH 64         /* poses paired between two writes of their sums */
#define FSX_CROSS_BLOCK 256

/* poses p0 .. p0 + n - 1 of the sorted records; row r (gamma2 g2[r]) holds the
 * poses from cum[r] on (relative to p0); rows past nrow repeat row 0 */
struct fsx_unit {
    int p0, n, z, b2;
    int g2[FSX_UROWS];
    unsigned cum[FSX_UROWS / 4];   /* a byte each */
    int nrow, pad;
};
static_assert(sizeof(fsx_unit) == 64, "one unit per 64-byte line");
static_assert(FSX_UPOSES == FSX_CROSS_BLOCK && FSX_UBATCH == 64, "a wavefront holds a batch's records");

/* One tile of the translation: up to FSX_CROSS_TILE l of one m.  Its operands are nks
 * steps from value bo of a ligand row and from value to of a translation block;
 * the l of entries e + lo .. e + hi - 1 of the chunk are stored.  A step takes 4
 * l1, in a split tile (odd > 0, FP64) 4 even and 4 odd l1 - |m|, summed apart
 * and added at the end (odd: the odd ones' distance in the ligand row).  The
 * FP64 matrix products being chains of fused multiply-adds in ascending order
 * (checked on 262,144 random 4x4x4 products), this keeps the order in which the
 * rows of the longer blocks were summed by pairs of lanes, bit for bit: the
 * fit's stopping tests amplify the last bit of a profile to 1e-7 of c2 in some
 * fits. */
struct fsx_tile {
    int bo, to, e, nks, odd, lo, hi, packed;
};

/* one launch: the nc entries (from entry cstart) of a chunk, every unit and q */
struct fsx_cross_job {
    double *acc;
    const void *R, *B, *T, *tw2;   /* tables of the chunk (R, B), of all m (T, tw2) */
    const fsx_tile *tiles;         /* the chunk's translation */
    const int *el, *em;            /* l and m of each entry */
    const fsx_unit *units;
    const int *tail;               /* tail[2]: number of units */
    const int4 *recs;
    int Q, L, nrows, ng, zn, Tn, ntiles, cstart, nc, npk, rsB, first, nx, urows, mirror, nbeta;
};

/* Uniform reads of tables that no one writes during a launch go through the
 * constant address space, to come as scalar loads: through ordinary pointers the
 * compiler has to assume that the sums' stores change them and takes vector
 * loads, whose waits also catch the operands in flight (L = 25, 300,000 poses FP32:
 * 75 against 67 ms). */
#define FSX_CONST __attribute__((address_space(4)))
template <typename T>
__device__ __forceinline__ const FSX_CONST T *fsx_const(const T *p) { return (const FSX_CONST T *)p; }

typedef float fsx_f4 __attribute__((ext_vector_type(4)));

/* Row stride (in complex elements) of U in LDS: FP32 the slots rounded up so that
 * the rows written by one matrix instruction (128 contiguous bytes of rows 6
 * strides apart) fall on different banks; FP64 one more than the slots, which
 * leaves room for three blocks of 8 rows at L = 15 */
template <typename F>
__host__ __device__ __forceinline__ int cross_us(int ns)
{
    return sizeof(F) == 4 ? (ns + 7) / 16 * 16 + 8 : ns + 1;
}
/* LDS of a block: U [urows][3][cross_us] complex, the unit's records (int2) and
 * sums (6 per pose) */
template <typename F>
__host__ __device__ __forceinline__ size_t cross_lds(int ns, int urows)
{
    return sizeof(F) * (2 * 3 * (size_t)urows * cross_us<F>(ns) + 6 * FSX_UBATCH) +
           sizeof(int2) * FSX_UBATCH;
}

/* l per translation tile: FP32 one 16x16x4 product, FP64 four 4x4x4 */
#define FSX_CROSS_TILE 16

/* Steps of a K x K block in natural order of l1 or split by parity, and values
 * per step of a tile of the translation table */
__host__ __device__ __forceinline__ int cross_steps(int K, int split)
{
    return split ? ((K + 1) / 2 + 3) / 4 : (K + 3) / 4;
}
__host__ __device__ __forceinline__ int cross_tstep(int split) { return 4 * FSX_CROSS_TILE << split; }

/* Workgroup barrier that orders LDS accesses only: unlike __syncthreads it
 * does not wait for the block's outstanding global stores (the cross-term
 * accumulator writes, which no other thread of the launch reads), so they
 * drain while the block goes on. */
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

/* a double moved between lanes by a DPP pattern (row_ror:8 = lane xor 8,
 * row_half_mirror = lane 7 - i in each group of 8, quad_perm) */
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double v)
{
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)u, CTRL, 0xf, 0xf, false);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), CTRL, 0xf, 0xf, false);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL,
                                                                 0xf, 0xf, false));
}
#define FSX_DPP_ROR8 0x128
#define FSX_DPP_HMIRROR 0x141
#define FSX_DPP_XOR1 0xB1
#define FSX_DPP_XOR2 0x4E

/* Cross-lane steps of the 64-lane transpose-reduce, on the two 32-bit halves
 * of a double.  v_permlane32_swap exchanges lanes 32..63 of its first operand
 * with lanes 0..31 of its second, v_permlane16_swap the odd 16-lane rows of
 * the first with the even rows of the second, so that the sum of the two
 * results is, in every lane, its own slot's value plus the partner lane's
 * value of the same slot (lanes below the split keep slot a, lanes above it
 * slot b). */
__device__ __forceinline__ double tr_swap32(double a, double b)
{
    const unsigned long long ua = __builtin_bit_cast(unsigned long long, a);
    const unsigned long long ub = __builtin_bit_cast(unsigned long long, b);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)ua, (unsigned)ub, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(ua >> 32), (unsigned)(ub >> 32),
                                                     false, false);
    const double r0 = __builtin_bit_cast(double, ((unsigned long long)hi[0] << 32) | lo[0]);
    const double r1 = __builtin_bit_cast(double, ((unsigned long long)hi[1] << 32) | lo[1]);
    return r0 + r1;
}
__device__ __forceinline__ double tr_swap16(double a, double b)
{
    const unsigned long long ua = __builtin_bit_cast(unsigned long long, a);
    const unsigned long long ub = __builtin_bit_cast(unsigned long long, b);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)ua, (unsigned)ub, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(ua >> 32), (unsigned)(ub >> 32),
                                                     false, false);
    const double r0 = __builtin_bit_cast(double, ((unsigned long long)hi[0] << 32) | lo[0]);
    const double r1 = __builtin_bit_cast(double, ((unsigned long long)hi[1] << 32) | lo[1]);
    return r0 + r1;
}
__device__ __forceinline__ float tr_swap32(float a, float b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a),
                                                    __builtin_bit_cast(unsigned, b), false, false);
    return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}
__device__ __forceinline__ float tr_swap16(float a, float b)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a),
                                                    __builtin_bit_cast(unsigned, b), false, false);
    return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}

/* ---- translation tiles ----
 * begin(): the lane's places in the unit's ligand rows and the translation
 * block; load(): the first operands of a tile; run(): its products (loading the
 * rest); store(): U to LDS, entry e of the chunk in slot e - npk, the packed m =
 * 0 entries (real) in the halves of slot e / 2.  Loads past a tile's last step
 * read the table's next values (in bounds: the tables are longer by
 * FSX_TAB_PAD), which the products leave out. */
#define FSX_TAB_PAD 512

/* FP32: 16x16x4 (lane i feeds A[i % 16][i / 16] and B[i / 16][i % 16]; result j of
 * lane i is D[4 (i / 16) + j][i % 16]).  Rows are (ligand row, re/im): the lane
 * holds re and im of rows 2h and 2h + 1, h = i / 16, at l = i % 16. */
struct cross_u32 {
    enum { UK = 4 };
    const float *Bq, *Tq;
    float sg;   /* sign of the lane's ligand values: a mirrored row's are (-1)^(l1 + m) conj */
    float b[UK][3], t[UK];
    fsx_f4 c[3];
    __device__ __forceinline__ void begin(const float *B, size_t row0, const int *g2, int rsB, bool mir,
                                          int ng, const float *T, int lane)
    {
        int g = g2[(lane & 15) >> 1];
        if (mir) g += 2 * g >= ng ? -(ng / 2) : ng / 2;
        Bq = B + (row0 + g) * rsB + (lane & 1) * 3 + (lane >> 4) * 6;
        Tq = T + lane;
        sg = mir && ((lane >> 4) + lane & 1) ? -1.f : 1.f;
    }
    __device__ __forceinline__ void ops(const float *Bp, const float *Tp)
    {
#pragma unroll
        for (int s = 0; s < UK; s++) {
#pragma unroll
            for (int Y = 0; Y < 3; Y++) b[s][Y] = Bp[s * 24 + Y];
            t[s] = Tp[s * 64];
        }
    }
    __device__ __forceinline__ void load(const fsx_tile &tl, int) { ops(Bq + tl.bo, Tq + tl.to); }
    __device__ __forceinline__ void run(const fsx_tile &tl, int)
    {
        const float *Bp = Bq + tl.bo, *Tp = Tq + tl.to;
#pragma unroll
        for (int Y = 0; Y < 3; Y++) c[Y] = (fsx_f4){0.f, 0.f, 0.f, 0.f};
        for (int k0 = 0; k0 < tl.nks; k0 += UK) {
#pragma unroll
            for (int s = 0; s < UK; s++)
                if (k0 + s < tl.nks) {
#pragma unroll
                    for (int Y = 0; Y < 3; Y++)
                        c[Y] = __builtin_amdgcn_mfma_f32_16x16x4f32(sg * b[s][Y], t[s], c[Y], 0, 0, 0);
                }
            if (k0 + UK < tl.nks) ops(Bp + (k0 + UK) * 24, Tp + (k0 + UK) * 64);
        }
    }
    __device__ __forceinline__ void store(const fsx_tile &tl, cplx32 *sU, int us, int npk, int urows,
                                          int lane)
    {
        const int h4 = lane >> 4, l = lane & 15, e = tl.e + l;
        if (l < tl.lo || l >= tl.hi || 2 * h4 >= urows) return;
        cplx32 *d = sU + h4 * 6 * us;
        if (tl.packed && e < 2 * npk) {
            float *f = reinterpret_cast<float *>(d) + e;
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int Y = 0; Y < 3; Y++) f[(3 * r + Y) * 2 * us] = e & 1 ? -c[Y][2 * r] : c[Y][2 * r];
        } else {
            d += e - npk;
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int Y = 0; Y < 3; Y++) {
                    cplx32 v;
                    v.re = c[Y][2 * r];
                    v.im = c[Y][2 * r + 1];
                    d[(3 * r + Y) * us] = v;
                }
        }
    }
};

/* FP64: four blocks of 4x4x4 (lane i feeds A[i % 4][i / 16] and B[i / 16][i % 4] of
 * block i / 4 % 4, and holds D[i / 16][i % 4] of it), at 1.4 times the rate of
 * 16x16x4 (13.3 against 9.8 multiply-adds per clock and SIMD, measured).
 * Natural order: block b takes the rows (re, im) of ligand rows 2b and 2b + 1.
 * Split: blocks 0 and 1 take the even l1, 2 and 3 the odd ones, of ligand rows 0..3
 * and, in a second product, 4..7. */
struct cross_u64 {
    enum { UK = 1, NT = 4 };
    const double *Bq, *Tq;             /* natural order */
    const double *Bs0, *Bs1, *Ts;      /* split: rows 0..3, rows 4..7 */
    double b[UK][2][3], t[UK][NT];
    double c[2][NT][3];
    __device__ __forceinline__ void begin(const double *B, size_t row0, const int *g2, int rsB, bool, int,
                                          const double *T, int lane)
    {
        const int h4 = lane >> 4, r4 = (lane & 7) >> 1, in = (lane & 1) * 3 + h4 * 6;
        Bq = B + (row0 + g2[(lane & 15) >> 1]) * rsB + in;
        Bs0 = B + (row0 + g2[r4]) * rsB + in;
        Bs1 = B + (row0 + g2[r4 + 4]) * rsB + in;
        Tq = T + (h4 * 4 + (lane & 3)) * NT;
        Ts = T + (((lane >> 3 & 1) * 4 + h4) * 4 + (lane & 3)) * NT;
    }
    __device__ __forceinline__ void ops(const fsx_tile &tl, int k0, int lane, bool two)
    {
        if (tl.odd) {
            const int o = tl.bo + (lane & 8 ? tl.odd : 0) + k0 * 24;
#pragma unroll
            for (int s = 0; s < UK; s++) {
#pragma unroll
                for (int Y = 0; Y < 3; Y++) b[s][0][Y] = Bs0[o + s * 24 + Y];
                if (two) {
#pragma unroll
                    for (int Y = 0; Y < 3; Y++) b[s][1][Y] = Bs1[o + s * 24 + Y];
                }
#pragma unroll
                for (int k = 0; k < NT; k++) t[s][k] = Ts[tl.to + (k0 + s) * 128 + k];
            }
        } else {
#pragma unroll
            for (int s = 0; s < UK; s++) {
#pragma unroll
                for (int Y = 0; Y < 3; Y++) b[s][0][Y] = Bq[tl.bo + (k0 + s) * 24 + Y];
#pragma unroll
                for (int k = 0; k < NT; k++) t[s][k] = Tq[tl.to + (k0 + s) * 64 + k];
            }
        }
    }
    __device__ __forceinline__ void load(const fsx_tile &tl, int urows)
    {
        ops(tl, 0, threadIdx.x & 63, urows > 4);
    }
    __device__ __forceinline__ void run(const fsx_tile &tl, int urows)
    {
        const bool two = tl.odd && urows > 4;
        const int nsub = (tl.hi + 3) >> 2;
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int k = 0; k < NT; k++)
#pragma unroll
                for (int Y = 0; Y < 3; Y++) c[r][k][Y] = 0.0;
        for (int k0 = 0; k0 < tl.nks; k0 += UK) {
#pragma unroll
            for (int s = 0; s < UK; s++)
                if (k0 + s < tl.nks) {
#pragma unroll
                    for (int k = 0; k < NT; k++)
                        if (k < nsub) {
#pragma unroll
                            for (int Y = 0; Y < 3; Y++)
                                c[0][k][Y] = __builtin_amdgcn_mfma_f64_4x4x4f64(b[s][0][Y], t[s][k], c[0][k][Y], 0, 0, 0);
                            if (two) {
#pragma unroll
                                for (int Y = 0; Y < 3; Y++)
                                    c[1][k][Y] = __builtin_amdgcn_mfma_f64_4x4x4f64(b[s][1][Y], t[s][k], c[1][k][Y], 0, 0, 0);
                            }
                        }
                }
            if (k0 + UK < tl.nks) ops(tl, k0 + UK, threadIdx.x & 63, urows > 4);
        }
    }
    __device__ __forceinline__ void store(const fsx_tile &tl, cplx *sU, int us, int npk, int urows, int lane)
    {
        const int h4 = lane >> 4, part = h4 & 1;
        int row = 2 * ((lane >> 2) & 3) + (h4 >> 1);
        if (tl.odd) {
            /* lanes of even l1 finish rows 0..3, those of odd l1 rows 4..7, each
             * with the other parity's sum from lane xor 8 */
            const bool hi = (lane & 8) != 0;
            row = 2 * ((lane >> 2) & 1) + (h4 >> 1) + (hi ? 4 : 0);
#pragma unroll
            for (int k = 0; k < NT; k++)
#pragma unroll
                for (int Y = 0; Y < 3; Y++) {
                    const double keep = hi ? c[1][k][Y] : c[0][k][Y], send = hi ? c[0][k][Y] : c[1][k][Y];
                    c[0][k][Y] = keep + dpp_mov<FSX_DPP_ROR8>(send);
                }
        }
        if (row >= urows) return;
        double *d = reinterpret_cast<double *>(sU + row * 3 * us);
#pragma unroll
        for (int k = 0; k < NT; k++) {
            const int l = 4 * k + (lane & 3), e = tl.e + l;
            if (l >= tl.lo && l < tl.hi) {
                if (tl.packed && e < 2 * npk) {
                    if (part == 0) {
#pragma unroll
                        for (int Y = 0; Y < 3; Y++) d[Y * 2 * us + e] = e & 1 ? -c[0][k][Y] : c[0][k][Y];
                    }
                } else {
#pragma unroll
                    for (int Y = 0; Y < 3; Y++) d[Y * 2 * us + 2 * (e - npk) + part] = c[0][k][Y];
                }
            }
        }
    }
};

/* J: slots per lane; PW: poses per wavefront */
template <int J, typename E, int PW>
__device__ __forceinline__ void cross_body(const fsx_cross_job &A)
{
#pragma clang fp contract(fast)
    typedef decltype(E::re) F;   /* arithmetic type of the contraction */
    extern __shared__ double smem_raw[];
    const int L = A.L, N = 2 * L + 1, Q = A.Q, npk = A.npk, ns = A.nc - npk;
    const int us = cross_us<F>(ns);
    E *sU = reinterpret_cast<E *>(smem_raw);             /* [urows][3][us] */
    int2 *sP = reinterpret_cast<int2 *>(sU + 3 * A.urows * us);
    F *sO = reinterpret_cast<F *>(sP + FSX_UBATCH);
    const int tid = threadIdx.x, lane = tid & (FSX_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / FSX_WAVE);
    const int nwave = FSX_CROSS_BLOCK / FSX_WAVE;
    /* pairing: PW poses per wavefront of LP lanes each, lane sl of a pose taking
     * slots sl, sl + LP, ... (J per lane).  With npk > 0 (conjugate-symmetric
     * coefficients, the chunk of m = 0) the m = 0 entries l = 2i and 2i + 1 share
     * slot i, both real after the turns by i^l and i^-l: the real part of the slot
     * is the first, the imaginary part the second (negated in U, so that Re(R U) of
     * the slot adds the two products); their twiddle is 1. */
    constexpr int LP = FSX_WAVE / PW;
    const int sl = lane % LP, half = lane / LP;
    const unsigned rstride = 3u * (unsigned)ns * (unsigned)sizeof(E);
    const unsigned ustride = 3u * (unsigned)us * (unsigned)sizeof(E);
    const unsigned soff = (unsigned)(sl * sizeof(E));
    /* the step to the lane's last slot (back to slot 0 when past the end) */
    const unsigned dlast = sl + LP * (J - 1) < ns ? (unsigned)(LP * (J - 1) * sizeof(E))
                                                  : (unsigned)0 - soff;
    /* byte offset of each slot's twiddle e^(-i m alpha2) within a row of tw2:
     * entries m = -L..L and a zero at 2L + 1, which a slot past the last one
     * reads; with mirrored rows (fsx_mirror), rows 2 alpha2 + x of one entry per
     * (m, (l + m) mod 2), x = 1 the poses with a mirrored receptor row (negative
     * for odd l + m) */
    const int twk = A.mirror ? 2 : 1;
    const unsigned twstride = (unsigned)(twk * (N + 1) * sizeof(E));
    unsigned emo[J];
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int ec = sl + LP * j, e = A.cstart + (ec < npk ? 2 * ec : ec + npk);
        const int m = ec < ns ? A.em[e] : L + 1;
        const int odd = A.mirror && ec >= npk && ec < ns ? (A.el[e] + m) & 1 : 0;
        emo[j] = (unsigned)((m + L) * twk + odd) * (unsigned)sizeof(E);
    }
    /* after the lane reduction: one pose: lanes 0, 8, .., 40 hold the six sums;
     * two poses: lanes 0, 8, 4, 16, 24, 20 of each half (bits 4, 3, 2 of the
     * lane select sum 3 b4 + (b2 ? 2 : b3)) */
    const bool b4 = lane & 16, b3 = lane & 8, b2 = lane & 4;
    const int slot = PW == 1 ? lane >> 3 : (b4 ? 3 : 0) + (b2 ? 2 : b3);
    const bool writer = PW == 1 ? (lane & 7) == 0 && slot < 6 : (lane & 3) == 0 && !(b2 && b3);
    const E *tw2 = reinterpret_cast<const E *>(A.tw2);
    /* items (q, unit) in nx contiguous ranges, one per XCD (blocks go to the
     * XCDs round-robin), each walked by that XCD's blocks together: at any
     * time they read the receptor rows of one q and the ligand rows of a few
     * beta2, which the XCD's L2 holds */
    const long nunits = fsx_const(A.tail)[2], items = nunits * Q;
    const int nx = A.nx, nw = gridDim.x / nx;
    const long per = (items + nx - 1) / nx;
    const long i0 = (blockIdx.x % nx) * per, i1 = i0 + per < items ? i0 + per : items;
    long it = i0 + blockIdx.x / nx;
    if (it >= i1) return;
    int q = (int)(it / nunits), uidx = (int)(it - q * nunits);
    /* what an item's start needs is read during the item before it: the unit,
     * the record of pose tid and the first operands of the wavefront's
     * translation */
    const FSX_CONST fsx_unit *u = fsx_const(A.units) + uidx;
    int4 rpf = make_int4(0, 0, 0, 0);
    if (tid < u->n) rpf = A.recs[u->p0 + tid];
    typename std::conditional<sizeof(F) == 4, cross_u32, cross_u64>::type U;
    /* translation tiles, dealt to the wavefronts in turn */
    int ti = 0;
    fsx_tile tl;
    auto tile_load = [&]() {
        const FSX_CONST fsx_tile *x = fsx_const(A.tiles) + ti;
        tl.bo = x->bo; tl.to = x->to; tl.e = x->e; tl.nks = x->nks;
        tl.odd = x->odd; tl.lo = x->lo; tl.hi = x->hi; tl.packed = x->packed;
        U.load(tl, A.urows);
    };
    auto item_begin = [&]() {
        const bool mir = A.mirror && u->b2 > (A.nbeta - 1) / 2;
        const int b2 = mir ? A.nbeta - 1 - u->b2 : u->b2;
        U.begin(reinterpret_cast<const F *>(A.B), (size_t)q * A.nrows + b2 * A.ng, A.units[uidx].g2, A.rsB, mir,
                A.ng, reinterpret_cast<const F *>(A.T) + ((size_t)u->z * Q + q) * A.Tn, lane);
        ti = wave;
        if (ti < A.ntiles) tile_load();
    };
    item_begin();
    for (;;) {
        const int p0 = u->p0, n = u->n;
        /* the record of pose tid: (receptor row, 8 alpha2 + row of the unit) */
        const int nrow = u->nrow;
        int r = 0;
#pragma unroll
        for (int k = 1; k < FSX_UROWS; k++) r += k < nrow && tid >= (int)(u->cum[k / 4] >> k % 4 * 8 & 255);
        const int2 mine = make_int2(rpf.y, (rpf.z << 3) | r);
        if (tid < FSX_UBATCH) sP[tid] = mine;
        /* ---- translation ---- */
        while (ti < A.ntiles) {
            const fsx_tile ct = tl;
            U.run(ct, A.urows);
            /* the next tile's first operands arrive while this one is stored */
            ti += nwave;
            if (ti < A.ntiles) tile_load();
            U.store(ct, sU, us, npk, A.urows, lane);
        }
        lds_barrier();
        /* the next item */
        it += nw;
        const bool more = it < i1;
        const int qc = q;
        if (more) {
            for (uidx += nw; uidx >= (int)nunits; uidx -= (int)nunits) q++;
            u = fsx_const(A.units) + uidx;
            if (tid < u->n) rpf = A.recs[u->p0 + tid];
            item_begin();
        }
        /* ---- pairing ---- */
        const char *RqB = reinterpret_cast<const char *>(A.R) + (size_t)qc * A.nrows * rstride;
        for (int pb = 0;;) {
        const int nb = min(n - pb, FSX_UBATCH);
        /* PW poses per step; one past the batch's last repeats some earlier
         * record of sP (in bounds), and nothing reads its sums */
        for (int pp = wave; PW * pp < nb; pp += nwave) {
            const int p = PW * pp + half;
            const int2 rec = sP[p];
            const int prow = rec.y & 7;
            E rr[3][J];
            F wr[J], wi[J];
            /* no branches, so that the J slots' loads are all in flight
             * together: a lane's slot past the last one (only the last of the
             * J can be) reads slot 0, and the pairing gives it a zero twiddle.
             * Receptor entries: the part's base (uniform, in scalar registers)
             * plus one 32-bit byte offset of the row and the lane's slot (the
             * host keeps a q's rows below 4 GiB and their count below 2^24),
             * the slot step LP j as the load's immediate offset */
            const unsigned roff = __umul24((unsigned)rec.x, rstride) + soff;
            const unsigned twr = __umul24((unsigned)rec.y >> 3, twstride);
#pragma unroll
            for (int j = 0; j < J; j++) {
                const E w = *reinterpret_cast<const E *>(reinterpret_cast<const char *>(tw2) +
                                                         (twr + emo[j]));
                wr[j] = w.re;
                wi[j] = w.im;
#pragma unroll
                for (int X = 0; X < 3; X++) {
                    const char *base = RqB + (size_t)X * ns * sizeof(E);
                    rr[X][j] = j < J - 1 ? *reinterpret_cast<const E *>(base + (size_t)roff +
                                                                        (size_t)(LP * j * sizeof(E)))
                                         : *reinterpret_cast<const E *>(base + (size_t)(roff + dlast));
                }
            }
            /* every load of the pose is issued before the first use */
            __builtin_amdgcn_sched_barrier(0);
            const E *sUp = reinterpret_cast<const E *>(reinterpret_cast<const char *>(sU) +
                                                       __umul24((unsigned)prow, ustride));
            /* Re of each product, accumulated term by term (one fused
             * multiply-add per term), the products of the imaginary parts
             * apart (FP32 tables): their sign is the pose's.  With two poses per
             * wavefront the even and the odd j are summed apart: those of lanes
             * i and i + 32 of the form with one pose, so that a pose's sums
             * have the same bits in both. */
            F sa[PW][6], sb[PW][6];
#pragma unroll
            for (int h = 0; h < PW; h++)
#pragma unroll
                for (int k = 0; k < 6; k++) sa[h][k] = sb[h][k] = 0;
#pragma unroll
            for (int j = 0; j < J; j++) {
                const bool ok = j < J - 1 || sl + LP * j < ns;
                const int ec = ok ? sl + LP * j : 0;
                const E rv = rr[0][j], rd = rr[1][j], rw = rr[2][j];
                const E uv = sUp[ec], ud = sUp[us + ec], uw = sUp[2 * us + ec];
                const F w_r = wr[j], w_i = wi[j];   /* zero past the last slot */
                /* twiddled receptor factor: w * R^X */
                const F vr = w_r * rv.re - w_i * rv.im, vi = w_r * rv.im + w_i * rv.re;
                const F dr = w_r * rd.re - w_i * rd.im, di = w_r * rd.im + w_i * rd.re;
                const F xr = w_r * rw.re - w_i * rw.im, xi = w_r * rw.im + w_i * rw.re;
                F *va = sa[j % PW], *vc = sizeof(E) == 8 ? sb[j % PW] : va;
                const F sg = sizeof(E) == 8 ? (F)1 : (F)-1;
                va[0] += vr * uv.re; vc[0] += sg * (vi * uv.im);
                va[1] += vr * ud.re; vc[1] += sg * (vi * ud.im);
                va[1] += dr * uv.re; vc[1] += sg * (di * uv.im);
                va[2] += vr * uw.re; vc[2] += sg * (vi * uw.im);
                va[2] += xr * uv.re; vc[2] += sg * (xi * uv.im);
                va[3] += dr * ud.re; vc[3] += sg * (di * ud.im);
                va[4] += dr * uw.re; vc[4] += sg * (di * uw.im);
                va[4] += xr * ud.re; vc[4] += sg * (xi * ud.im);
                va[5] += xr * uw.re; vc[5] += sg * (xi * uw.im);
            }
            if (sizeof(E) == 8) {
                const F sg = A.mirror && ((unsigned)rec.y >> 3 & 1) ? (F)1 : (F)-1;
#pragma unroll
                for (int h = 0; h < PW; h++)
#pragma unroll
                    for (int k = 0; k < 6; k++) sa[h][k] += sg * sb[h][k];
            }
            /* the cross-lane sums run in the contraction's type */
            F v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < 6; k++) v[k] = PW == 2 && J > 1 ? sa[0][k] + sa[PW - 1][k] : sa[0][k];
            if (PW == 1) {
                /* transpose-reduce over the 64 lanes: after the three halving
                 * steps lane bits 5,4,3 select the slot, then a sum over the 8
                 * lanes of bits 2,1,0; lanes 0, 8, .., 40 hold slots 0..5 */
#pragma unroll
                for (int i = 0; i < 4; i++) v[i] = tr_swap32(v[i], v[i + 4]);
#pragma unroll
                for (int i = 0; i < 2; i++) v[i] = tr_swap16(v[i], v[i + 2]);
                const F send = b3 ? v[0] : v[1];
                const F keep = b3 ? v[1] : v[0];
                v[0] = keep + dpp_mov<FSX_DPP_ROR8>(send);
                v[0] += dpp_mov<FSX_DPP_HMIRROR>(v[0]);
            } else {
                /* the same within each 32-lane half, on the six sums: bit 4
                 * pairs sums i and i + 3; bit 3 the first two of those, the
                 * third across itself; bit 2 the two results: the same pairs
                 * as above */
#pragma unroll
                for (int i = 0; i < 3; i++) v[i] = tr_swap16(v[i], v[i + 3]);
                {
                    const F send = b3 ? v[0] : v[1];
                    const F keep = b3 ? v[1] : v[0];
                    v[0] = keep + dpp_mov<FSX_DPP_ROR8>(send);
                    v[1] = v[2] + dpp_mov<FSX_DPP_ROR8>(v[2]);
                }
                const F send = b2 ? v[0] : v[1];
                const F keep = b2 ? v[1] : v[0];
                v[0] = keep + dpp_mov<FSX_DPP_HMIRROR>(send);
            }
            v[0] += dpp_mov<FSX_DPP_XOR1>(v[0]);
            v[0] += dpp_mov<FSX_DPP_XOR2>(v[0]);
            if (writer) sO[p * 6 + slot] = v[0];
        }
        /* the batch's sums to acc (pose-major [pose][q][6]), added to those of
         * the earlier m-chunks (one launch after another: the atomic add, which no
         * other block makes to the same value, spares the wait for the old one);
         * no barrier after the last batch: sO is written again only after the
         * next item's barrier */
        lds_barrier();
        for (int i = tid; i < nb * 6; i += FSX_CROSS_BLOCK) {
            const int ip = i / 6;
            double *d = A.acc + ((size_t)(p0 + pb + ip) * Q + qc) * 6 + (i - ip * 6);
            const double x = 2.0 * (double)sO[i];
            if (A.first) __builtin_nontemporal_store(x, d);
            else unsafeAtomicAdd(d, x);
        }
        pb += FSX_UBATCH;
        if (pb >= n) break;
        if (tid / FSX_UBATCH == pb / FSX_UBATCH) sP[tid % FSX_UBATCH] = mine;
        lds_barrier();
        }
        if (!more) return;
    }
}

/* wavefronts per SIMD the registers are held to */
template <typename E>
__host__ __device__ constexpr int cross_waves() { return sizeof(E) == 8 ? 4 : 3; }

template <int J, typename E, int PW>
__global__ void __launch_bounds__(FSX_CROSS_BLOCK, (cross_waves<E>()))
k_cross(const fsx_cross_job job)
{
    cross_body<J, E, PW>(job);
}

/* The launches of several complexes in one (the batched form): every block
 * takes its share of job 0's items, then of job 1's, and so on, so that no
 * launch drains between complexes.  The jobs of one launch share the template
 * parameters; a complex appears once per launch (its m-chunks are launched in
 * order, one launch per chunk index). */
template <int J, typename E, int PW>
__global__ void __launch_bounds__(FSX_CROSS_BLOCK, (cross_waves<E>()))
k_cross_jobs(const fsx_cross_job *jobs, int njobs)
{
    for (int k = 0; k < njobs; k++) {
        const fsx_cross_job jb = jobs[k];
        cross_body<J, E, PW>(jb);
        /* the next job lays out the LDS for its own chunk size */
        __syncthreads();
    }
}

#endif
