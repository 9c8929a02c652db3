/*
 * fsx_rules.h -- rules by which a call's sizes choose among kernel forms,
 * shared by the HIP side and host C (so that they can be exercised on the CPU).
 */
#ifndef FSX_RULES_H
#define FSX_RULES_H

/* Poses a wavefront of the cross-term pairing takes at a time, for chunks of ns
 * pairing slots.  Two poses of 32 lanes share the lane sums' instructions and
 * leave fewer lanes without a slot; one pose of 64 lanes has half the loads and
 * registers per lane.  Cross terms with 41 q, z 30 to 49 A, one against two poses:
 *   FP32  140,000 poses: L = 6 (25 slots) 0.90 and 0.51 ms, 7 (32) 0.88 and 0.49,
 *         10 (61) 0.96 and 0.91, 12 (85) 1.97 and 1.52, 13 (98) 1.95 and 1.96;
 *         20,000: 6 0.18 and 0.11, 12 0.36 and 0.32, 13 0.40 and 0.43, 15 (128) 0.47
 *         and 0.50, 16 (two chunks of about 72) 0.79 and 0.74, 20 (112) 1.18 and 1.28;
 *   FP64  140,000: 6 1.41 and 0.78, 10 1.64 and 1.37, 12 2.86 and 2.20, 15 3.16 and
 *         2.95; 20,000: 6 0.29 and 0.18, 15 1.09 and 1.06, 20 (118) 3.89 and 3.87. */
static inline int fsx_cross_pw(int mixed, int ns)
{
    return ns <= (mixed ? 96 : 128) ? 2 : 1;
}

/* Most cross-term blocks per CU; rows3: gamma2 rows per unit that the LDS leaves with
 * three; ns, pw: slots of the largest chunk and poses per wavefront; nrows: receptor
 * rows of a q; per_bucket: poses per (z, beta2, gamma2).
 * FP32: five; more only take each other's cache lines (300,000 poses at L = 25 98,
 * 76, 66.2, 65.6 and 73.7 ms with 2 to 6 blocks; 210,000 at L = 15 5.63, 4.64, 4.40,
 * 4.46 and 4.64).
 * FP64: as many as fit, three or four, but the receptor rows in flight (four
 * wavefronts of pw rows per block) take up the XCD's 4 MB of L2 themselves: 4.7 MB
 * with three blocks at L = 15, two poses per wavefront.  Two blocks
 *  - where three leave four rows per unit (from 172 slots on): two leave six or
 *    eight.  Cross terms, against three blocks: L = 18 (181 slots) 1.41 times with
 *    0.01 poses per bucket, 1.20 with 0.1, 0.95 with 0.2, 0.88 with 0.4, 0.85 with 2,
 *    0.86 with 6, 0.90 with 15; L = 20 (221) 1.02 with 0.4, 0.99 with 2, 0.95 with 6,
 *    0.92 with 15; L = 28 (217) 1.03, 1.00, 0.98, 0.95;
 *  - where the receptor rows of a q are 6 MB or more and the buckets so full that the
 *    pairing outweighs the translation.  64 x 19 grid, 6, 9 and 15 poses per bucket: L
 *    = 14 1.03, 0.96 and 0.90 times, L = 15 1.03, 0.94, 0.89 (two poses per
 *    wavefront), L = 17 0.97, 0.97, 0.95, L = 25 0.98, 1.00, 0.95 (one); 128 x 37 grid,
 *    L = 25, 5.2 per bucket 0.93, 2.5 1.06.  Tables of 4 MB (L = 15, 36 x 19) 1.12, 1.05,
 *    0.98. */
static inline int fsx_cross_blocks(int mixed, int rows3, int ns, int pw, long nrows, double per_bucket)
{
    if (mixed) return 5;
    if (rows3 <= 4) return per_bucket >= (ns <= 200 ? 0.2 : 4) ? 2 : 5;
    return 48.0 * ns * (double)nrows >= 6e6 && per_bucket >= (pw == 2 ? 8 : 5) ? 2 : 5;
}

/* Lanes per fit of the mixed form's lane-group fit: up to 8 q per lane, at least four
 * lanes.  They set the order of the sums over q, so they depend on nothing else.
 * The longest fit, a chain of dependent evaluations, sets the time of all but the
 * longest lists.  Fit stage, averages over L = 8, 10, 12, 15, with half as many lanes
 * and with these: 31 q (4 lanes) 2,000 fits 0.17 and 0.12 ms, 210,000 0.54 and 0.47;
 * 51 q (8) 60,000 0.57 and 0.48, 150,000 0.80 and 0.76, but 210,000 of one box 0.57 and
 * 0.67; 81 q (16) 2,000 0.24 and 0.20, 20,000 0.47 and 0.38, 150,000 0.96 and 1.14. */
static inline int fsx_fit_lanes(int Q)
{
    int fpl = 4;
    while (fpl < 64 && fpl * 8 < Q) fpl *= 2;
    return fpl;
}

/* Whether the (z, beta2) groups' counts are summed by a launch of their own, between
 * the two passes of the bucketing, instead of by every wavefront of the second pass.
 * Bucketing stage without and with it: 341 groups 33 and 34 us, 684 45 and 45, 3,737
 * 93 and 76, 18,000 261 and 98, 50,000 1,241 and 124, 180,000 13,978 and 218. */
static inline int fsx_unit_scan(long groups)
{
    return groups > 700;
}

#endif
