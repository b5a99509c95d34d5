// Strict F32 MatMul main kernel for outputs that do not divide into full rounds of 128 x 128
// tiles, of any size and alignment, with the products formed by the matrix cores.
//
// The contract and the use of an MFMA as a multiplier array are those of matmul_mfma.hip.
// Here v_mfma_f32_16x16x1_4b_f32 multiplies, in block b, A lane 16 b + i by B lane 16 b + j, and
// lane L's register 4 b + q holds block b's product (i = 4 (L / 16) + q, j = L % 16). The four
// blocks carry k0 .. k0 + 3, so a lane folds, for each of its four cells q, registers q,
// 4 + q, 8 + q and 12 + q in k order.
//
// What bounds it: issue. No vector instruction issues while an F32 MFMA runs, and a wave
// alone on its SIMD issues one instruction in about 4.7 cycles: 110 cycles per MFMA and its 16
// adds with one wave a SIMD, 90 with two, 73 with two waves of two 16 x 16 subtiles each, 66
// with four of those (64 is the ceiling). So few cells take 32 x 32 tiles of four 16 x 16
// waves (more SIMDs busy), more take 64 x 64 tiles of eight 16 x 32 waves. Everything else a
// wave issues is kept off that path: operands go from memory straight into LDS, ragged edges
// included (rows and columns past an edge re-read the last one inside; only the last, partial
// slab of k is zeroed, in LDS), and LDS reads serve several steps each. Measured against the
// kernels it replaced (register staging with bound checks, four 32 x 32 waves; sixteen 16 x 16
// waves on whole tiles): 777 x 3000 x 555 TN 72 against 197 us, 64 x 4096 x 4096 69 against 154,
// 1000 x 2048 x 1024 78 against 129, 1000 x 2048 x 2048 133 against 163, 1024^3 44 against 48.
#include "pcu_gemm_mid.hpp"

namespace pcu {

static inline bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

template <bool TA, bool TB, int TM, int TN, int SN>
static void mid_launch(hipStream_t s, int M, int N, int K, const float *A, const float *B, float *C,
                       const unsigned long long *re, const unsigned long long *ce, int thr,
                       int risk, unsigned long long *suspect, SumCheck sck, NodeGate gate)
{
    const dim3 grid((unsigned)((((uint64_t)M + TM - 1) / TM) * (((uint64_t)N + TN - 1) / TN)));
    const dim3 block(4 * TM * TN / (16 * SN));
    const bool vec = (TA ? M : K) % 4 == 0 && (TB ? K : N) % 4 == 0 && aligned16(A) && aligned16(B);
    if (vec) {
        hipLaunchKernelGGL((k_gemm_mid<TA, TB, TM, TN, SN, 4, false>), grid, block, 0, s, A, B, C, M, N, K, re, ce, thr, risk, suspect, sck, gate);
        if (sck.flag)
            hipLaunchKernelGGL((k_gemm_mid<TA, TB, TM, TN, SN, 4, true>), grid, block, 0, s, A, B, C, M, N, K, re, ce, thr, risk, suspect, sck, gate);
    } else {
        hipLaunchKernelGGL((k_gemm_mid<TA, TB, TM, TN, SN, 1, false>), grid, block, 0, s, A, B, C, M, N, K, re, ce, thr, risk, suspect, sck, gate);
        if (sck.flag)
            hipLaunchKernelGGL((k_gemm_mid<TA, TB, TM, TN, SN, 1, true>), grid, block, 0, s, A, B, C, M, N, K, re, ce, thr, risk, suspect, sck, gate);
    }
}

template <bool TA, bool TB>
static void mid_layout(hipStream_t s, MidTile tile, int M, int N, int K, const float *A,
                       const float *B, float *C, const unsigned long long *re,
                       const unsigned long long *ce, int thr, int risk,
                       unsigned long long *suspect, SumCheck sck, NodeGate gate)
{
    if (tile == MidTile::k32)
        mid_launch<TA, TB, 32, 32, 1>(s, M, N, K, A, B, C, re, ce, thr, risk, suspect, sck, gate);
    else
        mid_launch<TA, TB, 64, 64, 2>(s, M, N, K, A, B, C, re, ce, thr, risk, suspect, sck, gate);
}

// Estimated microseconds of each tile, from measurements on MI355X: the tiles of the fullest
// CU times what one takes, per 1024 k and fixed, and a fixed part. A 128 x 128 tile: 118 + 2.5
// (whole tiles) or 131 + 4 (bound checks; 140 alone on its CU), and 8. A 64 x 64 tile: 32.5 + 2 and
// 2.5, alone 36 and 5.5. Up to three 32 x 32 tiles run at once, 16 / 22.5 / 29 together and 4.5;
// more, 9.3 + 0.7 each and 2.5. The fixed parts decide short sums: kernels on 32 x 32 / 64 x 64 /
// 128 x 128 tiles, 768 x 19 x 2270 10.5 / 8.8 / 17.2 us, 1000 x 8 x 1500 9.3 / 7.7 / 14.4, 2048 x 19
// x 2048 20.6 / 16.2 / 18.5, 4096 x 32 x 2048 29.4 / 26.0 / 20.1, 3000 x 64 x 3000 41.6 / 39.0 /
// 43.4. Over K = 8 to 4000 and 512^2 to 8192^2 cells the estimates pick the fastest tile or one
// within 4% of it: 1500^3 125 / 154 / 216, 2050^3 315 / 341 / 602 (289 128 x 128 tiles are two
// rounds for one), 2048 x 256 x 2048 48.8 / 45.2 / 43.6, 2040 x 1024 x 2040 153 / 143 / 158, 4000^3
// 2393 / 2110 / 2230, 8190 x 512 x 8190 1346 / 1171 / 1098.
static MidTile mid_choose(uint64_t M, uint64_t N, uint64_t K, bool whole, double &us)
{
    const auto per_cu = [&](uint64_t t) {
        const uint64_t tiles = ((M + t - 1) / t) * ((N + t - 1) / t);
        return (double)((tiles + kGfx950Cus - 1) / kGfx950Cus);
    };
    const double k = (double)K / 1024.0, c32 = per_cu(32), c64 = per_cu(64), c128 = per_cu(128);
    const double t32 = c32 <= 3 ? (9.5 + 6.5 * c32) * k + 4.5 : c32 * (9.3 * k + 0.7) + 2.5;
    const double t64 = c64 <= 1 ? 36 * k + 5.5 : c64 * (32.5 * k + 2) + 2.5;
    const double t128 = 8 + c128 * (whole ? 118 * k + 2.5 : (c128 <= 1 ? 140 : 131) * k + 4);
    us = t32 < t64 ? t32 : t64;
    if (t128 <= us) {
        us = t128;
        return MidTile::k128;
    }
    return t32 < t64 ? MidTile::k32 : MidTile::k64;
}

MidTile mid_tile_f32(uint64_t M, uint64_t N, uint64_t K, bool whole)
{
    double us;
    return mid_choose(M, N, K, whole, us);
}

double mid_time_f32(uint64_t M, uint64_t N, uint64_t K)
{
    double us;
    (void)mid_choose(M, N, K, M % 128 == 0 && N % 128 == 0 && K % 16 == 0, us);
    return us;
}

// A lane's byte offset from its operand's tile must fit 32 bits: 64 rows of the stored matrix
// and one slab. And a launch holds fewer than 2^32 threads: 32 x 32 tiles take 256 each (an
// output of 2^34 cells reaches that; 128 x 128 tiles take an eighth of the threads).
bool mid_fits_f32(uint64_t M, uint64_t N, uint64_t K, bool ta, bool tb)
{
    const uint64_t lda = ta ? M : K, ldb = tb ? K : N;
    return lda < (1u << 24) && ldb < (1u << 24) && ((M + 31) / 32) * ((N + 31) / 32) <= UINT32_MAX / 256;
}

hipError_t launch_gemm_mid_f32(hipStream_t s, MidTile tile, int M, int N, int K, bool ta, bool tb,
                               const float *A, const float *B, float *C,
                               const unsigned long long *row_exp, const unsigned long long *col_exp,
                               int thr, int risk, unsigned long long *suspect, SumCheck sck,
                               NodeGate gate)
{
    if (!ta && !tb)
        mid_layout<false, false>(s, tile, M, N, K, A, B, C, row_exp, col_exp, thr, risk, suspect, sck, gate);
    else if (!ta && tb)
        mid_layout<false, true>(s, tile, M, N, K, A, B, C, row_exp, col_exp, thr, risk, suspect, sck, gate);
    else if (ta && !tb)
        mid_layout<true, false>(s, tile, M, N, K, A, B, C, row_exp, col_exp, thr, risk, suspect, sck, gate);
    else
        mid_layout<true, true>(s, tile, M, N, K, A, B, C, row_exp, col_exp, thr, risk, suspect, sck, gate);
    return hipGetLastError();
}

} // namespace pcu
