// The MatMul kernel of the 32 x 32 and 64 x 64 tiles (gfx950): F32, any size, layout and
// alignment. matmul_mid.hip holds the strict form and what bounds it, matmul_native.hip the
// native one.
#pragma once

#include "pcu_device.hpp"
#include "pcu_gemm_stage.hpp"
#include "pcu_kernels.hpp"

#include <type_traits>

#pragma clang fp contract(off)

namespace pcu {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kMidBK = 32; // k of a slab

// A stage of one operand: X rows of op(A) (or columns of op(B)) by 32 k, filled by NI direct
// loads of W words a lane: W = 4 where every row of the stored matrix is 16-byte aligned, else
// 1. KC: the operand is stored with k contiguous (op(A) untransposed, op(B) transposed). Lane
// (i, b) reads element (x, 4 s + b) at step s; the layouts let it take several steps in one
// LDS instruction (a direct load costs the wave about 19 cycles and an LDS read about 12 that
// the MFMA before them does not hide) with the words of each on distinct banks.
//  * KC, W = 4: an instruction moves 32 k of the 8 rows q, q + NI, ..., 260 words from one
//    instruction's to the next's; with X = 32 the two halves of a row trade places in every
//    second group of 8 rows. A two-word read serves two steps.
//  * KC, W = 1: an instruction moves 32 k of rows 2 q and 2 q + 1, 68 words apart, fetched in
//    an order that puts the lane's four k of 16 side by side: element (x, 16 h + 4 s + b) at
//    68 (x / 2) + 32 (x % 2) + 16 h + 4 b + s. One 16-byte read serves four steps.
//  * else: k rows of X words, rotated by a multiple of 16 words that depends on k % 4. One
//    two-word read serves two steps; with PAIR (two subtiles a wave, lane i owning columns
//    2 i and 2 i + 1) one two-pair read does.
template <bool KC, int X, bool PAIR, int W> struct MidStage {
    static_assert(X == 64 || (X == 32 && !PAIR), "stage extents");
    static constexpr int NI = X / (2 * W);
    static constexpr int kPitch = 64 * W + (KC ? 4 : 0); // words from one instruction's to the next's
    static constexpr int kWords = NI * kPitch;
    static __device__ __forceinline__ int turn(int k)
    {
        return PAIR ? 32 * (k & 1) : (X == 64 ? 16 * (k & 3) : 8 * (k & 2));
    }
    static __device__ __forceinline__ int swap(int x) { return X == 32 ? (x >> 3) & 1 : 0; }
    // Row (column) and k of the first word that lane l of instruction q moves.
    static __device__ __forceinline__ int x_of(int q, int l)
    {
        if (KC)
            return W == 4 ? q + NI * (l >> 3) : 2 * q + (l >> 5);
        return (W * l - turn(k_of(q, l))) & (X - 1);
    }
    static __device__ __forceinline__ int k_of(int q, int l)
    {
        if (KC)
            return W == 4 ? 4 * ((l & 7) ^ (4 * swap(x_of(q, l)))) : (l & 16) + 4 * (l & 3) + ((l >> 2) & 3);
        return W * (64 * q + l) / X;
    }
    // Word of element (x, b), b < 4, of half h of the slab, and the words from there to step s
    // of the half.
    static __device__ __forceinline__ int at(int x, int b, int h)
    {
        if (KC)
            return W == 4 ? kPitch * (x % NI) + 32 * (x / NI) + 16 * (h ^ swap(x)) + b
                          : 68 * (x >> 1) + 32 * (x & 1) + 16 * h + 4 * b;
        return X * (16 * h + b) + ((x + turn(b)) & (X - 1));
    }
    static constexpr int kStep = KC ? (W == 4 ? 4 : 1) : 4 * X;
};

// One workgroup computes a TM x TN tile with waves of 16 x 16 SN cells, k in slabs of 32.
// NATIVE (explicitly permitted native compound arithmetic): the matrix cores accumulate,
// v_mfma_f32_16x16x4_f32 folding the same four k in their own order and rounding (lane and
// register layouts are those of the four-block form); no fault is classified.
template <bool TA, bool TB, int TM, int TN, int SN, int W, bool CHECK, bool NATIVE = false>
__global__ __launch_bounds__(4 * TM * TN / (16 * SN), 4) void k_gemm_mid(
    const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ C, int M,
    int N, int K, const unsigned long long *__restrict__ row_exp,
    const unsigned long long *__restrict__ col_exp, int thr, int check_risk,
    unsigned long long *suspect, SumCheck sck, NodeGate gate)
{
    if (block_gate_closed(gate))
        return;
    constexpr int BK = kMidBK, NS = BK / 4;       // steps of 4 k a slab
    constexpr int NWN = TN / (16 * SN), NW = TM / 16 * NWN;
    constexpr bool PAIR = SN == 2 && !TB;
    using SA = MidStage<!TA, TM, false, W>;
    using SB = MidStage<TB, TN, PAIR, W>;
    // Column of the wave's that lane i owns in subtile t.
    auto col_of = [](int i, int t) { return PAIR ? 2 * i + t : 16 * t + i; };
    constexpr int kST = 4;                                // stages
    constexpr int LA = SA::NI / NW, LB = SB::NI / NW; // a wave's loads a slab
    static_assert(SA::NI % NW == 0 && SB::NI % NW == 0, "every wave loads alike");
    __shared__ __align__(16) float As[kST][SA::kWords];
    __shared__ __align__(16) float Bs[kST][SB::kWords];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = 16 * (wv / NWN), wn = 16 * SN * (wv % NWN);
    int tm, tn;
    tile_of(blockIdx.x, (M + TM - 1) / TM, (N + TN - 1) / TN, tm, tn);
    const int m0 = tm * TM, n0 = tn * TN;
    // RejectSubnormal with the partial-sum check: each form takes its own tiles, as in
    // k_strict_gemm_mfma.
    if (!NATIVE && sck.flag != nullptr &&
        tile_exp_sum_below<TM, TN>(row_exp, col_exp, m0, n0, M, N, sck.thr) != CHECK)
        return;
    SubLanes subl;
    const int cls = kClassSubnormal;
    __shared__ unsigned char fine_ss[CHECK ? kSumMaxSuperSlabs : 1];
    SumGate<BK> sgate{nullptr, false};
    bool chk = true; // the current slab's sums are checked (checking form)
    if constexpr (CHECK) {
        if (sck.tbl_a != nullptr) {
            tile_fine_superslabs<TM, TN>(sck, m0, n0, M, N, K, fine_ss);
            sgate.fine = fine_ss;
        }
    }

    // Rows and columns past the edges read the last one inside (their cells are not stored).
    const int lda = TA ? M : K, ldb = TB ? K : N;
    const int lim_a = M - m0 - 1, lim_b = N - n0 - 1;
    const int nfull = K / BK, rem = K % BK, ntot = nfull + (rem != 0);
    // Byte offset of the word that this lane moves in the wave's instruction j from the
    // operand's base for the slab; k is held below `klim`.
    auto off_a = [&](int j, int klim) {
        const int q = wv + NW * j;
        const int x = SA::x_of(q, lane), k = SA::k_of(q, lane);
        const int xm = TA ? lim_a - (W - 1) : lim_a, km = TA ? klim : klim - (W - 1);
        const uint32_t xi = x < xm ? x : xm, ki = k < km ? k : km;
        return 4u * (TA ? ki * (uint32_t)lda + xi : xi * (uint32_t)lda + ki);
    };
    auto off_b = [&](int j, int klim) {
        const int q = wv + NW * j;
        const int x = SB::x_of(q, lane), k = SB::k_of(q, lane);
        const int xm = TB ? lim_b : lim_b - (W - 1), km = TB ? klim - (W - 1) : klim;
        const uint32_t xi = x < xm ? x : xm, ki = k < km ? k : km;
        return 4u * (TB ? xi * (uint32_t)ldb + ki : ki * (uint32_t)ldb + xi);
    };
    uint32_t oa[LA], ob[LB];
#pragma unroll
    for (int j = 0; j < LA; j++)
        oa[j] = off_a(j, BK - 1);
#pragma unroll
    for (int j = 0; j < LB; j++)
        ob[j] = off_b(j, BK - 1);
    const float *ga = TA ? A + m0 : A + (size_t)m0 * K; // the next slab to load
    const float *gb = TB ? B + (size_t)n0 * K : B + n0;
    const size_t da = TA ? (size_t)BK * lda : BK, db = TB ? BK : (size_t)BK * ldb;
    const uint32_t lds_a = lds_address(&As[0][0]) + 4u * SA::kPitch * wv;
    const uint32_t lds_b = lds_address(&Bs[0][0]) + 4u * SB::kPitch * wv;
    // Part `part` of `parts` of the next slab's loads, into the stage `sta` (`stb`) bytes into
    // the operand's stages.
    auto load_part = [&](uint32_t sta, uint32_t stb, int part, int parts) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < LA + LB; j++) {
            if (j * parts / (LA + LB) != part)
                continue;
            if (j < LA)
                load_lds<W>(ga, oa[j], lds_a + sta + 4u * SA::kPitch * NW * j);
            else
                load_lds<W>(gb, ob[j - LA], lds_b + stb + 4u * SB::kPitch * NW * (j - LA));
        }
        if (part == parts - 1) {
            ga += da;
            gb += db;
        }
    };
    // The last, partial slab: words past K are read from its last k (its loads take the
    // offsets of tail_offsets) and then overwritten with +0 by the wave that loaded them
    // (zero_tail, after its loads have landed).
    auto tail_offsets = [&]() {
#pragma unroll
        for (int j = 0; j < LA; j++)
            oa[j] = off_a(j, rem - 1);
#pragma unroll
        for (int j = 0; j < LB; j++)
            ob[j] = off_b(j, rem - 1);
    };
    auto zero_tail = [&]() {
        float *as = As[nfull % kST], *bs = Bs[nfull % kST];
#pragma unroll
        for (int j = 0; j < LA; j++) {
            const int q = wv + NW * j;
            if (SA::k_of(q, lane) >= rem)
#pragma unroll
                for (int e = 0; e < W; e++)
                    as[SA::kPitch * q + W * lane + e] = 0.0f;
        }
#pragma unroll
        for (int j = 0; j < LB; j++) {
            const int q = wv + NW * j;
            if (SB::k_of(q, lane) >= rem)
#pragma unroll
                for (int e = 0; e < W; e++)
                    bs[SB::kPitch * q + W * lane + e] = 0.0f;
        }
    };

    typedef float v4f __attribute__((ext_vector_type(4)));
    float acc[SN][4];
    v4f sum[SN]; // NATIVE
#pragma unroll
    for (int t = 0; t < SN; t++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            acc[t][q] = 0.0f;
            sum[t][q] = 0.0f;
        }
    v16f zero;
#pragma unroll
    for (int r = 0; r < 16; r++)
        zero[r] = 0.0f;
    auto mma = [&](float a, float b) { return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, zero, 0, 0, 0); };
    // Fold one MFMA's products: each cell q adds its k0, k0 + 1, k0 + 2, k0 + 3 products in
    // turn; the four cells' chains interleave.
    auto fold = [&](float (&c)[4], const v16f &p, auto ck) __attribute__((always_inline)) {
        constexpr bool CK = decltype(ck)::value;
        if (SN == 2)
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int blk = 0; blk < 4; blk++) {
#pragma unroll
            for (int q = 0; q < 4; q++)
                c[q] = c[q] + p[4 * blk + q];
            if constexpr (CK) {
                if (chk)
                    check_subnormal4(subl, c[0], c[1], c[2], c[3], cls);
            }
        }
        asm volatile("" : "+v"(c[0]), "+v"(c[1]), "+v"(c[2]), "+v"(c[3]));
        if (SN == 2)
            __builtin_amdgcn_s_setprio(0);
    };
    auto off_grid = [&]() {
        bool o = false;
#pragma unroll
        for (int t = 0; t < SN; t++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                o |= sum_off_grid(acc[t][q]);
        return __builtin_amdgcn_ballot_w64(o) != 0;
    };

    // The lane's operand words in a stage; step s of a slab adds kStep s.
    const int i = lane & 15, b = lane >> 4;
    constexpr uint32_t kStA = 4u * SA::kWords, kStB = 4u * SB::kWords; // bytes of a stage
    for (int st = 0; st < kST - 1 && st < ntot; st++) {
        if (st == nfull)
            tail_offsets();
        load_part(kStA * st, kStB * st, 0, 1);
    }
    if (ntot > 2)
        wait_loads_but<LA + LB>(); // slab 2 may still be on its way
    else
        wait_lds_loads();
    if (rem != 0 && nfull < 2)
        zero_tail();
    __syncthreads();
    // Operands of four steps (half a slab), read while the four before them are computed.
    float xa[2][4], xb[2][SN][4];
    // Word offsets of the lane's operands in each half of the stage of the current slab, and
    // the stage's offsets.
    int ra[2], rb[2][SN], ca = 0, cb = 0, na = SA::kWords, nb = SB::kWords;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        ra[h] = SA::at(wm + i, b, h);
#pragma unroll
        for (int t = 0; t < SN; t++)
            rb[h][t] = SB::at(wn + col_of(i, t), b, h);
    }
    const float *const a0 = As[0], *const b0 = Bs[0];
    uint32_t sta = (kST - 1) * kStA, stb = (kST - 1) * kStB; // the stage to load into
    // Part `part` of two of the reads of half h of the slab whose stages begin at sa and sb,
    // into register set h.
    auto rd = [&](int sa, int sb, int h, int part) __attribute__((always_inline)) {
        const float *pa = a0 + (ra[h] + sa);
        if constexpr (!TA && W == 1) {
            if (part == 0) {
                const float4 v = *reinterpret_cast<const float4 *>(pa);
                xa[h][0] = v.x;
                xa[h][1] = v.y;
                xa[h][2] = v.z;
                xa[h][3] = v.w;
            }
        } else {
#pragma unroll
            for (int s = 2 * part; s < 2 * part + 2; s++)
                xa[h][s] = pa[SA::kStep * s];
        }
        if constexpr (PAIR) {
            const float *pb = b0 + (rb[h][0] + sb);
#pragma unroll
            for (int s = 2 * part; s < 2 * part + 2; s++) {
                const float2 v = *reinterpret_cast<const float2 *>(pb + SB::kStep * s);
                xb[h][0][s] = v.x;
                xb[h][SN - 1][s] = v.y;
            }
        } else {
#pragma unroll
            for (int t = 0; t < SN; t++) {
                const float *pb = b0 + (rb[h][t] + sb);
                if constexpr (TB && W == 1) {
                    if (part == (SN == 2 ? t : 0)) {
                        const float4 v = *reinterpret_cast<const float4 *>(pb);
                        xb[h][t][0] = v.x;
                        xb[h][t][1] = v.y;
                        xb[h][t][2] = v.z;
                        xb[h][t][3] = v.w;
                    }
                } else {
#pragma unroll
                    for (int s = 2 * part; s < 2 * part + 2; s++)
                        xb[h][t][s] = pb[SB::kStep * s];
                }
            }
        }
    };
    v16f p;
    if (nfull > 0) {
        rd(0, 0, 0, 0);
        rd(0, 0, 0, 1);
        if constexpr (!NATIVE)
            p = mma(xa[0][0], xb[0][0][0]);
    }
    // One full slab. Slab kt + 1 was published by the barrier before, so its first operands
    // are read and its first MFMA issued before the barrier that ends this slab (NEXT). The
    // loads of slab kt + 3 (LOADS) are spread over the steps, each behind an MFMA, and have
    // until the end of the next slab to land: with few waves a CU a slab is shorter than a
    // load takes. The forms with and without them are separate code: branches inside the
    // steps made the compiler move the products through accumulator registers (about 1.6x
    // slower).
    auto slab = [&](auto loads_c, auto next_c, int kt, auto ck) __attribute__((always_inline)) {
        constexpr bool kLoads = decltype(loads_c)::value, kNext = decltype(next_c)::value;
        if constexpr (decltype(ck)::value)
            chk = sgate.at(kt, off_grid);
        if constexpr (kLoads) {
            if (kt + 3 == nfull)
                tail_offsets();
        }
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int g = s >> 2, g1 = ((s + 1) >> 2) & 1, n = s & 3, n1 = (s + 1) & 3;
            const bool more = s + 1 < NS || kNext;
            v16f q;
            if constexpr (NATIVE) {
#pragma unroll
                for (int t = 0; t < SN; t++)
                    sum[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[g][n], xb[g][t][n], sum[t], 0, 0, 0);
            } else if constexpr (SN == 2)
                q = mma(xa[g][n], xb[g][SN - 1][n]);
            else if (more)
                q = mma(xa[g1][n1], xb[g1][0][n1]);
            __builtin_amdgcn_sched_barrier(0); // the reads and loads issue while it runs
            // The next half's operands: the other register set, unless this step's MFMAs
            // still read it (one subtile a wave runs one step ahead).
            if (n == 1 || n == 2) {
                if (s < 4)
                    rd(ca, cb, 1, n - 1);
                else if (kNext)
                    rd(na, nb, 0, n - 1);
            }
            if constexpr (kLoads)
                load_part(sta, stb, s, NS);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (NATIVE)
                continue;
            fold(acc[0], p, ck);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (SN == 2) {
                if (more)
                    p = mma(xa[g1][n1], xb[g1][0][n1]);
                __builtin_amdgcn_sched_barrier(0);
                fold(acc[SN - 1], q, ck);
                __builtin_amdgcn_sched_barrier(0);
            } else if (more) {
                p = q;
            }
        }
        if constexpr (kLoads) {
            wait_loads_but<LA + LB>();
            sta = sta == (kST - 1) * kStA ? 0 : sta + kStA;
            stb = stb == (kST - 1) * kStB ? 0 : stb + kStB;
        } else if constexpr (kNext) {
            wait_lds_loads();
        }
        if (kNext && kt + 2 == nfull && rem != 0)
            zero_tail();
        if constexpr (kNext) {
            ca = na;
            cb = nb;
            na = na == (kST - 1) * SA::kWords ? 0 : na + SA::kWords;
            nb = nb == (kST - 1) * SB::kWords ? 0 : nb + SB::kWords;
            __syncthreads();
        }
    };
    const std::integral_constant<bool, CHECK> ck;
    const std::true_type yes;
    const std::false_type no;
    int kt = 0;
    for (; kt + kST - 1 < ntot; kt++)
        slab(yes, yes, kt, ck);
    for (; kt + 1 < nfull; kt++)
        slab(no, yes, kt, ck);
    if (kt < nfull)
        slab(no, no, kt, ck);
    if (rem != 0) {
        if constexpr (CHECK)
            chk = sgate.at(nfull, off_grid);
        const float *at = As[nfull % kST], *bt = Bs[nfull % kST];
        const int steps = (rem + 3) / 4;
        for (int s = 0; s < steps; s++) {
            const float a = at[SA::at(wm + i, b, s >> 2) + SA::kStep * (s & 3)];
            if constexpr (NATIVE) {
#pragma unroll
                for (int t = 0; t < SN; t++)
                    sum[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        a, bt[SB::at(wn + col_of(i, t), b, s >> 2) + SB::kStep * (s & 3)], sum[t], 0, 0, 0);
                continue;
            }
            v16f r[SN];
#pragma unroll
            for (int t = 0; t < SN; t++)
                r[t] = mma(a, bt[SB::at(wn + col_of(i, t), b, s >> 2) + SB::kStep * (s & 3)]);
#pragma unroll
            for (int t = 0; t < SN; t++)
                fold(acc[t], r[t], ck);
        }
    }

    if constexpr (NATIVE) {
#pragma unroll
        for (int t = 0; t < SN; t++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                acc[t][q] = sum[t][q];
    }
    // Epilogue: cells (m0 + wm + 4 (lane / 16) + q, n0 + wn + col_of(lane % 16, t)).
    const bool sub = CHECK && ((subl.flush() >> lane) & 1);
    uint64_t key = kNoFault;
    const bool pairs = PAIR && (N & 1) == 0 && ((uintptr_t)C & 7u) == 0;
    int cexp[SN];
#pragma unroll
    for (int t = 0; t < SN; t++) {
        const int c = n0 + wn + col_of(i, t);
        cexp[t] = check_risk && c < N ? exp_of(col_exp[c]) : 0;
        if (sub && m0 + wm < M && c < N) // the wave's cells lie in one 32 x 32 block
            flag_sum_block(sck, m0 + wm, c);
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int row = m0 + wm + 4 * b + q;
        if (row >= M)
            continue;
        const int rexp = check_risk ? exp_of(row_exp[row]) : 0;
        const int c0 = n0 + wn + col_of(i, 0);
        if (pairs && c0 < N)
            *reinterpret_cast<float2 *>(&C[(size_t)row * N + c0]) = make_float2(acc[0][q], acc[SN - 1][q]);
#pragma unroll
        for (int t = 0; t < SN; t++) {
            const int c = n0 + wn + col_of(i, t);
            if (c >= N)
                continue;
            const float v = acc[t][q];
            const uint64_t cell = (uint64_t)row * N + c;
            if (!pairs)
                C[cell] = v;
            if (NATIVE)
                continue;
            bool bad = !finite_bits(v) || sub;
            if (check_risk)
                bad |= rexp + cexp[t] < thr;
            if (bad)
                key = cell < key ? cell : key;
        }
    }
    if constexpr (!NATIVE)
        block_record_min<NW>(key, suspect);
}


} // namespace pcu
