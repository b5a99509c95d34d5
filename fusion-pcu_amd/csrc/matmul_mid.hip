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
#include "pcu_device.hpp"
#include "pcu_gemm_stage.hpp"
#include "pcu_kernels.hpp"

#include <type_traits>

#pragma clang fp contract(off)

namespace pcu {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kMidBK = 32; // k of a slab

// Direct global -> LDS load of W words a lane: lane l's words land at lds + 4 W l bytes. base
// and lds are uniform across the wave. Issued from inline assembly, so the compiler does not
// track it: the caller waits for it before the barrier that publishes the stage.
template <int W> __device__ __forceinline__ void load_lds(const float *base, uint32_t off, uint32_t lds)
{
    static_assert(W == 1 || W == 4, "words a lane");
    if constexpr (W == 4)
        asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base)
                     : "memory", "m0");
    else
        asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(off), "s"(base)
                     : "memory", "m0");
}
// Wait until at most N of this wave's loads are outstanding: they complete in the order they
// were issued.
template <int N> __device__ __forceinline__ void wait_loads_but()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void wait_lds_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

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
template <bool TA, bool TB, int TM, int TN, int SN, int W, bool CHECK>
__global__ __launch_bounds__(4 * TM * TN / (16 * SN), 4) void k_strict_gemm_mid(
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
    if (sck.flag != nullptr &&
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
    const uint32_t lds_a = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)&As[0][0] + 4u * SA::kPitch * wv;
    const uint32_t lds_b = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)&Bs[0][0] + 4u * SB::kPitch * wv;
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

    float acc[SN][4];
#pragma unroll
    for (int t = 0; t < SN; t++)
#pragma unroll
        for (int q = 0; q < 4; q++)
            acc[t][q] = 0.0f;
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
            if constexpr (SN == 2)
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
            v16f r[SN];
#pragma unroll
            for (int t = 0; t < SN; t++)
                r[t] = mma(a, bt[SB::at(wn + col_of(i, t), b, s >> 2) + SB::kStep * (s & 3)]);
#pragma unroll
            for (int t = 0; t < SN; t++)
                fold(acc[t], r[t], ck);
        }
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
            bool bad = !finite_bits(v) || sub;
            if (check_risk)
                bad |= rexp + cexp[t] < thr;
            if (bad)
                key = cell < key ? cell : key;
        }
    }
    block_record_min<NW>(key, suspect);
}

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
        hipLaunchKernelGGL((k_strict_gemm_mid<TA, TB, TM, TN, SN, 4, false>), grid, block, 0, s, A, B, C, M, N, K, re, ce, thr, risk, suspect, sck, gate);
        if (sck.flag)
            hipLaunchKernelGGL((k_strict_gemm_mid<TA, TB, TM, TN, SN, 4, true>), grid, block, 0, s, A, B, C, M, N, K, re, ce, thr, risk, suspect, sck, gate);
    } else {
        hipLaunchKernelGGL((k_strict_gemm_mid<TA, TB, TM, TN, SN, 1, false>), grid, block, 0, s, A, B, C, M, N, K, re, ce, thr, risk, suspect, sck, gate);
        if (sck.flag)
            hipLaunchKernelGGL((k_strict_gemm_mid<TA, TB, TM, TN, SN, 1, true>), grid, block, 0, s, A, B, C, M, N, K, re, ce, thr, risk, suspect, sck, gate);
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
// CU times what one takes, per 1024 k and fixed. A 128 x 128 tile: 118 (whole tiles) or 131
// (bound checks; 140 alone on its CU) + 4. A 64 x 64 tile: 32.5 + 2, alone 36 + 4. Up to three
// 32 x 32 tiles run at once, 16 / 22.5 / 29 + 3 together; more, 9.3 + 0.5 each. The estimates
// pick the faster tile or one within 2% of it over 1024^3, 1500^3, 2050^3, 3001^3, 4000^3,
// 1536 x 1024 x 1536, 1920 x 1024 x 1920, 100 x 2000 x 9000, 8190 x 512 x 8190 and the shapes
// above: no single bound on the number of tiles does (a 2050 x 2050 output takes 541 us on
// 289 128 x 128 tiles, two rounds for one, and 329 on 4225 of 32 x 32; 8190 x 8190 takes 1119
// and 1303).
static MidTile mid_choose(uint64_t M, uint64_t N, uint64_t K, bool whole, double &us)
{
    const auto per_cu = [&](uint64_t t) {
        const uint64_t tiles = ((M + t - 1) / t) * ((N + t - 1) / t);
        return (double)((tiles + kGfx950Cus - 1) / kGfx950Cus);
    };
    const double k = (double)K / 1024.0, c32 = per_cu(32), c64 = per_cu(64), c128 = per_cu(128);
    const double t32 = c32 <= 3 ? (9.5 + 6.5 * c32) * k + 3 : c32 * (9.3 * k + 0.5);
    const double t64 = c64 <= 1 ? 36 * k + 4 : c64 * (32.5 * k + 2);
    const double t128 = c128 * ((whole ? 118 : c128 <= 1 ? 140 : 131) * k + 4);
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
// and one slab.
bool mid_fits_f32(uint64_t M, uint64_t N, uint64_t K, bool ta, bool tb)
{
    const uint64_t lda = ta ? M : K, ldb = tb ? K : N;
    return lda < (1u << 24) && ldb < (1u << 24);
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
