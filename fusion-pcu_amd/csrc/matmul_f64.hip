// F64 MatMul (strict, and native with fused multiply-adds) on 64 x 64 tiles, of any size and
// alignment, for grids that leave CUs idle with larger tiles.
//
// A workgroup of 256 threads, 4 x 4 cells a thread, walks k in slabs of 16. Operands go from
// memory straight into LDS at every size and alignment, four stages deep: rows and columns past
// an edge re-read the last one inside, and only the last, partial slab of k is zeroed, in LDS.
// What bounds it: with one workgroup a CU each SIMD has one wave, whose 32 multiplies and adds
// a k take about 145 cycles and whose LDS reads (64 bytes a lane and k) 128 cycles of the CU's
// LDS bandwidth, so an operand layout must not need more of them: an operand with k contiguous
// is kept that way in LDS, and a 16-byte read gives two k of one row.
#include "pcu_device.hpp"
#include "pcu_gemm_stage.hpp"
#include "pcu_kernels.hpp"

#include <type_traits>

#pragma clang fp contract(off)

namespace pcu {

constexpr int kF64BK = 16, kF64T = 64; // k of a slab, tile side

// A stage of one operand: 64 rows of op(A) (columns of op(B)) by 16 k, in words. W = 4 where
// every row of the stored matrix is 16-byte aligned, else 1. KC: k contiguous in memory.
//  * KC, W = 4: an instruction moves 16 k of the 8 rows q, q + 8, ..., 260 words from one
//    instruction's to the next's; KC, W = 1: 16 k of rows 2 q and 2 q + 1, 68 words apart.
//    Either way the rows that one read of the wave takes start on distinct banks.
//  * else: k rows of 64 elements.
template <bool KC, int W> struct F64Stage {
    static constexpr int NI = 2048 / (64 * W);
    static constexpr int kPitch = 64 * W + (KC ? 4 : 0);
    static constexpr int kWords = NI * kPitch;
    // Element of the first word that lane l of instruction q moves, and (W = 1) which half.
    static __device__ __forceinline__ int x_of(int q, int l)
    {
        if (KC)
            return W == 4 ? q + 8 * (l >> 3) : 2 * q + (l >> 5);
        return W == 4 ? 2 * (l & 31) : 32 * (q & 1) + (l >> 1);
    }
    static __device__ __forceinline__ int k_of(int q, int l)
    {
        if (KC)
            return W == 4 ? 2 * (l & 7) : (l & 31) >> 1;
        return W == 4 ? 2 * q + (l >> 5) : q >> 1;
    }
    // Element offset of element (x, 0) in the stage; k adds kStep each.
    static __device__ __forceinline__ int at(int x)
    {
        if (KC)
            return W == 4 ? kPitch / 2 * (x % 8) + 16 * (x / 8) : 34 * (x >> 1) + 16 * (x & 1);
        return x;
    }
    static constexpr int kStep = KC ? 1 : 64;
};

template <bool TA, bool TB, int W, bool NATIVE>
__global__ __launch_bounds__(256, 2) void k_gemm_f64_mid(
    const double *__restrict__ A, const double *__restrict__ B, double *__restrict__ C, int M,
    int N, int K, const unsigned long long *__restrict__ row_exp,
    const unsigned long long *__restrict__ col_exp, int thr, int check_risk,
    unsigned long long *suspect, NodeGate gate)
{
    if (block_gate_closed(gate))
        return;
    constexpr int BK = kF64BK, T = kF64T, ND = BK / 2, kST = 4; // ND: steps of two k a slab
    using SA = F64Stage<!TA, W>;
    using SB = F64Stage<TB, W>;
    constexpr int LA = SA::NI / 4, LB = SB::NI / 4; // a wave's loads a slab
    __shared__ __align__(16) double As[kST][SA::kWords / 2];
    __shared__ __align__(16) double Bs[kST][SB::kWords / 2];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tx = tid & 15, ty = tid >> 4;
    int tm, tn;
    tile_of(blockIdx.x, (M + T - 1) / T, (N + T - 1) / T, tm, tn);
    const int m0 = tm * T, n0 = tn * T;
    // The thread's rows 4 ty + r; its columns: two adjacent pairs 32 apart where op(B) is read
    // along its columns, else four columns 16 apart.
    auto col_of = [&](int j) { return TB ? tx + 16 * j : 32 * (j >> 1) + 2 * tx + (j & 1); };

    const int lda = TA ? M : K, ldb = TB ? K : N;
    const int lim_a = M - m0 - 1, lim_b = N - n0 - 1;
    const int nfull = K / BK, rem = K % BK, ntot = nfull + (rem != 0);
    constexpr int E = W == 4 ? 2 : 1; // elements a lane moves (or half of one)
    auto offset = [&](auto kc_c, int x, int k, int lim, int klim, uint32_t ld) {
        constexpr bool KC = decltype(kc_c)::value;
        const int xm = KC ? lim : lim - (E - 1), km = KC ? klim - (E - 1) : klim;
        const uint32_t xi = x < xm ? x : xm, ki = k < km ? k : km;
        return 8u * (KC ? xi * ld + ki : ki * ld + xi) + (W == 1 ? 4u * (lane & 1) : 0u);
    };
    uint32_t oa[LA], ob[LB];
    auto offsets = [&](int klim) {
#pragma unroll
        for (int j = 0; j < LA; j++)
            oa[j] = offset(std::integral_constant<bool, !TA>{}, SA::x_of(wv + 4 * j, lane),
                           SA::k_of(wv + 4 * j, lane), lim_a, klim, (uint32_t)lda);
#pragma unroll
        for (int j = 0; j < LB; j++)
            ob[j] = offset(std::integral_constant<bool, TB>{}, SB::x_of(wv + 4 * j, lane),
                           SB::k_of(wv + 4 * j, lane), lim_b, klim, (uint32_t)ldb);
    };
    offsets(BK - 1);
    const double *ga = TA ? A + m0 : A + (size_t)m0 * K; // the next slab to load
    const double *gb = TB ? B + (size_t)n0 * K : B + n0;
    const size_t da = TA ? (size_t)BK * lda : BK, db = TB ? BK : (size_t)BK * ldb;
    const uint32_t lds_a = lds_address(&As[0][0]) + 4u * SA::kPitch * wv;
    const uint32_t lds_b = lds_address(&Bs[0][0]) + 4u * SB::kPitch * wv;
    constexpr uint32_t kStA = 4u * SA::kWords, kStB = 4u * SB::kWords; // bytes of a stage
    auto load_part = [&](uint32_t sta, uint32_t stb, int part, int parts) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < LA + LB; j++) {
            if (j * parts / (LA + LB) != part)
                continue;
            if (j < LA)
                load_lds<W>(ga, oa[j], lds_a + sta + 4u * SA::kPitch * 4 * j);
            else
                load_lds<W>(gb, ob[j - LA], lds_b + stb + 4u * SB::kPitch * 4 * (j - LA));
        }
        if (part == parts - 1) {
            ga += da;
            gb += db;
        }
    };
    auto zero_tail = [&]() {
        double *as = As[nfull % kST], *bs = Bs[nfull % kST];
        if (W == 1 && (lane & 1) != 0)
            return; // the even lane of a pair clears the element
#pragma unroll
        for (int j = 0; j < LA; j++) {
            const int q = wv + 4 * j;
            if (SA::k_of(q, lane) >= rem)
#pragma unroll
                for (int e = 0; e < E; e++)
                    as[(SA::kPitch * q + W * lane) / 2 + e] = 0.0;
        }
#pragma unroll
        for (int j = 0; j < LB; j++) {
            const int q = wv + 4 * j;
            if (SB::k_of(q, lane) >= rem)
#pragma unroll
                for (int e = 0; e < E; e++)
                    bs[(SB::kPitch * q + W * lane) / 2 + e] = 0.0;
        }
    };
    for (int st = 0; st < kST - 1 && st < ntot; st++) {
        if (st == nfull)
            offsets(rem - 1);
        load_part(kStA * st, kStB * st, 0, 1);
    }
    if (ntot > 2)
        wait_loads_but<LA + LB>(); // slab 2 may still be on its way
    else
        wait_lds_loads();
    if (rem != 0 && nfull < 2)
        zero_tail();
    __syncthreads();

    double acc[4][4];
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
        for (int j = 0; j < 4; j++)
            acc[r][j] = 0.0;
    // Operands of two k, read one step ahead.
    double xa[2][4][2], xb[2][4][2];
    const double *const a0 = As[0], *const b0 = Bs[0];
    int fa[4], fb[4]; // offsets of the thread's rows and columns in a stage
#pragma unroll
    for (int r = 0; r < 4; r++) {
        fa[r] = SA::at(4 * ty + r);
        fb[r] = SB::at(col_of(r));
    }
    int ca = 0, cb = 0, na = SA::kWords / 2, nb = SB::kWords / 2; // the stages of this slab and the next
    auto rd_one = [&](auto kc_c, const double *x0, const int (&f)[4], int step, int d,
                      double (&x)[4][2]) __attribute__((always_inline)) {
        if constexpr (decltype(kc_c)::value) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const double2 v = *reinterpret_cast<const double2 *>(x0 + f[r] + 2 * step * d);
                x[r][0] = v.x;
                x[r][1] = v.y;
            }
        } else {
#pragma unroll
            for (int kk = 0; kk < 2; kk++)
#pragma unroll
                for (int r = 0; r < 4; r += 2) {
                    const double2 v = *reinterpret_cast<const double2 *>(x0 + f[r] + step * (2 * d + kk));
                    x[r][kk] = v.x;
                    x[r + 1][kk] = v.y;
                }
        }
    };
    auto rd = [&](int sa, int sb, int d, int g) __attribute__((always_inline)) {
        rd_one(std::integral_constant<bool, !TA>{}, a0 + sa, fa, SA::kStep, d, xa[g]);
        rd_one(std::integral_constant<bool, TB>{}, b0 + sb, fb, SB::kStep, d, xb[g]);
    };
    auto compute = [&](int g) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < 2; kk++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                if constexpr (NATIVE) {
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        acc[r][j] = fma(xa[g][r][kk], xb[g][j][kk], acc[r][j]);
                } else {
                    // The products first: no add waits on the multiply just before it.
                    double p[4];
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        p[j] = xa[g][r][kk] * xb[g][j][kk];
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        acc[r][j] = acc[r][j] + p[j];
                }
                // Emits nothing; ties the row's sums to this point of the stream.
                asm volatile("" : "+v"(acc[r][0]), "+v"(acc[r][1]), "+v"(acc[r][2]), "+v"(acc[r][3]));
            }
    };
    uint32_t sta = (kST - 1) * kStA, stb = (kST - 1) * kStB; // the stage to load into
    if (nfull > 0)
        rd(0, 0, 0, 0);
    // One full slab; the pipeline is that of matmul_mid.hip: slab kt + 1 was published by the
    // barrier before, and the loads of slab kt + 3 have until the end of the next slab to land.
    auto slab = [&](auto loads_c, auto next_c, int kt) __attribute__((always_inline)) {
        constexpr bool kLoads = decltype(loads_c)::value, kNext = decltype(next_c)::value;
        if constexpr (kLoads) {
            if (kt + 3 == nfull)
                offsets(rem - 1);
        }
#pragma unroll
        for (int d = 0; d < ND; d++) {
            if (d + 1 < ND)
                rd(ca, cb, d + 1, (d + 1) & 1);
            else if (kNext)
                rd(na, nb, 0, 0);
            if constexpr (kLoads)
                load_part(sta, stb, d, ND);
            __builtin_amdgcn_sched_barrier(0);
            compute(d & 1);
            asm volatile("" ::: "memory"); // the next step's reads stay below this one
            __builtin_amdgcn_sched_barrier(0);
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
            na = na == (kST - 1) * SA::kWords / 2 ? 0 : na + SA::kWords / 2;
            nb = nb == (kST - 1) * SB::kWords / 2 ? 0 : nb + SB::kWords / 2;
            __syncthreads();
        }
    };
    const std::true_type yes;
    const std::false_type no;
    int kt = 0;
    for (; kt + kST - 1 < ntot; kt++)
        slab(yes, yes, kt);
    for (; kt + 1 < nfull; kt++)
        slab(no, yes, kt);
    if (kt < nfull)
        slab(no, no, kt);
#pragma unroll 1
    for (int d = 0; 2 * d < rem; d++) {
        rd((nfull % kST) * (SA::kWords / 2), (nfull % kST) * (SB::kWords / 2), d, 0);
        compute(0);
    }

    uint64_t key = kNoFault;
    const bool pairs = !TB && (N & 1) == 0 && ((uintptr_t)C & 15u) == 0;
    int cexp[4];
#pragma unroll
    for (int j = 0; j < 4; j++)
        cexp[j] = check_risk && n0 + col_of(j) < N ? exp_of(col_exp[n0 + col_of(j)]) : 0;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int row = m0 + 4 * ty + r;
        if (row >= M)
            continue;
        const int rexp = check_risk ? exp_of(row_exp[row]) : 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int c = n0 + col_of(j);
            if (c >= N)
                continue;
            const uint64_t cell = (uint64_t)row * N + c;
            if (!pairs)
                C[cell] = acc[r][j];
            else if ((j & 1) == 0)
                *reinterpret_cast<double2 *>(&C[cell]) = make_double2(acc[r][j], acc[r][j | 1]);
            if constexpr (!NATIVE) {
                bool bad = !finite_bits(acc[r][j]);
                if (check_risk)
                    bad |= rexp + cexp[j] < thr;
                if (bad)
                    key = cell < key ? cell : key;
            }
        }
    }
    if constexpr (!NATIVE)
        wave_record_first(key, suspect);
}

static inline bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

template <bool TA, bool TB>
static void f64_mid_launch(hipStream_t s, bool native, int M, int N, int K, const double *A,
                           const double *B, double *C, const unsigned long long *re,
                           const unsigned long long *ce, int thr, int risk,
                           unsigned long long *suspect, NodeGate gate)
{
    const dim3 grid((unsigned)((((uint64_t)M + kF64T - 1) / kF64T) * (((uint64_t)N + kF64T - 1) / kF64T)));
    const bool vec = (TA ? M : K) % 2 == 0 && (TB ? K : N) % 2 == 0 && aligned16(A) && aligned16(B);
    if (native) {
        if (vec)
            hipLaunchKernelGGL((k_gemm_f64_mid<TA, TB, 4, true>), grid, dim3(256), 0, s, A, B, C, M, N, K, re, ce, thr, risk, suspect, gate);
        else
            hipLaunchKernelGGL((k_gemm_f64_mid<TA, TB, 1, true>), grid, dim3(256), 0, s, A, B, C, M, N, K, re, ce, thr, risk, suspect, gate);
    } else if (vec) {
        hipLaunchKernelGGL((k_gemm_f64_mid<TA, TB, 4, false>), grid, dim3(256), 0, s, A, B, C, M, N, K, re, ce, thr, risk, suspect, gate);
    } else {
        hipLaunchKernelGGL((k_gemm_f64_mid<TA, TB, 1, false>), grid, dim3(256), 0, s, A, B, C, M, N, K, re, ce, thr, risk, suspect, gate);
    }
}

// Whether these tiles are the faster ones, from measurements on MI355X: the tiles of the fullest
// CU times microseconds per 1024 k. Strict: a 64 x 64 tile 91 alone on its CU, two 156, more 74
// each; a 128 x 128 tile 345 alone, 272 beside others (1024 x 1024 x 2048 156 us against 205 on
// 128 x 64 tiles, which these replaced, 1920 x 1024 x 1920 302 / 310, 2048^3 589 / 690, 3000 x
// 1024 x 3000 666 / 815, 4096 x 1024 x 4096 1184 / 1110). Native: 60, 104 and 48.5 each against
// 205 and 170 (1000^3 68 against 188 us). A lane's byte offset from its operand's tile must fit
// 32 bits (64 rows and one slab).
bool mid_wanted_f64(uint64_t M, uint64_t N, uint64_t K, bool ta, bool tb, bool native)
{
    const auto per_cu = [&](uint64_t t) {
        const uint64_t tiles = ((M + t - 1) / t) * ((N + t - 1) / t);
        return (double)((tiles + kGfx950Cus - 1) / kGfx950Cus);
    };
    if ((ta ? M : K) >= (1u << 23) || (tb ? K : N) >= (1u << 23))
        return false;
    const double c64 = per_cu(64), c128 = per_cu(128);
    if (native)
        return (c64 <= 2 ? 16 + 44 * c64 : 48.5 * c64) < (c128 <= 1 ? 205 : 170 * c128);
    return (c64 <= 2 ? 26 + 65 * c64 : 74 * c64) < (c128 <= 1 ? 345 : 272 * c128);
}

hipError_t launch_gemm_mid_f64(hipStream_t s, bool native, int M, int N, int K, bool ta, bool tb,
                               const double *A, const double *B, double *C,
                               const unsigned long long *row_exp, const unsigned long long *col_exp,
                               int thr, int risk, unsigned long long *suspect, NodeGate gate)
{
    if (!ta && !tb)
        f64_mid_launch<false, false>(s, native, M, N, K, A, B, C, row_exp, col_exp, thr, risk, suspect, gate);
    else if (!ta && tb)
        f64_mid_launch<false, true>(s, native, M, N, K, A, B, C, row_exp, col_exp, thr, risk, suspect, gate);
    else if (ta && !tb)
        f64_mid_launch<true, false>(s, native, M, N, K, A, B, C, row_exp, col_exp, thr, risk, suspect, gate);
    else
        f64_mid_launch<true, true>(s, native, M, N, K, A, B, C, row_exp, col_exp, thr, risk, suspect, gate);
    return hipGetLastError();
}

} // namespace pcu
