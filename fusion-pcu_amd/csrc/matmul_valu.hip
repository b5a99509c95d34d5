// The vector-unit MatMul kernel on 128 x 128 tiles: strict F64 (F32 with the vector-unit engine),
// and native F64 (fused multiply-adds).
#include "pcu_device.hpp"
#include "pcu_gemm_stage.hpp"
#include "pcu_kernels.hpp"

#include <limits.h>

#pragma clang fp contract(off)

namespace pcu {

static inline bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

// ------------------------------------------------------------------- main tile

constexpr int BM = 128, BN = 128; // output tile of the vector-unit kernel

// Tile shape of the vector-unit kernel: 128 x 128 outputs per 256-thread workgroup (8 x 8
// per thread); binary64 stages twice as deep a k-slab, halving its barriers.
template <typename T> struct ValuCfg {
    static constexpr int BM = 128, BN = 128, BK = sizeof(T) == 4 ? 8 : 16;
    static constexpr int kThreads = 256;
    static constexpr int LDA = BM + 4, LDB = BN + 4; // row pitch of the k-major LDS stages
    static constexpr int EA = BM * BK / kThreads, EB = BN * BK / kThreads;
    // Binary64 splits a thread's 8 elements of a B k-row into 16-byte runs 32 apart when A
    // is untransposed (1.3-2% faster at 4096^3 and 2048x4096x2048) and keeps one contiguous
    // run under a transposed A (splitting measured 2.5% slower there).
    template <bool TA> static constexpr bool kSplitRunsB = sizeof(T) == 8 && !TA;
};

// Direct global -> LDS load of 16 bytes a lane: lane l's run lands at lds + 16 l bytes (lds is
// the wave's base, uniform across the wave).
// Issued from inline assembly, so the compiler does not model it: as a builtin it counts as
// a second kind of LDS event, after which every LDS read waits for all reads before it
// (lgkmcnt(0)) instead of only the ones it needs. The caller waits for it (wait_lds_loads)
// before the barrier that publishes the stage.
__device__ __forceinline__ void load_lds16(const void *g, void *lds)
{
    const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)lds;
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(base), "v"(g)
                 : "memory", "m0");
}

// NATIVE (explicitly permitted native compound arithmetic): one fused multiply-add per
// (cell, k) and no fault screen.
// WHOLE: every slab of every tile is whole (see the MFMA kernel).
// CHECK: the RejectSubnormal form with the partial-sum check (sck), its own instantiation.
template <typename T, bool TA, bool TB, bool VA, bool VB, bool NATIVE = false, bool WHOLE = false,
          bool CHECK = false>
__global__ __launch_bounds__(256, 2) void k_strict_gemm(
    const T *__restrict__ A, const T *__restrict__ B, T *__restrict__ C, int M, int N, int K,
    const unsigned long long *__restrict__ row_exp, const unsigned long long *__restrict__ col_exp,
    int thr, int check_risk, int vec_c, unsigned long long *suspect, SumCheck sck, NodeGate gate)
{
    if (block_gate_closed(gate))
        return;
    using Cfg = ValuCfg<T>;
    constexpr int BK = Cfg::BK;
    // Reading each k row's operands one row ahead measured 2-8% faster with a transposed
    // operand or a partial tile, and 3-9% slower for whole untransposed binary64 tiles.
    constexpr bool kAhead = TA || TB || !WHOLE;
    // Binary64 whole tiles with op(B) untransposed move op(B), and op(A) when transposed, from
    // global memory straight into LDS (global_load_lds_dwordx4: each wave instruction fills
    // one 1 KiB k row of a stage, so the stages keep their padded k-major layout). Their two
    // stages are separate LDS objects indexed at compile time, so the compiler can tell a
    // direct load into one stage from the reads of the other.
    constexpr bool kDirect = sizeof(T) == 8 && WHOLE && !TB;
    __shared__ __align__(16) T As[2][BK][Cfg::LDA];
    __shared__ __align__(16) T Bs[2][BK][Cfg::LDB];
    __shared__ __align__(16) T A0[BK][Cfg::LDA], A1[BK][Cfg::LDA];
    __shared__ __align__(16) T B0[BK][Cfg::LDB], B1[BK][Cfg::LDB];

    const int tid = threadIdx.x;
    const int tx = tid % 16, ty = tid / 16;
    // The lane's 8 columns come in RUN adjacent columns per run: binary32 lanes own 2 runs
    // of 4 (64 columns apart), binary64 lanes 4 runs of 2 (32 apart), so that each 16-byte
    // LDS read of B covers 256 contiguous bytes over the 16 lanes of a row (no bank
    // conflicts) and each 16-byte store is coalesced the same way.
    constexpr int RUN = 16 / sizeof(T), RUNS = 8 / RUN, RUN_STRIDE = BN / RUNS;
    auto col_of = [&](int j) { return (j / RUN) * RUN_STRIDE + tx * RUN + (j % RUN); };

    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    int tile_m, tile_n;
    tile_of(blockIdx.x, tiles_m, tiles_n, tile_m, tile_n);
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    // RejectSubnormal with the partial-sum check (sck.flag set) launches both forms over the
    // whole grid: a tile that may meet a product below 2^sck.thr is computed by the CHECK form,
    // which checks every partial sum it forms, and every other tile by the plain form.
    if (!NATIVE && sck.flag != nullptr &&
        tile_exp_sum_below<BM, BN>(row_exp, col_exp, m0, n0, M, N, sck.thr) != CHECK)
        return;
    SubLanes subl; // lanes that met a nonzero subnormal partial sum
    const int cls = kClassSubnormal;
    auto run_form = [&](auto &&run) { run(std::integral_constant<bool, CHECK && !NATIVE>{}); };
    // The checking form checks the superslabs that need it (SumGate).
    __shared__ unsigned char fine_ss[kSumMaxSuperSlabs];
    SumGate<BK> sgate{nullptr, false};
    bool chk = true; // the current slab's sums are checked (checking form)
    if constexpr (CHECK && !NATIVE) {
        if (sck.tbl_a != nullptr) {
            tile_fine_superslabs<BM, BN>(sck, m0, n0, M, N, K, fine_ss);
            sgate.fine = fine_ss;
        }
    }

    T acc[8][8];
#pragma unroll
    for (int i = 0; i < 8; i++)
#pragma unroll
        for (int j = 0; j < 8; j++)
            acc[i][j] = (T)0;

    SlabStager<T, Cfg, TA, TB, VA, VB> stage;

    const int ktiles = (K + BK - 1) / BK;
    if (WHOLE)
        stage.begin_whole(A, B, M, N, K, m0, n0, tid);
    // One slab's products and sums from the stage (Ac, Bc).
    auto compute = [&](const T (*Ac)[Cfg::LDA], const T (*Bc)[Cfg::LDB], auto ck) __attribute__((always_inline)) {
        constexpr bool CK = decltype(ck)::value;
        if constexpr (kAhead) {
            // The slab is unrolled; row k + 1's operands are read from LDS into the other
            // register set before row k is computed, and sched_barrier keeps the reads
            // there. Binary64 forms products 4 at a time to stay within two waves' registers.
            constexpr int PB = sizeof(T) == 8 ? 4 : 8;
            T a[2][8], b[2][8];
            auto rd = [&](int k) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    a[k & 1][i] = Ac[k][ty * 4 + i];
                    a[k & 1][4 + i] = Ac[k][64 + ty * 4 + i];
                }
#pragma unroll
                for (int j = 0; j < 8; j++)
                    b[k & 1][j] = Bc[k][col_of(j)];
            };
            rd(0);
#pragma unroll
            for (int k = 0; k < BK; k++) {
                if (k + 1 < BK)
                    rd(k + 1);
                __builtin_amdgcn_sched_barrier(0);
                const T(&x)[8] = a[k & 1];
                const T(&y)[8] = b[k & 1];
                // Per row, the products first and then their sums: no add waits on the
                // multiply just before it.
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    if (NATIVE) {
#pragma unroll
                        for (int j = 0; j < 8; j++)
                            acc[i][j] = fma(x[i], y[j], acc[i][j]);
                    } else {
#pragma unroll
                        for (int h = 0; h < 8; h += PB) {
                            T p[PB];
#pragma unroll
                            for (int j = 0; j < PB; j++)
                                p[j] = x[i] * y[h + j];
#pragma unroll
                            for (int j = 0; j < PB; j++)
                                acc[i][h + j] = acc[i][h + j] + p[j];
                            if constexpr (CK) {
                                if (chk) {
#pragma unroll
                                    for (int j = 0; j < PB; j += 4)
                                        check_subnormal4(subl, acc[i][h + j], acc[i][h + j + 1],
                                                         acc[i][h + j + 2], acc[i][h + j + 3], cls);
                                }
                            }
                        }
                    }
                    // Emits nothing; ties the row's eight sums to this point of the stream.
                    asm volatile("" : "+v"(acc[i][0]), "+v"(acc[i][1]), "+v"(acc[i][2]),
                                 "+v"(acc[i][3]), "+v"(acc[i][4]), "+v"(acc[i][5]),
                                 "+v"(acc[i][6]), "+v"(acc[i][7]));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            // Binary64 unrolls four k rows (220 VGPRs): two measured up to 6% slower by box
            // and shape, a whole slab spills.
#pragma unroll(sizeof(T) == 4 ? BK : 4)
            for (int k = 0; k < BK; k++) {
                T a[8], b[8];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    a[i] = Ac[k][ty * 4 + i];
                    a[4 + i] = Ac[k][64 + ty * 4 + i];
                }
#pragma unroll
                for (int j = 0; j < 8; j++)
                    b[j] = Bc[k][col_of(j)];
                // Per row, the eight rounded products first and then the eight rounded sums:
                // no add waits on the multiply just before it (F64 measured 4% faster than
                // alternating multiply/add through one temporary).
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    if (NATIVE) {
#pragma unroll
                        for (int j = 0; j < 8; j++)
                            acc[i][j] = fma(a[i], b[j], acc[i][j]);
                    } else {
                        T p[8];
#pragma unroll
                        for (int j = 0; j < 8; j++)
                            p[j] = a[i] * b[j];
#pragma unroll
                        for (int j = 0; j < 8; j++)
                            acc[i][j] = acc[i][j] + p[j];
                        if constexpr (CK) {
                            if (chk) {
#pragma unroll
                                for (int j = 0; j < 8; j += 4)
                                    check_subnormal4(subl, acc[i][j], acc[i][j + 1],
                                                     acc[i][j + 2], acc[i][j + 3], cls);
                            }
                        }
                    }
                }
            }
        }
    };
    auto off_grid = [&]() {
        bool o = false;
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int j = 0; j < 8; j++)
                o |= sum_off_grid(acc[i][j]);
        return __builtin_amdgcn_ballot_w64(o) != 0;
    };
    // Slab kt; the checking form checks its sums when the gate opens it.
    auto gcompute = [&](const T (*Ac)[Cfg::LDA], const T (*Bc)[Cfg::LDB], int kt, auto ck)
                        __attribute__((always_inline)) {
        if constexpr (decltype(ck)::value)
            chk = sgate.at(kt, off_grid);
        compute(Ac, Bc, ck);
    };
    if constexpr (!kDirect) {
        if (ktiles > 0) {
            if (WHOLE)
                stage.fetch_whole();
            else
                stage.fetch(A, B, M, N, K, m0, n0, 0, tid);
            stage.stash(As[0], Bs[0], tid);
        }
        __syncthreads();
        auto run = [&](auto ck) {
            for (int kt = 0; kt < ktiles; kt++) {
                const int cur = kt & 1;
                if (kt + 1 < ktiles) {
                    if (WHOLE)
                        stage.fetch_whole();
                    else
                        stage.fetch(A, B, M, N, K, m0, n0, (kt + 1) * BK, tid);
                }
                gcompute(As[cur], Bs[cur], kt, ck);
                if (kt + 1 < ktiles)
                    stage.stash(As[cur ^ 1], Bs[cur ^ 1], tid);
                __syncthreads();
            }
        };
        run_form(run);
    } else {
        // Wave w moves k rows w, w + 4, w + 8 and w + 12 of each directly loaded operand; lane
        // l's 16 bytes are the row's columns 2 l and 2 l + 1.
        const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
        const T *gb = B + (size_t)wv * N + n0 + 2 * lane;
        const T *ga = TA ? A + (size_t)wv * M + m0 + 2 * lane : A;
        auto load = [&](T (*Ad)[Cfg::LDA], T (*Bd)[Cfg::LDB]) {
#pragma unroll
            for (int r = 0; r < 4; r++)
                load_lds16(gb + (size_t)4 * r * N, &Bd[wv + 4 * r][0]);
            gb += (size_t)BK * N;
            if constexpr (TA) {
#pragma unroll
                for (int r = 0; r < 4; r++)
                    load_lds16(ga + (size_t)4 * r * M, &Ad[wv + 4 * r][0]);
                ga += (size_t)BK * M;
            } else {
                stage.fetch_whole_a();
            }
        };
        auto stash = [&](T (*Ad)[Cfg::LDA]) {
            if constexpr (!TA)
                stage.stash_a(Ad, tid);
        };
        if (ktiles > 0) {
            load(A0, B0);
            stash(A0);
        }
        wait_lds_loads();
        __syncthreads();
        // Two slabs per trip: stage 0 holds even slabs, stage 1 odd ones.
        auto slab = [&](auto cur_c, int kt, auto ck) __attribute__((always_inline)) {
            constexpr int cur = decltype(cur_c)::value;
            T (*Ac)[Cfg::LDA] = cur ? A1 : A0;
            T (*Bc)[Cfg::LDB] = cur ? B1 : B0;
            T (*An)[Cfg::LDA] = cur ? A0 : A1;
            T (*Bn)[Cfg::LDB] = cur ? B0 : B1;
            if (kt + 1 < ktiles)
                load(An, Bn);
            gcompute(Ac, Bc, kt, ck);
            if (kt + 1 < ktiles)
                stash(An);
            wait_lds_loads();
            __syncthreads();
        };
        auto run = [&](auto ck) {
            for (int kt = 0; kt < ktiles; kt += 2) {
                slab(std::integral_constant<int, 0>{}, kt, ck);
                if (kt + 1 < ktiles)
                    slab(std::integral_constant<int, 1>{}, kt + 1, ck);
            }
        };
        run_form(run);
    }

    // Epilogue: publish the tile and find the first suspect cell of this lane.
    const bool sub = CHECK && ((subl.flush() >> (threadIdx.x & 63)) & 1);
    uint64_t key = kNoFault;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        int r = m0 + (i < 4 ? ty * 4 + i : 64 + ty * 4 + (i - 4));
        if (r >= M)
            continue;
        int rexp = check_risk ? exp_of(row_exp[r]) : 0;
#pragma unroll
        for (int h = 0; h < RUNS; h++) {
            int c0 = n0 + col_of(h * RUN);
            T *dst = C + (size_t)r * N + c0;
            if (vec_c && c0 + RUN <= N) {
                if (sizeof(T) == 4)
                    *reinterpret_cast<float4 *>(dst) =
                        make_float4(acc[i][h * 4], acc[i][h * 4 + 1], acc[i][h * 4 + 2], acc[i][h * 4 + 3]);
                else
                    *reinterpret_cast<double2 *>(dst) = make_double2(acc[i][h * 2], acc[i][h * 2 + 1]);
            } else {
#pragma unroll
                for (int j = 0; j < RUN; j++)
                    if (c0 + j < N)
                        dst[j] = acc[i][h * RUN + j];
            }
#pragma unroll
            for (int j = 0; j < RUN; j++) {
                int c = c0 + j;
                if (NATIVE || c >= N)
                    continue;
                bool bad = !finite_bits(acc[i][h * RUN + j]) || sub;
                if (check_risk)
                    bad |= rexp + exp_of(col_exp[c]) < thr;
                if (sub)
                    flag_sum_block(sck, r, c);
                if (bad) {
                    uint64_t cell = (uint64_t)r * N + c;
                    key = cell < key ? cell : key;
                }
            }
        }
    }
    if (!NATIVE)
        wave_record_fault(key, suspect);
}

template <typename T, bool TA, bool TB>
static void gemm_dispatch(hipStream_t s, dim3 grid, const T *A, const T *B, T *C, int M, int N,
                          int K, const unsigned long long *re, const unsigned long long *ce,
                          int thr, int risk, unsigned long long *suspect, SumCheck sck,
                          NodeGate gate)
{
    bool va = (TA ? (M % 4 == 0) : (K % 4 == 0)) && aligned16(A);
    bool vb = (TB ? (K % 4 == 0) : (N % 4 == 0)) && aligned16(B);
    int vc = (N % 4 == 0) && aligned16(C);
    using Cfg = ValuCfg<T>;
    if (va && vb && M % Cfg::BM == 0 && N % Cfg::BN == 0 && K % Cfg::BK == 0)
        { hipLaunchKernelGGL((k_strict_gemm<T, TA, TB, true, true, false, true>), grid, dim3(256), 0, s, A, B, C, M, N, K, re, ce, thr, risk, vc, suspect, sck, gate); if (sck.flag) hipLaunchKernelGGL((k_strict_gemm<T, TA, TB, true, true, false, true, true>), grid, dim3(256), 0, s, A, B, C, M, N, K, re, ce, thr, risk, vc, suspect, sck, gate); }
    else if (va && vb)
        { hipLaunchKernelGGL((k_strict_gemm<T, TA, TB, true, true, false, false>), grid, dim3(256), 0, s, A, B, C, M, N, K, re, ce, thr, risk, vc, suspect, sck, gate); if (sck.flag) hipLaunchKernelGGL((k_strict_gemm<T, TA, TB, true, true, false, false, true>), grid, dim3(256), 0, s, A, B, C, M, N, K, re, ce, thr, risk, vc, suspect, sck, gate); }
    else if (va)
        { hipLaunchKernelGGL((k_strict_gemm<T, TA, TB, true, false, false, false>), grid, dim3(256), 0, s, A, B, C, M, N, K, re, ce, thr, risk, vc, suspect, sck, gate); if (sck.flag) hipLaunchKernelGGL((k_strict_gemm<T, TA, TB, true, false, false, false, true>), grid, dim3(256), 0, s, A, B, C, M, N, K, re, ce, thr, risk, vc, suspect, sck, gate); }
    else if (vb)
        { hipLaunchKernelGGL((k_strict_gemm<T, TA, TB, false, true, false, false>), grid, dim3(256), 0, s, A, B, C, M, N, K, re, ce, thr, risk, vc, suspect, sck, gate); if (sck.flag) hipLaunchKernelGGL((k_strict_gemm<T, TA, TB, false, true, false, false, true>), grid, dim3(256), 0, s, A, B, C, M, N, K, re, ce, thr, risk, vc, suspect, sck, gate); }
    else
        { hipLaunchKernelGGL((k_strict_gemm<T, TA, TB, false, false, false, false>), grid, dim3(256), 0, s, A, B, C, M, N, K, re, ce, thr, risk, vc, suspect, sck, gate); if (sck.flag) hipLaunchKernelGGL((k_strict_gemm<T, TA, TB, false, false, false, false, true>), grid, dim3(256), 0, s, A, B, C, M, N, K, re, ce, thr, risk, vc, suspect, sck, gate); }
}

template <typename T>
static void gemm_layout(hipStream_t s, dim3 grid, bool ta, bool tb, const T *A, const T *B, T *C,
                        int M, int N, int K, const unsigned long long *re,
                        const unsigned long long *ce, int thr, int risk,
                        unsigned long long *suspect, SumCheck sck, NodeGate gate)
{
    if (!ta && !tb) gemm_dispatch<T, false, false>(s, grid, A, B, C, M, N, K, re, ce, thr, risk, suspect, sck, gate);
    else if (!ta && tb) gemm_dispatch<T, false, true>(s, grid, A, B, C, M, N, K, re, ce, thr, risk, suspect, sck, gate);
    else if (ta && !tb) gemm_dispatch<T, true, false>(s, grid, A, B, C, M, N, K, re, ce, thr, risk, suspect, sck, gate);
    else gemm_dispatch<T, true, true>(s, grid, A, B, C, M, N, K, re, ce, thr, risk, suspect, sck, gate);
}

hipError_t launch_gemm_valu(hipStream_t s, int dtype, int M, int N, int K, bool ta, bool tb,
                            const void *A, const void *B, void *C,
                            const unsigned long long *row_exp, const unsigned long long *col_exp,
                            int thr, int risk, unsigned long long *suspect, SumCheck sck,
                            NodeGate gate)
{
    const dim3 grid((unsigned)((((uint64_t)M + BM - 1) / BM) * (((uint64_t)N + BN - 1) / BN)));
    if (dtype == 0)
        gemm_layout<float>(s, grid, ta, tb, (const float *)A, (const float *)B, (float *)C, M, N, K, row_exp, col_exp, thr, risk, suspect, sck, gate);
    else
        gemm_layout<double>(s, grid, ta, tb, (const double *)A, (const double *)B, (double *)C, M, N, K, row_exp, col_exp, thr, risk, suspect, sck, gate);
    return hipGetLastError();
}

template <bool TA, bool TB>
static void native_f64_dispatch(hipStream_t s, dim3 grid, const double *A, const double *B,
                                double *C, int M, int N, int K, NodeGate gate)
{
    const bool va = (TA ? (M % 4 == 0) : (K % 4 == 0)) && aligned16(A);
    const bool vb = (TB ? (K % 4 == 0) : (N % 4 == 0)) && aligned16(B);
    const int vc = (N % 4 == 0) && aligned16(C);
    using Cfg = ValuCfg<double>;
    if (va && vb && M % Cfg::BM == 0 && N % Cfg::BN == 0 && K % Cfg::BK == 0)
        hipLaunchKernelGGL((k_strict_gemm<double, TA, TB, true, true, true, true>), grid, dim3(256), 0, s, A, B, C, M, N, K, nullptr, nullptr, 0, 0, vc, nullptr, SumCheck{}, gate);
    else if (va && vb)
        hipLaunchKernelGGL((k_strict_gemm<double, TA, TB, true, true, true>), grid, dim3(256), 0, s, A, B, C, M, N, K, nullptr, nullptr, 0, 0, vc, nullptr, SumCheck{}, gate);
    else if (va)
        hipLaunchKernelGGL((k_strict_gemm<double, TA, TB, true, false, true>), grid, dim3(256), 0, s, A, B, C, M, N, K, nullptr, nullptr, 0, 0, vc, nullptr, SumCheck{}, gate);
    else if (vb)
        hipLaunchKernelGGL((k_strict_gemm<double, TA, TB, false, true, true>), grid, dim3(256), 0, s, A, B, C, M, N, K, nullptr, nullptr, 0, 0, vc, nullptr, SumCheck{}, gate);
    else
        hipLaunchKernelGGL((k_strict_gemm<double, TA, TB, false, false, true>), grid, dim3(256), 0, s, A, B, C, M, N, K, nullptr, nullptr, 0, 0, vc, nullptr, SumCheck{}, gate);
}

hipError_t launch_native_matmul(hipStream_t s, int dtype, uint64_t rows, uint64_t inner,
                                uint64_t cols, bool ta, bool tb, const void *a, const void *b,
                                void *c, NodeGate gate)
{
    if (rows > (uint64_t)INT_MAX || cols > (uint64_t)INT_MAX || inner > (uint64_t)INT_MAX)
        return hipErrorInvalidValue;
    if (rows == 0 || cols == 0)
        return hipSuccess;
    const int M = (int)rows, N = (int)cols, K = (int)inner;
    if (dtype == 0)
        return launch_native_gemm_f32(s, M, N, K, ta, tb, (const float *)a, (const float *)b, (float *)c, gate);
    const dim3 grid((unsigned)(((rows + BM - 1) / BM) * ((cols + BN - 1) / BN)));
    const double *A = (const double *)a, *B = (const double *)b;
    double *C = (double *)c;
    if (mid_wanted_f64(rows, cols, inner, ta, tb, true))
        return launch_gemm_mid_f64(s, true, M, N, K, ta, tb, A, B, C, nullptr, nullptr, 0, 0, nullptr, gate);
    if (!ta && !tb) native_f64_dispatch<false, false>(s, grid, A, B, C, M, N, K, gate);
    else if (!ta && tb) native_f64_dispatch<false, true>(s, grid, A, B, C, M, N, K, gate);
    else if (ta && !tb) native_f64_dispatch<true, false>(s, grid, A, B, C, M, N, K, gate);
    else native_f64_dispatch<true, true>(s, grid, A, B, C, M, N, K, gate);
    return hipGetLastError();
}

} // namespace pcu
