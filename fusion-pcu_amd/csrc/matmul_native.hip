// Native F32 MatMul (explicitly permitted native compound arithmetic): the matrix cores
// accumulate, in their own order and rounding, and no fault is classified. 128 x 128 tiles for
// full rounds of whole ones, the 32 x 32 and 64 x 64 tiles of pcu_gemm_mid.hpp for the rest.
#include "pcu_gemm_mid.hpp"

namespace pcu {

static inline bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

// 128 x 128 tiles: v_mfma_f32_32x32x2_f32 folds k and k + 1 of a 32 x 32 subtile per instruction.
template <class Cfg, bool TA, bool TB, bool VA, bool VB, bool WHOLE = false>
__global__ __launch_bounds__(Cfg::kThreads, Cfg::kWavesPerSimd) void k_native_gemm_mfma(
    const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ C, int M,
    int N, int K, NodeGate gate)
{
    if (block_gate_closed(gate))
        return;
    typedef float v16f __attribute__((ext_vector_type(16)));
    constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK, SM = Cfg::SM, SN = Cfg::SN;
    constexpr int S = SM * SN;
    // Whole tiles load op(A), and op(B) when untransposed, straight into LDS, in the strict
    // kernel's layouts (k-major rows with odd rows rotated by 32 floats; op(A) untransposed
    // in k quads), unpadded; a transposed op(B) goes through registers.
    constexpr bool kDirectA = WHOLE, kDirectB = WHOLE && !TB;
    constexpr int LDA = kDirectA ? BM : Cfg::LDA, LDB = kDirectB ? BN : Cfg::LDB;
    __shared__ __align__(16) float As[2][BK][LDA];
    __shared__ __align__(16) float Bs[2][BK][LDB];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave / Cfg::WN) * SM * 32, wn = (wave % Cfg::WN) * SN * 32;
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    int tm, tn;
    tile_of(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;

    v16f acc[S];
#pragma unroll
    for (int t = 0; t < S; t++)
#pragma unroll
        for (int r = 0; r < 16; r++)
            acc[t][r] = 0.0f;

    SlabStager<float, Cfg, TA, TB, VA, VB> stage;
    const int ktiles = (K + BK - 1) / BK;
    if (WHOLE)
        stage.begin_whole(A, B, M, N, K, m0, n0, tid);
    const int half = lane >> 5, col = lane & 31;
    if constexpr (WHOLE) {
        // Wave w moves IPW 1 KiB runs of each directly loaded operand a slab: runs
        // q = IPW w .. IPW w + IPW - 1, run q landing at 256 q floats of the stage. In rows of
        // 128 floats run q is rows 2q (lanes 0-31) and 2q + 1 (lanes 32-63); in k quads it
        // is quad q / 2, rows 64 (q % 2) + lane.
        constexpr int W = Cfg::kThreads / 64, IPW = BM * BK / 256 / W;
        static_assert(BM == 128 && BN == 128 && IPW * W * 256 == BM * BK && IPW % 2 == 0,
                      "the runs below are laid out for 128 x 128 tiles");
        const int wv = __builtin_amdgcn_readfirstlane(wave);
        const int rot = half ? (col + 8) & 31 : col;
        const float *ga = nullptr, *gb = nullptr;
        uint32_t lo_a = 0, lo_b = 0;
        size_t da = 0, db = 0, ra = 0, rb = 0; // slab advance, and run r's base offset / r
        if constexpr (!TA) {
            // run q = IPW w + r: quad IPW w / 2 + r / 2, rows 64 (r % 2) + lane
            ga = A + (size_t)m0 * K + 4 * (IPW / 2 * wv);
            lo_a = (uint32_t)lane * (uint32_t)K * 4u;
            da = BK;
        } else {
            ga = A + (size_t)(2 * IPW * wv) * M + m0;
            lo_a = ((uint32_t)half * (uint32_t)M + 4u * rot) * 4u;
            da = (size_t)BK * M;
            ra = (size_t)2 * M;
        }
        if constexpr (kDirectB) {
            gb = B + (size_t)(2 * IPW * wv) * N + n0;
            lo_b = ((uint32_t)half * (uint32_t)N + 4u * rot) * 4u;
            db = (size_t)BK * N;
            rb = (size_t)2 * N;
        }
        auto run_a = [&](int r) {
            return TA ? ga + r * ra : ga + (size_t)(64 * (r & 1)) * K + 4 * (r >> 1);
        };
        auto load_slab = [&](auto st_c) {
            constexpr int st = decltype(st_c)::value;
#pragma unroll
            for (int r = 0; r < IPW; r++)
                load_lds<4>(run_a(r), lo_a, lds_address(&As[st][0][0] + 256 * (IPW * wv + r)));
            ga += da;
            if constexpr (kDirectB) {
#pragma unroll
                for (int r = 0; r < IPW; r++)
                    load_lds<4>(gb + r * rb, lo_b, lds_address(&Bs[st][0][0] + 256 * (IPW * wv + r)));
                gb += db;
            } else {
                stage.fetch_whole_b();
            }
        };
        auto stash_slab = [&](auto st_c) {
            if constexpr (!kDirectB)
                stage.stash_b(Bs[decltype(st_c)::value], tid);
        };
        // Operand offsets of k pair kk (k = kk + half) from the stage base.
        auto a_at = [&](int kk, int i) {
            const int m = wm + 32 * i + col;
            return TA ? 128 * kk + (half ? 128 + ((m - 32) & 127) : m)
                      : 512 * (kk >> 2) + (kk & 3) + 4 * m + half;
        };
        auto b_at = [&](int kk, int j) {
            const int n = wn + 32 * j + col;
            return kDirectB ? 128 * kk + (half ? 128 + ((n - 32) & 127) : n) : (kk + half) * LDB + n;
        };
        if (ktiles > 0) {
            load_slab(std::integral_constant<int, 0>{});
            stash_slab(std::integral_constant<int, 0>{});
        }
        wait_lds_loads();
        __syncthreads();
        // Two slabs a trip, so each stage index is fixed at compile time.
        auto slab = [&](auto cur_c, int kt) __attribute__((always_inline)) {
            constexpr int cur = decltype(cur_c)::value;
            const std::integral_constant<int, cur ^ 1> nxt_c;
            if (kt + 1 < ktiles)
                load_slab(nxt_c);
            const float *as = &As[cur][0][0], *bs = &Bs[cur][0][0];
#pragma unroll
            for (int kk = 0; kk < BK; kk += 2) {
                float a[SM], b[SN];
#pragma unroll
                for (int i = 0; i < SM; i++)
                    a[i] = as[a_at(kk, i)];
#pragma unroll
                for (int j = 0; j < SN; j++)
                    b[j] = bs[b_at(kk, j)];
#pragma unroll
                for (int t = 0; t < S; t++)
                    acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t / SN], b[t % SN], acc[t], 0, 0, 0);
            }
            if (kt + 1 < ktiles)
                stash_slab(nxt_c);
            wait_lds_loads();
            __syncthreads();
        };
        for (int kt = 0; kt < ktiles; kt += 2) {
            slab(std::integral_constant<int, 0>{}, kt);
            if (kt + 1 < ktiles)
                slab(std::integral_constant<int, 1>{}, kt + 1);
        }
    } else {
        if (ktiles > 0) {
            stage.fetch(A, B, M, N, K, m0, n0, 0, tid);
            stage.stash(As[0], Bs[0], tid);
        }
        __syncthreads();
        for (int kt = 0; kt < ktiles; kt++) {
            const int cur = kt & 1;
            if (kt + 1 < ktiles)
                stage.fetch(A, B, M, N, K, m0, n0, (kt + 1) * BK, tid);
#pragma unroll
            for (int kk = 0; kk < BK; kk += 2) {
                float a[SM], b[SN];
#pragma unroll
                for (int i = 0; i < SM; i++)
                    a[i] = As[cur][kk + half][wm + 32 * i + col];
#pragma unroll
                for (int j = 0; j < SN; j++)
                    b[j] = Bs[cur][kk + half][wn + 32 * j + col];
#pragma unroll
                for (int t = 0; t < S; t++)
                    acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t / SN], b[t % SN], acc[t], 0, 0, 0);
            }
            if (kt + 1 < ktiles)
                stage.stash(As[cur ^ 1], Bs[cur ^ 1], tid);
            __syncthreads();
        }
    }
#pragma unroll
    for (int t = 0; t < S; t++) {
        const int c = n0 + wn + 32 * (t % SN) + col;
        if (c >= N)
            continue;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int row = m0 + wm + 32 * (t / SN) + 8 * (r >> 2) + 4 * half + (r & 3);
            if (row < M)
                C[(size_t)row * N + c] = acc[t][r];
        }
    }
}

// Whether an operand's tiles load directly as whole ones: every row 16-byte aligned, and a lane's
// byte offset from its run's base within 32 bits.
static bool native_direct(const float *A, const float *B, uint64_t M, uint64_t N, uint64_t K, bool ta, bool tb)
{
    const uint64_t span_a = ta ? M + 128 : 64 * K, span_b = N + 128;
    return (ta ? M : K) % 4 == 0 && (tb ? K : N) % 4 == 0 && aligned16(A) && aligned16(B) &&
           4 * span_a <= UINT32_MAX && (tb || 4 * span_b <= UINT32_MAX);
}

template <class Cfg, bool TA, bool TB>
static void native_dispatch(hipStream_t s, const float *A, const float *B, float *C, int M, int N,
                            int K, NodeGate gate)
{
    const dim3 grid((unsigned)(((M + Cfg::BM - 1) / Cfg::BM) * ((N + Cfg::BN - 1) / Cfg::BN)));
    const dim3 block(Cfg::kThreads);
    const bool va = (TA ? (M % 4 == 0) : (K % 4 == 0)) && aligned16(A);
    const bool vb = (TB ? (K % 4 == 0) : (N % 4 == 0)) && aligned16(B);
    const bool whole = M % Cfg::BM == 0 && N % Cfg::BN == 0 && K % Cfg::BK == 0 && native_direct(A, B, M, N, K, TA, TB);
    if (whole)
        hipLaunchKernelGGL((k_native_gemm_mfma<Cfg, TA, TB, true, true, true>), grid, block, 0, s, A, B, C, M, N, K, gate);
    else if (va && vb)
        hipLaunchKernelGGL((k_native_gemm_mfma<Cfg, TA, TB, true, true>), grid, block, 0, s, A, B, C, M, N, K, gate);
    else if (va)
        hipLaunchKernelGGL((k_native_gemm_mfma<Cfg, TA, TB, true, false>), grid, block, 0, s, A, B, C, M, N, K, gate);
    else if (vb)
        hipLaunchKernelGGL((k_native_gemm_mfma<Cfg, TA, TB, false, true>), grid, block, 0, s, A, B, C, M, N, K, gate);
    else
        hipLaunchKernelGGL((k_native_gemm_mfma<Cfg, TA, TB, false, false>), grid, block, 0, s, A, B, C, M, N, K, gate);
}

// 4 waves of 64 x 64 over a 128 x 128 tile: four independent accumulators per wave keep
// the matrix core busy between dependent MFMAs.
using NativeCfg = MfmaCfg<2, 2, 2, 2, 32, 2>;

template <bool TA, bool TB, int TM, int TN, int SN>
static void native_mid_launch(hipStream_t s, int M, int N, int K, const float *A, const float *B,
                              float *C, NodeGate gate)
{
    const dim3 grid((unsigned)((((uint64_t)M + TM - 1) / TM) * (((uint64_t)N + TN - 1) / TN)));
    const dim3 block(4 * TM * TN / (16 * SN));
    const bool vec = (TA ? M : K) % 4 == 0 && (TB ? K : N) % 4 == 0 && aligned16(A) && aligned16(B);
    if (vec)
        hipLaunchKernelGGL((k_gemm_mid<TA, TB, TM, TN, SN, 4, false, true>), grid, block, 0, s, A, B, C, M, N, K, nullptr, nullptr, 0, 0, nullptr, SumCheck{}, gate);
    else
        hipLaunchKernelGGL((k_gemm_mid<TA, TB, TM, TN, SN, 1, false, true>), grid, block, 0, s, A, B, C, M, N, K, nullptr, nullptr, 0, 0, nullptr, SumCheck{}, gate);
}

template <bool TA, bool TB>
static void native_mid_layout(hipStream_t s, MidTile tile, int M, int N, int K, const float *A,
                              const float *B, float *C, NodeGate gate)
{
    if (tile == MidTile::k32)
        native_mid_launch<TA, TB, 32, 32, 1>(s, M, N, K, A, B, C, gate);
    else
        native_mid_launch<TA, TB, 64, 64, 2>(s, M, N, K, A, B, C, gate);
}

static hipError_t launch_native_mid(hipStream_t s, MidTile tile, int M, int N, int K, bool ta, bool tb,
                                    const float *A, const float *B, float *C, NodeGate gate)
{
    if (!ta && !tb)
        native_mid_layout<false, false>(s, tile, M, N, K, A, B, C, gate);
    else if (!ta && tb)
        native_mid_layout<false, true>(s, tile, M, N, K, A, B, C, gate);
    else if (ta && !tb)
        native_mid_layout<true, false>(s, tile, M, N, K, A, B, C, gate);
    else
        native_mid_layout<true, true>(s, tile, M, N, K, A, B, C, gate);
    return hipGetLastError();
}

// Estimated microseconds of each tile, from measurements on MI355X: the tiles of the fullest CU
// times what one takes, per 1024 k and fixed. A whole 128 x 128 tile 68 alone on its CU, 59
// beside others (a bound-checked one 85 and more: taken only where the smaller tiles cannot address
// the operands, 3001 x 2999 x 3003 took 1065 us on them and 446 on 64 x 64 tiles). A 64 x 64 tile 17 + 1, alone 20 + 2.5; a 32 x 32 tile
// 5.4 + 0.4, up to two 8.1 and 14 + 2.5 together. Against 128 x 128 tiles: 1024 x 2048 x 1024
// 44 against 137 us, 1024 x 2048 x 2048 76 / 139, 64 x 4096 x 1024 35 / 348, 777 x 3000 x 555
// 41 / 351; 4096^3 1038 / 957.
static MidTile native_tile(uint64_t M, uint64_t N, uint64_t K, bool whole)
{
    const auto per_cu = [&](uint64_t t) {
        const uint64_t tiles = ((M + t - 1) / t) * ((N + t - 1) / t);
        return (double)((tiles + kGfx950Cus - 1) / kGfx950Cus);
    };
    const double k = (double)K / 1024.0, c32 = per_cu(32), c64 = per_cu(64), c128 = per_cu(128);
    const double t32 = c32 <= 2 ? (2.2 + 5.9 * c32) * k + 2.5 : c32 * (5.4 * k + 0.4);
    const double t64 = c64 <= 1 ? 20 * k + 2.5 : c64 * (17 * k + 1);
    if (whole && c128 * ((c128 <= 1 ? 68 : 59) * k + 4) <= (t32 < t64 ? t32 : t64))
        return MidTile::k128;
    return t32 < t64 ? MidTile::k32 : MidTile::k64;
}

// The tile that a native MatMul of these operands takes.
static MidTile native_choice(const float *A, const float *B, uint64_t M, uint64_t N, uint64_t K, bool ta, bool tb)
{
    const bool whole = M % NativeCfg::BM == 0 && N % NativeCfg::BN == 0 && K % NativeCfg::BK == 0 &&
                       native_direct(A, B, M, N, K, ta, tb);
    return mid_fits_f32(M, N, K, ta, tb) ? native_tile(M, N, K, whole) : MidTile::k128;
}

// native_choice as a tile side, for tests of the choice.
extern "C" int pcu_internal_native_matmul_tile(const void *a, const void *b, uint64_t rows, uint64_t inner,
                                               uint64_t cols, int ta, int tb)
{
    const MidTile t = native_choice((const float *)a, (const float *)b, rows, cols, inner, ta != 0, tb != 0);
    return t == MidTile::k32 ? 32 : (t == MidTile::k64 ? 64 : 128);
}

hipError_t launch_native_gemm_f32(hipStream_t s, int M, int N, int K, bool ta, bool tb,
                                  const float *A, const float *B, float *C, NodeGate gate)
{
    const MidTile tile = native_choice(A, B, (uint64_t)M, (uint64_t)N, (uint64_t)K, ta, tb);
    if (tile != MidTile::k128)
        return launch_native_mid(s, tile, M, N, K, ta, tb, A, B, C, gate);
    if (!ta && !tb) native_dispatch<NativeCfg, false, false>(s, A, B, C, M, N, K, gate);
    else if (!ta && tb) native_dispatch<NativeCfg, false, true>(s, A, B, C, M, N, K, gate);
    else if (ta && !tb) native_dispatch<NativeCfg, true, false>(s, A, B, C, M, N, K, gate);
    else native_dispatch<NativeCfg, true, true>(s, A, B, C, M, N, K, gate);
    return hipGetLastError();
}

} // namespace pcu
