// Strict F32/F64 MatMul of few cells: one launch does the whole MatMul, one cell a lane.
//
// Each 256-thread workgroup owns 16 x 16 cells (wave w rows 4 w .. 4 w + 3, lane row r of 16
// lanes one of them) and walks k in chunks of 1 KiB a row, staged in LDS with k contiguous. A
// block sees all of k for its rows and columns, so it folds their smallest exponents as it
// stages them and screens its own cells; the suspect cells (a non-finite result, or exponents that
// allow a tiny product) are searched, each by its own lane, until the block's earliest fault lies
// before the cells left, and that fault is folded into the node's word with atomicMin, so the word
// ends with the MatMul's first fault.
//
// What bounds it: the chain of sums. A wave's add that depends on the one two instructions
// before it issues 14 cycles after it with one or two waves a SIMD, so a cell cannot take less
// than about 14 cycles a k, whatever feeds it. op(A) is read from LDS once per 64 k (binary64:
// 32), each lane row of 16 holding its own row's k, and reaches the product as a broadcast
// within the lane row (row_newbcast) that costs no instruction for binary32; op(B) takes one
// 16-byte read per 4 k (2). The next chunk's loads are in flight while a chunk is computed.
// Short sums are bound by what a workgroup costs apart from them: loads, four barriers and the
// LDS it holds. Sums that fit a chunk have one stage (four workgroups a CU against the two
// stages' two), those of 256 bytes a row a stage of that size (six). Whole calls with one form
// of two stages for every K, and with these: binary32 512 x 8 x 512 20.3 -> 16.4 us, 512 x 64 x
// 512 21.1 -> 17.5, 512 x 256 x 512 23.2 -> 21.5, binary64 512 x 8 x 512 20.3 -> 17.0.
#include "pcu_device.hpp"
#include "pcu_gemm_search.hpp"
#include "pcu_kernels.hpp"

#include <limits.h>
#include <utility>

#pragma clang fp contract(off)

namespace pcu {

// Order keys of the screen: a smaller nonzero |v| has a smaller key, zero the largest, and a
// non-finite value one above every finite one. Two instructions an element (binary64: on the
// high word, with a nonzero low word of the tiniest subnormals standing as its last bit).
__device__ __forceinline__ uint32_t exp_key(float v) { return (bits_of(v) << 1) - 1u; }
__device__ __forceinline__ uint32_t exp_key(double v)
{
    const uint64_t b = bits_of(v);
    const uint32_t lo = (uint32_t)b;
    return ((((uint32_t)(b >> 32)) | (lo < 1u ? lo : 1u)) << 1) - 1u;
}
// floor(log2 |v|) of the key's value (binary64 subnormals: a lower bound), kExpNone for zero and
// non-finite.
template <typename T> __device__ __forceinline__ int key_exp(uint32_t key)
{
    const uint32_t b = (key + 1u) >> 1;
    if constexpr (sizeof(T) == 4) {
        return ilog2_abs(__uint_as_float(b));
    } else {
        const uint32_t e = b >> 20;
        return b == 0 || e == 0x7ff ? kExpNone : (e ? (int)e - 1023 : -1074);
    }
}

// f(0) .. f(N - 1), each with its number as a constant.
template <class F, int... J>
__device__ __forceinline__ void each_of(F &&f, std::integer_sequence<int, J...>)
{
    (f(std::integral_constant<int, J>{}), ...);
}
template <int N, class F> __device__ __forceinline__ void each(F &&f)
{
    each_of(f, std::make_integer_sequence<int, N>{});
}

// Stands for a zero operand in the search's stages where only tiny products are looked for: its
// product with any operand is far above the smallest normal.
template <typename T> constexpr T kZeroStand = sizeof(T) == 4 ? (T)0x1p100 : (T)0x1p1000;

// Waves a SIMD that the registers must leave room for: the LDS of the shortest form lets eight
// workgroups run on a CU, of the longer one-chunk form four, of the two-stage form two.
template <int L, bool ONE> constexpr int kSmallWaves = ONE ? (L == 1 ? 6 : 4) : 2;

// The first fault of one cell in the kc k of a staged chunk (as: its row, bs: its column, zeros or
// their stands up to the next 16 k), kNoFault when there is none or `on` is false. `step`: the
// first k's Multiply. ADDS: t carries the cell's sum from chunk to chunk, and every product and
// sum is checked; else only for a tiny product, with zeros staged as kZeroStand. 64 bytes of k at a
// time, whose smallest product (and sum, where subnormal ones are rejected) says whether they go
// through the exact classifiers: a compare for each k would have cost three times the products.
template <typename T, bool ADDS>
__device__ __forceinline__ uint64_t chunk_first_fault(const T *as, const T *bs, int kc, T &t, bool on,
                                                      uint64_t step, int policy)
{
    constexpr int P = 16 / (int)sizeof(T), U = 4 * P;
    const bool reject_sub = policy == kPolicyRejectSubnormal;
    for (int k = 0; k < kc; k += U) {
        uint4 qa[U / P], qb[U / P];
#pragma unroll
        for (int g = 0; g < U / P; g++) {
            qa[g] = *reinterpret_cast<const uint4 *>(as + k + P * g);
            qb[g] = *reinterpret_cast<const uint4 *>(bs + k + P * g);
        }
        const T *a = reinterpret_cast<const T *>(qa), *b = reinterpret_cast<const T *>(qb);
        T n = t, least = (T)1;
#pragma unroll
        for (int c = 0; c < U; c++) {
            const T p = a[c] * b[c];
            least = __builtin_elementwise_min(least, __builtin_elementwise_abs(p));
            if (ADDS) {
                n = n + p;
                if (reject_sub)
                    least = __builtin_elementwise_min(least, __builtin_elementwise_abs(n));
            }
        }
        // (A non-finite sum stays so, and a NaN is no minimum.)
        const bool look = (policy != kPolicyAllowGradual && at_most_min_normal(least)) || (ADDS && !finite_bits(n));
        if (on && look) {
#pragma unroll 1
            for (int c = 0; c < U; c++) {
                const T x = as[k + c], y = bs[k + c], p = x * y;
                uint32_t kind = classify_mul(x, y, p, policy);
                if (kind != kOk && (ADDS || kind == kUnderflow))
                    return pack_fault(step + 2 * (uint64_t)(k + c), kind);
                if (ADDS) {
                    kind = classify_add(t, p, t + p, policy);
                    if (kind != kOk)
                        return pack_fault(step + 2 * (uint64_t)(k + c) + 1, kind);
                    t = t + p;
                }
            }
        }
        t = n;
    }
    return kNoFault;
}

// VA, VB: every row of the stored matrix is 16-byte aligned. L: 16-byte runs of each operand that a
// thread stages at a time, 256 L bytes of k a row. ONE: all of K is one chunk, in one stage.
template <typename T, bool TA, bool TB, bool VA, bool VB, int L, bool ONE>
__global__ __launch_bounds__(256, (kSmallWaves<L, ONE>)) void k_strict_gemm_small(
    const T *__restrict__ A, const T *__restrict__ B, T *__restrict__ C, int M, int N, int K,
    int thr, int risk, int policy, unsigned long long *fault, NodeGate gate, ProgramClose close)
{
    if (block_gate_closed(gate)) {
        program_close_block(close);
        return;
    }
    constexpr int P = 16 / (int)sizeof(T);     // elements of 16 bytes
    constexpr int BK = 16 * P * L;             // k of a chunk
    constexpr int BKP = BK + P;                // row pitch: one 16-byte pad
    constexpr int kST = ONE ? 1 : 2;           // stages
    __shared__ __align__(16) T As[kST][16][BKP];
    __shared__ __align__(16) T Bs[kST][16][BKP];
    __shared__ uint32_t rkey[16], ckey[16];
    __shared__ unsigned long long best; // the earliest fault that this block knows of
    __shared__ int first_sus;           // its first suspect cell, and whether that is finite
    const int tid = threadIdx.x;
    const int ty = tid >> 4, tx = tid & 15; // the thread's cell
    const int tiles_n = (N + 15) / 16;
    const int m0 = (int)(blockIdx.x / tiles_n) * 16, n0 = (int)(blockIdx.x % tiles_n) * 16;
    if (tid < 16) {
        rkey[tid] = 0xffffffffu;
        ckey[tid] = 0xffffffffu;
    }
    if (tid == 0)
        first_sus = INT_MAX;
    // A thread stages runs of P k of one row of op(A) and one column of op(B), 16 P k apart, in
    // an order that keeps each global access coalesced: 16 threads along k where k is
    // contiguous, else 16 threads along the rows (columns).
    const int xa = TA ? tx : ty, ka = P * (TA ? ty : tx);
    const int xb = TB ? ty : tx, kb = P * (TB ? tx : ty);
    const int row = m0 + xa, col = n0 + xb;
    const T *pa = TA ? A + (row < M ? row : M - 1) : A + (size_t)(row < M ? row : M - 1) * K;
    const T *pb = TB ? B + (size_t)(col < N ? col : N - 1) * K : B + (col < N ? col : N - 1);
    T va[L][P], vb[L][P];
    // One operand's runs of the chunk at k0. FULL: the chunk lies inside K. Else what lies past K
    // is loaded from its end, so that every load of the chunk is in flight at once (a load
    // under a condition is waited for before the next), and is +0.
    auto fetch = [&](const T *p, size_t ld, auto kc_c, auto vec_c, auto full_c, int kt, int k0,
                     T (&v)[L][P]) __attribute__((always_inline)) {
        constexpr bool KC = decltype(kc_c)::value, VEC = KC && decltype(vec_c)::value;
        constexpr bool FULL = decltype(full_c)::value;
        uint4 q[L];
        const size_t first = KC ? 0 : (size_t)(k0 + kt) * ld, last = KC ? 0 : (size_t)(K - 1) * ld;
#pragma unroll
        for (int j = 0; j < L; j++) {
            const int k = k0 + kt + 16 * P * j;
            if constexpr (VEC) { // K is a multiple of P
                q[j] = *reinterpret_cast<const uint4 *>(p + (FULL || k < K ? k : K - P));
            } else {
#pragma unroll
                for (int c = 0; c < P; c++) {
                    const bool in = FULL || k + c < K;
                    v[j][c] = p[KC ? (size_t)(in ? k + c : K - 1) : (in ? first + (size_t)(16 * P * j + c) * ld : last)];
                }
            }
        }
#pragma unroll
        for (int j = 0; j < L; j++) {
            const int k = k0 + kt + 16 * P * j;
            const T *e = reinterpret_cast<const T *>(&q[j]);
#pragma unroll
            for (int c = 0; c < P; c++) {
                if constexpr (VEC)
                    v[j][c] = e[c];
                if (!FULL && k + c >= K)
                    v[j][c] = (T)0;
            }
        }
    };
    auto fetch_chunk = [&](auto full_c, int k0) __attribute__((always_inline)) {
        fetch(pa, (size_t)M, std::integral_constant<bool, !TA>{}, std::integral_constant<bool, VA>{}, full_c, ka, k0, va);
        fetch(pb, (size_t)N, std::integral_constant<bool, TB>{}, std::integral_constant<bool, VB>{}, full_c, kb, k0, vb);
    };
    const std::true_type yes;
    const std::false_type no;
    uint32_t amin = 0xffffffffu, bmin = 0xffffffffu;
    // STAND: zeros are staged as kZeroStand.
    auto stash_chunk = [&](int buf, auto stand_c) __attribute__((always_inline)) {
        constexpr bool STAND = decltype(stand_c)::value;
#pragma unroll
        for (int j = 0; j < L; j++) {
            uint4 qa, qb;
            T *ea = reinterpret_cast<T *>(&qa), *eb = reinterpret_cast<T *>(&qb);
#pragma unroll
            for (int c = 0; c < P; c++) {
                ea[c] = STAND && is_zero(va[j][c]) ? kZeroStand<T> : va[j][c];
                eb[c] = STAND && is_zero(vb[j][c]) ? kZeroStand<T> : vb[j][c];
                const uint32_t x = exp_key(va[j][c]), y = exp_key(vb[j][c]);
                amin = x < amin ? x : amin;
                bmin = y < bmin ? y : bmin;
            }
            *reinterpret_cast<uint4 *>(&As[buf][xa][ka + 16 * P * j]) = qa;
            *reinterpret_cast<uint4 *>(&Bs[buf][xb][kb + 16 * P * j]) = qb;
        }
    };
    T acc = (T)0;
    // 16 P k of the stage are a block: lane tx of a lane row holds its row's k = P tx ..
    // P tx + P - 1 of it, and group j of P k takes lane j's.
    constexpr int BL = 16 * P;
    auto load16 = [](const T *p, T (&v)[P]) __attribute__((always_inline)) {
        const uint4 q = *reinterpret_cast<const uint4 *>(p);
        const T *e = reinterpret_cast<const T *>(&q);
#pragma unroll
        for (int c = 0; c < P; c++)
            v[c] = e[c];
    };
    auto products = [](auto j_c, const T (&a)[P], const T (&b)[P], T (&p)[P]) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < P; c++)
            p[c] = row_lane<decltype(j_c)::value>(a[c]) * b[c];
    };
    // `blocks` whole blocks, four k at a time. While four products are summed the next four
    // are formed, and op(B) is read 16 k ahead (an LDS read takes longer than 12); the last
    // block's reads ahead repeat its own first groups.
    constexpr int G = 4 / P, NQ = 16 / G; // groups of four k; fours a block
    auto whole_blocks = [&](const T *as, const T *bs, int blocks) __attribute__((always_inline)) {
        T a[P], an[P], b[4][G][P], p[2][G][P];
        load16(as + P * tx, a);
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int g = 0; g < G; g++)
                load16(bs + 4 * q + P * g, b[q][g]);
        products(std::integral_constant<int, 0>{}, a, b[0][0], p[0][0]);
        products(std::integral_constant<int, G - 1>{}, a, b[0][G - 1], p[0][G - 1]);
        for (int i = 0; i < blocks; i++) {
            const int ahead = i + 1 < blocks ? BL : 0;
            as += ahead;
            load16(as + P * tx, an);
            each<NQ>([&](auto q_c) __attribute__((always_inline)) {
                constexpr int q = decltype(q_c)::value, n = (q + 1) % NQ; // n: the next four
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int g = 0; g < G; g++)
                    load16(bs + (q < NQ - 4 ? 4 * (q + 4) : ahead + 4 * (q + 4 - NQ)) + P * g, b[q & 3][g]);
                const T(&x)[P] = q + 1 < NQ ? a : an;
                products(std::integral_constant<int, G * n>{}, x, b[n & 3][0], p[n & 1][0]);
                if constexpr (G == 2)
                    products(std::integral_constant<int, G * n + G - 1>{}, x, b[n & 3][G - 1], p[n & 1][G - 1]);
#pragma unroll
                for (int g = 0; g < G; g++)
#pragma unroll
                    for (int c = 0; c < P; c++)
                        acc = acc + p[q & 1][g][c];
            });
            __builtin_amdgcn_sched_barrier(0);
            bs += ahead;
#pragma unroll
            for (int c = 0; c < P; c++)
                a[c] = an[c];
        }
    };
    // The last, partial block, four groups at a time (zeros pad the last), op(B) read four groups
    // ahead.
    auto part_block = [&](const T *as, const T *bs, int left) __attribute__((always_inline)) {
        T a[P], b[2][4][P];
        load16(as + P * tx, a);
#pragma unroll
        for (int g = 0; g < 4; g++)
            load16(bs + P * g, b[0][g]);
        each<4>([&](auto u_c) __attribute__((always_inline)) {
            constexpr int u = decltype(u_c)::value;
            if (4 * P * u < left) {
                if constexpr (u < 3)
#pragma unroll
                    for (int g = 0; g < 4; g++)
                        load16(bs + P * (4 * u + 4 + g), b[(u + 1) & 1][g]);
                each<4>([&](auto g_c) __attribute__((always_inline)) {
                    constexpr int g = decltype(g_c)::value;
                    T p[P];
                    products(std::integral_constant<int, 4 * u + g>{}, a, b[u & 1][g], p);
#pragma unroll
                    for (int c = 0; c < P; c++)
                        acc = acc + p[c];
                });
            }
        });
    };
    auto last_chunk = [&](int buf, int kc) __attribute__((always_inline)) {
        if (kc >= BL)
            whole_blocks(&As[buf][ty][0], &Bs[buf][tx][0], kc / BL);
        if (kc % BL != 0)
            part_block(&As[buf][ty][kc / BL * BL], &Bs[buf][tx][kc / BL * BL], kc % BL);
    };
    if constexpr (ONE) {
        fetch_chunk(no, 0);
        stash_chunk(0, no);
        __syncthreads();
        last_chunk(0, K);
    } else {
        // A chunk that another follows. The two kinds of next chunk are separate code: where their
        // loads met, the compiler waited for them before the sums.
        auto chunk = [&](auto full_c, int k0, int buf) __attribute__((always_inline)) {
            fetch_chunk(full_c, k0 + BK);
            whole_blocks(&As[buf][ty][0], &Bs[buf][tx][0], BK / BL);
            stash_chunk(buf ^ 1, no);
            __syncthreads();
        };
        fetch_chunk(yes, 0); // K > BK
        stash_chunk(0, no);
        __syncthreads();
        int k0 = 0, buf = 0;
        for (; k0 + 2 * BK <= K; k0 += BK, buf ^= 1)
            chunk(yes, k0, buf);
        if (k0 + BK < K) {
            chunk(no, k0, buf);
            k0 += BK;
            buf ^= 1;
        }
        last_chunk(buf, K - k0);
    }
    if (amin != 0xffffffffu)
        atomicMin(&rkey[xa], amin);
    if (bmin != 0xffffffffu)
        atomicMin(&ckey[xb], bmin);
    __syncthreads(); // every exponent folded
    const int crow = m0 + ty, ccol = n0 + tx;
    bool sus = false;
    if (crow < M && ccol < N) {
        C[(size_t)crow * N + ccol] = acc;
        sus = !finite_bits(acc) || (risk && key_exp<T>(rkey[ty]) + key_exp<T>(ckey[tx]) < thr);
    }
    if (!__syncthreads_or(sus)) {
        program_close_block(close);
        return;
    }
    // The search. Nothing is left to it where another block has already recorded a fault before this
    // one's first suspect cell: a NaN in a row or column of many blocks costs few of them a walk and
    // an atomic on the node's word. A block whose first suspect cell is not finite has its first
    // fault there (such a result comes of a fault), and a wave walks that cell alone.
    const uint64_t mask = __ballot(sus);
    if (mask != 0 && (tid & 63) == __ffsll((long long)mask) - 1)
        atomicMin(&first_sus, 2 * tid + (int)finite_bits(acc));
    if (tid == 0)
        best = __atomic_load_n(fault, __ATOMIC_RELAXED);
    __syncthreads();
    const int i = first_sus >> 1;
    const uint64_t cell0 = (uint64_t)(m0 + (i >> 4)) * N + n0 + (i & 15);
    if (best < pack_fault(cell0 * (uint64_t)K * 2, 0)) {
        program_close_block(close);
        return;
    }
    if (!(first_sus & 1)) {
        if (tid < 64) {
            const uint64_t w = cell_first_fault(A, B, (uint64_t)M, (uint64_t)N, (uint64_t)K, (int)TA, (int)TB,
                                                cell0, policy, true);
            if (w != kNoFault && tid == 0) {
                atomicMin(fault, (unsigned long long)w);
                gate_record(gate);
            }
        }
        program_close_block(close);
        return;
    }
    // Else every suspect cell's lane walks its own k again, the chunks staged as before, until its
    // first fault. A finite cell (and so each of its sums) can only fault in a tiny product, unless
    // subnormal sums are rejected; a block of such cells forms no sums. One lane a cell, so a block
    // whose every cell is suspect costs about as much again as the products did: 64 x 4096 x 1024
    // binary32 124 us, 53 clean, where a wave for each cell, 64 k at a time, took 5000.
    const uint64_t first_step = ((uint64_t)crow * N + ccol) * (uint64_t)K * 2; // of the lane's cell
    const bool adds = policy == kPolicyRejectSubnormal || __syncthreads_or(sus && !finite_bits(acc));
    T t = (T)0;
    for (int k0 = 0; k0 < K; k0 += BK) {
        if (!adds || !ONE) { // a single chunk still stands in its stage
            fetch_chunk(no, k0);
            if (adds)
                stash_chunk(0, no);
            else
                stash_chunk(0, yes);
            __syncthreads();
        }
        uint64_t key = kNoFault;
        if (__ballot(sus)) {
            const int kc = K - k0 < BK ? K - k0 : BK;
            const uint64_t step = first_step + 2 * (uint64_t)k0;
            key = adds ? chunk_first_fault<T, true>(&As[0][ty][0], &Bs[0][tx][0], kc, t, sus, step, policy)
                       : chunk_first_fault<T, false>(&As[0][ty][0], &Bs[0][tx][0], kc, t, sus, step, policy);
            if (key != kNoFault)
                atomicMin(&best, (unsigned long long)key);
        }
        __syncthreads();
        // Cells after a cell with a fault need no walk.
        sus = sus && key == kNoFault && pack_fault(first_step, 0) < best;
        if (!__syncthreads_or(sus))
            break;
    }
    if (tid == 0 && best != kNoFault) {
        atomicMin(fault, best);
        gate_record(gate);
    }
    program_close_block(close);
}

static inline bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

template <typename T, bool TA, bool TB>
static void small_launch(hipStream_t s, dim3 grid, const T *A, const T *B, T *C, int M, int N, int K,
                         int thr, int risk, int policy, unsigned long long *fault, NodeGate gate,
                         ProgramClose close)
{
    constexpr int P = 16 / (int)sizeof(T);
    const bool va = !TA && K % P == 0 && aligned16(A), vb = TB && K % P == 0 && aligned16(B);
    auto form = [&](auto va_c, auto vb_c) {
        constexpr bool VA = decltype(va_c)::value, VB = decltype(vb_c)::value;
        if (K <= 16 * P)
            hipLaunchKernelGGL((k_strict_gemm_small<T, TA, TB, VA, VB, 1, true>), grid, dim3(256), 0, s, A, B, C, M, N, K, thr, risk, policy, fault, gate, close);
        else if (K <= 64 * P)
            hipLaunchKernelGGL((k_strict_gemm_small<T, TA, TB, VA, VB, 4, true>), grid, dim3(256), 0, s, A, B, C, M, N, K, thr, risk, policy, fault, gate, close);
        else
            hipLaunchKernelGGL((k_strict_gemm_small<T, TA, TB, VA, VB, 4, false>), grid, dim3(256), 0, s, A, B, C, M, N, K, thr, risk, policy, fault, gate, close);
    };
    if ((TA || va) && (!TB || vb))
        form(std::integral_constant<bool, !TA>{}, std::integral_constant<bool, TB>{});
    else
        form(std::false_type{}, std::false_type{});
}

template <typename T>
static void small_layout(hipStream_t s, dim3 grid, bool ta, bool tb, const T *A, const T *B, T *C,
                         int M, int N, int K, int thr, int risk, int policy,
                         unsigned long long *fault, NodeGate gate, ProgramClose close)
{
    if (!ta && !tb)
        small_launch<T, false, false>(s, grid, A, B, C, M, N, K, thr, risk, policy, fault, gate, close);
    else if (!ta && tb)
        small_launch<T, false, true>(s, grid, A, B, C, M, N, K, thr, risk, policy, fault, gate, close);
    else if (ta && !tb)
        small_launch<T, true, false>(s, grid, A, B, C, M, N, K, thr, risk, policy, fault, gate, close);
    else
        small_launch<T, true, true>(s, grid, A, B, C, M, N, K, thr, risk, policy, fault, gate, close);
}

// Estimated microseconds of this kernel, from kernel times on MI355X of 1 to 64 workgroups a CU and
// K = 8 to 4096 (a fixed part, and each workgroup of the fullest CU its own): the forms of one chunk
// have 4 to 6 workgroups of a CU beside each other, the two-stage form two. Kernels of 4 / 8 / 16
// workgroups a CU: binary32 K = 8 4.4 / 5.7 / 9.7 us, K = 64 5.2 / 7.8 / 12.2, K = 256 10.9 / 15.4 /
// 26.6, K = 1024 28.8 / 54.4 / 102.9; binary64 K = 8 4.4 / 6.3 / 9.5, K = 64 8.3 / 13.0 / 21.5, K =
// 256 17.1 / 30.2 / 56.3, K = 1024 53.6 / 102 / 196.
static double small_time(int dtype, double c, uint64_t inner)
{
    const double K = (double)inner, k = K / 1024.0;
    if (dtype == 0) {
        if (inner <= 64)
            return 3.3 + c * (0.33 + 0.0033 * K);
        if (inner <= 256)
            return 4 + c * (0.62 + 0.0028 * K);
        return c <= 1 ? 4.5 + 8.6 * k : 3 + c * (0.7 + 5.79 * k);
    }
    if (inner <= 32)
        return 3.3 + c * (0.3 + 0.0085 * K);
    if (inner <= 128)
        return 4.5 + c * (0.6 + 0.0065 * K);
    return c <= 1 ? 3.5 + 16.5 * k : 4 + c * (0.15 + 12.5 * k);
}

// Against the screened tile kernels: their screen (about 4.5 us, 2 more for each 1024 k of a row,
// and both operands at 6 MB a us), the tiles as mid_time_f32 and mid_wanted_f64 put them with the store
// of the output (and, binary64, a fixed part), and the further launches (0.5 us; whole calls of
// either route otherwise take their kernels and 11.5 us). AllowGradual needs no screen, only a
// launch that opens the words (2.5 to 3.2 us: binary32 768 x 19 x 2270 25.0 us on tiles, 26.2 here;
// 512 x 256 x 1024 24.1 / 25.9, 26.5 / 26.5 under IEEE). Whole calls, this kernel against the tiles,
// on both sides of the line: binary32 512 x 8 x 1024 18.0 / 21.0 us, 1024 x 8 x 1024 20.7 / 22.2, 4096
// x 8 x 512 26.0 / 24.5, 1024 x 64 x 1024 23.8 / 24.9, 512 x 100 x 1024 23.2 / 23.8, 1024 x 100 x 1024
// 30.4 / 26.7, 512 x 256 x 512 21.5 / 25.3, 512 x 1024 x 256 28.7 / 50; binary64 1024 x 8 x 1024 21.7
// / 23.0, 4096 x 8 x 512 27.5 / 25.8, 512 x 128 x 1024 27.9 / 33.1, 1024 x 128 x 1024 44 / 34.
bool gemm_small_wanted(int dtype, uint64_t rows, uint64_t inner, uint64_t cols, int policy)
{
    const auto per_cu = [&](uint64_t t) {
        const uint64_t tiles = ((rows + t - 1) / t) * ((cols + t - 1) / t);
        return (double)((tiles + kGfx950Cus - 1) / kGfx950Cus);
    };
    // A launch holds fewer than 2^32 threads: one a cell.
    if (((rows + 15) / 16) * ((cols + 15) / 16) > UINT32_MAX / 256)
        return false;
    const double k = (double)inner / 1024.0, cells = (double)rows * (double)cols;
    const double mb = ((double)rows + (double)cols) * (double)inner * (dtype == 0 ? 4e-6 : 8e-6);
    double tiles = policy == kPolicyAllowGradual ? (dtype == 0 ? 2.5 : 3.2) : 4.5 + 2 * k + mb / 6 + 0.5;
    if (dtype == 0) {
        tiles += mid_time_f32(rows, cols, inner) + 0.5 + 1e-6 * cells;
    } else {
        const double c64 = per_cu(64);
        tiles += (c64 <= 2 ? 26 + 65 * c64 : 74 * c64) * k + 3.5 + 1.8e-6 * cells;
    }
    return small_time(dtype, per_cu(16), inner) < tiles;
}

hipError_t launch_gemm_small(hipStream_t s, int dtype, int M, int N, int K, bool ta, bool tb,
                             const void *A, const void *B, void *C, int thr, int risk, int policy,
                             unsigned long long *fault, NodeGate gate, ProgramClose close,
                             bool *closed)
{
    const dim3 grid((unsigned)((((uint64_t)M + 15) / 16) * (((uint64_t)N + 15) / 16)));
    if (grid.x > kCloseMaxBlocks)
        close = ProgramClose{}; // the publication launch ends the program
    if (closed)
        *closed = close.words != nullptr;
    if (dtype == 0)
        small_layout<float>(s, grid, ta, tb, (const float *)A, (const float *)B, (float *)C, M, N, K, thr, risk, policy, fault, gate, close);
    else
        small_layout<double>(s, grid, ta, tb, (const double *)A, (const double *)B, (double *)C, M, N, K, thr, risk, policy, fault, gate, close);
    return hipGetLastError();
}

} // namespace pcu
