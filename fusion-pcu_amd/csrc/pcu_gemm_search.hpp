// The exact first-fault search of one strict MatMul cell (gfx950), shared by the replay and the
// small-output kernel.
#pragma once

#include "pcu_device.hpp"

namespace pcu {

// Lane l's value of v, on every lane (l uniform across the wave).
__device__ __forceinline__ float lane_value(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double lane_value(double v, int l)
{
    const uint64_t x = bits_of(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), l);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// First fault of one output cell, found by a whole wave (every lane returns the same). One
// pass over k in chunks of 64, the next chunk's operands loaded while the current one is
// classified: the lanes form the chunk's products and classify them, which gives the
// chunk's first faulting Multiply. When `walk_adds` is set (a non-finite result, where a sum
// can overflow, or RejectSubnormal, where a subnormal sum faults), every lane then folds the
// chunk's products before that Multiply in k order, as the contract orders the sums. Those
// products are finite, so a sum there can only fault by overflowing (the running sum turns,
// and stays, infinite) or, under RejectSubnormal, by being subnormal: the chunk is folded
// with plain adds and that check, and only a chunk that trips it is folded again with the
// exact add classifier to name the step. A Multiply at k comes before the Add at k. Returns
// kNoFault or the packed fault word.
template <typename T>
__device__ __forceinline__ uint64_t cell_first_fault(const T *__restrict__ A, const T *__restrict__ B,
                                                     uint64_t M, uint64_t N, uint64_t K, int ta,
                                                     int tb, uint64_t cell, int policy,
                                                     bool walk_adds)
{
    const int lane = threadIdx.x & 63;
    const uint64_t r = cell / N, c = cell % N;
    auto load = [&](uint64_t k0, T &a, T &b) {
        const uint64_t k = k0 + lane;
        a = (T)0;
        b = (T)0;
        if (k < K) {
            a = ta ? A[k * M + r] : A[r * K + k];
            b = tb ? B[c * K + k] : B[k * N + c];
        }
    };
    const bool reject_sub = policy == kPolicyRejectSubnormal;
    T total = (T)0;
    T a, b;
    load(0, a, b);
    for (uint64_t k0 = 0; k0 < K; k0 += 64) {
        T na = (T)0, nb = (T)0;
        if (k0 + 64 < K)
            load(k0 + 64, na, nb);
        const T p = a * b;
        uint32_t kind = kOk;
        if (k0 + lane < K)
            kind = classify_mul(a, b, p, policy);
        const uint64_t mask = __ballot(kind != kOk);
        const int l_m = mask ? __ffsll((long long)mask) - 1 : 64;
        if (walk_adds) {
            const int in_k = K - k0 < 64 ? (int)(K - k0) : 64;
            const int here = l_m < in_k ? l_m : in_k; // products summed before any fault
            T t = total;
            bool sub = false;
            if (here == 64) {
#pragma unroll
                for (int j = 0; j < 64; j++) {
                    t = t + lane_value(p, j);
                    sub |= reject_sub && subnormal(t);
                }
            } else {
                for (int j = 0; j < here; j++) {
                    t = t + lane_value(p, j);
                    sub |= reject_sub && subnormal(t);
                }
            }
            if (!finite_bits(t) || sub) {
                for (int j = 0; j < here; j++) {
                    const T pj = lane_value(p, j);
                    const T nxt = total + pj;
                    const uint32_t k_add = classify_add(total, pj, nxt, policy);
                    if (k_add != kOk)
                        return pack_fault((cell * K + k0 + j) * 2 + 1, k_add);
                    total = nxt;
                }
            }
            total = t;
        }
        if (mask)
            return pack_fault((cell * K + k0 + l_m) * 2, __shfl(kind, l_m, 64));
        a = na;
        b = nb;
    }
    return kNoFault;
}

// Lane 0's value, on every lane of the wave.
__device__ __forceinline__ uint64_t wave_uniform_u64(uint64_t v)
{
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}

} // namespace pcu
