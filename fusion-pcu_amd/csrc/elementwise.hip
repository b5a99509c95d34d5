// Bandwidth-bound strict kernels: checked Add/Sub/Mul/Div (tensor or uniform right
// operand), ReLU, ReLU-backward, fused Add->ReLU, strict SGD and strict MSE.
//
// Layout: dense row-major tensors in HBM. One thread moves one 16-byte vector per operand
// (4 floats or 2 doubles) and the grid covers the whole tensor in 256-thread blocks, with
// non-temporal loads and stores: on MI355X this streams at about 83% of the 8 TB/s HBM
// peak, ahead of every grid-stride shape tried (2^28 f32 SGD: 6.55-6.64 TB/s, against
// 6.32-6.52 with 128-thread blocks and 6.43 / 6.34 with 512 / 1024). The last vector may be partial (scalar
// accesses for its in-range elements). Faults are screened per lane, resolved exactly
// only on flagged lanes, and reduced with one ballot per wave and one atomicMin per
// faulting wave into the op's 64-bit fault word.
#include "pcu_device.hpp"
#include "pcu_kernels.hpp"

#include <limits.h>

#pragma clang fp contract(off)

namespace pcu {

constexpr int kEwThreads = 256;

template <typename T> struct Vec;
template <> struct Vec<float> {
    typedef float type __attribute__((ext_vector_type(4)));
    static constexpr int width = 4;
};
template <> struct Vec<double> {
    typedef double type __attribute__((ext_vector_type(2)));
    static constexpr int width = 2;
};

template <typename T, bool VEC> struct Lanes {
    static constexpr int W = VEC ? Vec<T>::width : 1;
};

// Elements [base, base + W) of p that lie below n (the rest read as +0 and must be masked
// by the caller). A whole vector is one non-temporal 16-byte load.
template <typename T, bool VEC>
__device__ __forceinline__ void load_lanes(const T *p, uint64_t base, uint64_t n,
                                           T (&v)[Lanes<T, VEC>::W])
{
    constexpr int W = Lanes<T, VEC>::W;
    if (VEC && base + W <= n) {
        typedef typename Vec<T>::type V;
        const V q = __builtin_nontemporal_load(reinterpret_cast<const V *>(p + base));
#pragma unroll
        for (int j = 0; j < W; j++)
            v[j] = q[j];
    } else {
#pragma unroll
        for (int j = 0; j < W; j++)
            v[j] = base + j < n ? __builtin_nontemporal_load(p + base + j) : (T)0;
    }
}

template <typename T, bool VEC, bool NT = true>
__device__ __forceinline__ void store_lanes(T *p, uint64_t base, uint64_t n,
                                            const T (&v)[Lanes<T, VEC>::W])
{
    constexpr int W = Lanes<T, VEC>::W;
    if (VEC && base + W <= n) {
        typedef typename Vec<T>::type V;
        V q;
#pragma unroll
        for (int j = 0; j < W; j++)
            q[j] = v[j];
        if (NT)
            __builtin_nontemporal_store(q, reinterpret_cast<V *>(p + base));
        else
            *reinterpret_cast<V *>(p + base) = q;
    } else {
#pragma unroll
        for (int j = 0; j < W; j++)
            if (base + j < n) {
                if (NT)
                    __builtin_nontemporal_store(v[j], p + base + j);
                else
                    p[base + j] = v[j];
            }
    }
}

// First element index of this thread's vector and the distance to its next one (the grid
// normally covers the tensor, so the loop body runs once).
#define PCU_EW_LOOP(W)                                                                          \
    const uint64_t pcu_stride = (uint64_t)gridDim.x * kEwThreads * (W);                         \
    for (uint64_t base = ((uint64_t)blockIdx.x * kEwThreads + threadIdx.x) * (W); base < n;     \
         base += pcu_stride)

template <typename T, int OP>
__device__ __forceinline__ T apply(T a, T b)
{
    if (OP == kOpAdd) return a + b;
    if (OP == kOpSub) return a - b;
    if (OP == kOpMul) return a * b;
    return a / b;
}

template <typename T, int OP>
__device__ __forceinline__ bool suspect(T a, T b, T r, int policy)
{
    if (OP == kOpAdd || OP == kOpSub) return add_suspect(a, b, r, policy);
    if (OP == kOpMul) return mul_suspect(a, b, r, policy);
    return div_suspect(a, b, r, policy);
}

template <typename T, int OP>
__device__ __forceinline__ uint32_t classify(T a, T b, T r, int policy)
{
    if (OP == kOpAdd || OP == kOpSub) return classify_add(a, b, r, policy);
    if (OP == kOpMul) return classify_mul(a, b, r, policy);
    return classify_div(a, b, r, policy);
}

// ------------------------------------------------------------ checked binary
// The checked elementwise and SGD kernels may run in place (out equal to an operand), so
// none of their pointers is __restrict__: a fault is classified from register values after
// the store, and the compiler may not reload an operand from memory the store overwrote.

template <typename T, int OP, bool UNIFORM, bool VEC>
__global__ __launch_bounds__(kEwThreads) void k_binary(const T *a,
                                                       const T *b, T b_value,
                                                       T *out, uint64_t n,
                                                       int policy, unsigned long long *fault, NodeGate gate)
{
    if (wave_gate_closed(gate))
        return;
    constexpr int W = Lanes<T, VEC>::W;
    uint64_t key = kNoFault;
    PCU_EW_LOOP(W)
    {
        T x[W], y[W], r[W];
        load_lanes<T, VEC>(a, base, n, x);
        if (UNIFORM) {
#pragma unroll
            for (int j = 0; j < W; j++)
                y[j] = b_value;
        } else {
            load_lanes<T, VEC>(b, base, n, y);
        }
        bool any = false;
#pragma unroll
        for (int j = 0; j < W; j++) {
            r[j] = apply<T, OP>(x[j], y[j]);
            any |= base + j < n && suspect<T, OP>(x[j], y[j], r[j], policy);
        }
        store_lanes<T, VEC>(out, base, n, r);
        if (any && key == kNoFault) {
#pragma unroll
            for (int j = 0; j < W; j++) {
                if (base + j >= n || key != kNoFault)
                    continue;
                const uint32_t kind = classify<T, OP>(x[j], y[j], r[j], policy);
                if (kind != kOk)
                    key = pack_fault(base + j, kind);
            }
        }
    }
    wave_record_fault(key, fault, gate);
}

// -------------------------------------------------------------------- relu

template <typename T, bool VEC>
__global__ __launch_bounds__(kEwThreads) void k_relu(const T *x, T *out,
                                                     uint64_t n, int policy,
                                                     unsigned long long *fault, NodeGate gate)
{
    if (wave_gate_closed(gate))
        return;
    constexpr int W = Lanes<T, VEC>::W;
    uint64_t key = kNoFault;
    PCU_EW_LOOP(W)
    {
        T v[W], r[W];
        load_lanes<T, VEC>(x, base, n, v);
        bool any = false;
#pragma unroll
        for (int j = 0; j < W; j++) {
            r[j] = relu_select(v[j]);
            any |= base + j < n &&
                   (!finite_bits(v[j]) || (policy == kPolicyRejectSubnormal && subnormal(r[j])));
        }
        store_lanes<T, VEC>(out, base, n, r);
        if (any && key == kNoFault) {
#pragma unroll
            for (int j = 0; j < W; j++) {
                if (base + j >= n || key != kNoFault)
                    continue;
                const uint32_t kind = classify_relu(v[j], r[j], policy);
                if (kind != kOk)
                    key = pack_fault(base + j, kind);
            }
        }
    }
    wave_record_fault(key, fault, gate);
}

// ---------------------------------------------------------- relu backward

template <typename T, bool VEC>
__global__ __launch_bounds__(kEwThreads) void k_relu_backward(const T *x,
                                                              const T *up,
                                                              T *out, uint64_t n,
                                                              int policy,
                                                              unsigned long long *fault, NodeGate gate)
{
    if (wave_gate_closed(gate))
        return;
    constexpr int W = Lanes<T, VEC>::W;
    uint64_t key = kNoFault;
    PCU_EW_LOOP(W)
    {
        T v[W], u[W], r[W];
        load_lanes<T, VEC>(x, base, n, v);
        load_lanes<T, VEC>(up, base, n, u);
        bool any = false;
#pragma unroll
        for (int j = 0; j < W; j++) {
            r[j] = strictly_positive(v[j]) ? u[j] : (T)0;
            any |= base + j < n && (!finite_bits(v[j]) || !finite_bits(u[j]) ||
                                    (policy == kPolicyRejectSubnormal && subnormal(r[j])));
        }
        store_lanes<T, VEC>(out, base, n, r);
        if (any && key == kNoFault) {
#pragma unroll
            for (int j = 0; j < W; j++) {
                if (base + j >= n || key != kNoFault)
                    continue;
                const uint32_t kind = classify_relu_backward(v[j], u[j], r[j], policy);
                if (kind != kOk)
                    key = pack_fault(base + j, kind);
            }
        }
    }
    wave_record_fault(key, fault, gate);
}

// ------------------------------------------------------------ fused add->relu
// The Add node's faults go to fault_add and the ReLU node's to fault_relu, so the
// node-major first-fault order is the same as running the two nodes one after the other
// (a ReLU of a successful, hence finite, sum can only fault under RejectSubnormal).

template <typename T, bool UNIFORM, bool VEC>
__global__ __launch_bounds__(kEwThreads) void k_add_relu(const T *a,
                                                         const T *b, T b_value,
                                                         T *out, uint64_t n,
                                                         int policy,
                                                         unsigned long long *fault_add,
                                                         unsigned long long *fault_relu, NodeGate gate)
{
    if (wave_gate_closed(gate))
        return;
    constexpr int W = Lanes<T, VEC>::W;
    uint64_t key_add = kNoFault, key_relu = kNoFault;
    PCU_EW_LOOP(W)
    {
        T x[W], y[W], sum[W], r[W];
        load_lanes<T, VEC>(a, base, n, x);
        if (UNIFORM) {
#pragma unroll
            for (int j = 0; j < W; j++)
                y[j] = b_value;
        } else {
            load_lanes<T, VEC>(b, base, n, y);
        }
        bool any = false;
#pragma unroll
        for (int j = 0; j < W; j++) {
            sum[j] = x[j] + y[j];
            r[j] = relu_select(sum[j]);
            any |= base + j < n && (add_suspect(x[j], y[j], sum[j], policy) ||
                                    (policy == kPolicyRejectSubnormal && subnormal(r[j])));
        }
        store_lanes<T, VEC>(out, base, n, r);
        if (any) {
#pragma unroll
            for (int j = 0; j < W; j++) {
                if (base + j >= n)
                    continue;
                const uint32_t ka = classify_add(x[j], y[j], sum[j], policy);
                if (ka != kOk) {
                    if (key_add == kNoFault)
                        key_add = pack_fault(base + j, ka);
                } else {
                    const uint32_t kr = classify_relu(sum[j], r[j], policy);
                    if (kr != kOk && key_relu == kNoFault)
                        key_relu = pack_fault(base + j, kr);
                }
            }
        }
    }
    wave_record_fault(key_add, fault_add, gate);
    wave_record_fault(key_relu, fault_relu, NodeGate{gate.word, gate.node + 1});
}

// ---------------------------------------------------------- fused chains
// Consecutive elementwise nodes of a prepared program, each an operand of the next, in one
// pass over the elements: the values between steps stay in registers, and only the values
// another node reads are stored. Each step's faults go to its own node's word and every
// step is classified as its own kernel classifies it, so the node-major first fault is the
// one the nodes give one after another (a step may also record a fault on a value a
// faulting earlier step produced: the earlier node's fault is the one reported).
template <typename T> __device__ __forceinline__ T chain_uniform(uint64_t bits)
{
    if constexpr (sizeof(T) == 4)
        return __builtin_bit_cast(float, (uint32_t)bits);
    else
        return __builtin_bit_cast(double, bits);
}

template <typename T> __device__ __forceinline__ T chain_binary(int op, T a, T b)
{
    switch (op) {
    case kOpAdd: return a + b;
    case kOpSub: return a - b;
    case kOpMul: return a * b;
    default: return a / b;
    }
}

template <typename T> __device__ __forceinline__ bool chain_suspect(int op, T a, T b, T r, int policy)
{
    if (op == kOpAdd || op == kOpSub) return add_suspect(a, b, r, policy);
    if (op == kOpMul) return mul_suspect(a, b, r, policy);
    return div_suspect(a, b, r, policy);
}

template <typename T> __device__ __forceinline__ uint32_t chain_classify(int op, T a, T b, T r, int policy)
{
    if (op == kOpAdd || op == kOpSub) return classify_add(a, b, r, policy);
    if (op == kOpMul) return classify_mul(a, b, r, policy);
    return classify_div(a, b, r, policy);
}

// A chain's step operations known when the kernel is compiled: op of step s in bits
// 4s..4s+3 of SIG, or SIG < 0 (read from the launch). The common chains get kernels of
// their own, with the other operations' code folded away.
constexpr int chain_sig_op(int sig, int s) { return sig < 0 ? -1 : (sig >> (4 * s)) & 15; }
constexpr int chain_sig(int op0, int op1, int op2 = -1, int op3 = -1)
{
    return op0 | op1 << 4 | (op2 < 0 ? 0 : op2 << 8) | (op3 < 0 ? 0 : op3 << 12);
}
constexpr int kSigSubMul = chain_sig(kOpSub, kOpMul);                          // MSE gradient
constexpr int kSigAddRelu = chain_sig(kOpAdd, kStepRelu);                       // bias + ReLU
constexpr int kSigSubMulReluBack = chain_sig(kOpSub, kOpMul, kStepReluBackward); // C1 backward

// The other operand of step S on the lanes [base, base + W) (nothing for a ReLU).
template <typename T, bool VEC, int S, int SIG>
__device__ __forceinline__ void chain_other(const ChainLaunch &c, uint64_t base, uint64_t n,
                                            T (&o)[Lanes<T, VEC>::W])
{
    constexpr int W = Lanes<T, VEC>::W;
    const ChainStep &st = c.step[S];
    constexpr int kop = chain_sig_op(SIG, S);
    const int op = kop >= 0 ? kop : st.op;
    if (S >= c.steps || op == kStepRelu)
        return;
    if (st.other) {
        load_lanes<T, VEC>((const T *)st.other, base, n, o);
    } else {
        const T u = chain_uniform<T>(st.other_bits);
#pragma unroll
        for (int j = 0; j < W; j++)
            o[j] = u;
    }
}

// The first fault of a chain step on the lanes [base, base + W) (kNoFault: none), the rare
// path once a lane is suspect. Out of line, so that the classifiers' code and registers stay
// out of the streaming loop (inlined into each step they spilled scalar registers into
// vector lanes).
template <typename T, int W> struct LaneVals {
    T x[W];
};
template <typename T, int W>
__device__ __forceinline__ uint64_t chain_first_fault_body(int op, int policy, bool right,
                                                           const LaneVals<T, W> &v,
                                                           const LaneVals<T, W> &o,
                                                           const LaneVals<T, W> &r, uint64_t base,
                                                           uint64_t n)
{
#pragma unroll
    for (int j = 0; j < W; j++) {
        if (base + j >= n)
            break;
        uint32_t kind;
        if (op == kStepRelu) {
            kind = classify_relu(v.x[j], r.x[j], policy);
        } else {
            const T a = right ? o.x[j] : v.x[j], b = right ? v.x[j] : o.x[j];
            kind = op == kStepReluBackward ? classify_relu_backward(a, b, r.x[j], policy)
                                           : chain_classify(op, a, b, r.x[j], policy);
        }
        if (kind != kOk)
            return pack_fault(base + j, kind);
    }
    return kNoFault;
}
// The call itself makes the kernel keep its scalar arguments in vector lanes across it, so
// the kernels with their operations fixed at compile time (small once folded) inline it.
template <typename T, int W>
__device__ __noinline__ uint64_t chain_first_fault(int op, int policy, bool right, LaneVals<T, W> v,
                                                   LaneVals<T, W> o, LaneVals<T, W> r,
                                                   uint64_t base, uint64_t n)
{
    return chain_first_fault_body<T, W>(op, policy, right, v, o, r, base, n);
}

// Step S of a chain on the lanes [base, base + W): v holds the value the step takes and is
// replaced by the step's result, o the step's other operand (chain_other); key keeps the
// step's first fault in this thread.
template <typename T, bool VEC, int S, int SIG>
__device__ __forceinline__ void chain_step(const ChainLaunch &c, uint64_t base, uint64_t n,
                                           T (&v)[Lanes<T, VEC>::W], const T (&o)[Lanes<T, VEC>::W],
                                           uint64_t &key)
{
    constexpr int W = Lanes<T, VEC>::W;
    const ChainStep &st = c.step[S];
    constexpr int kop = chain_sig_op(SIG, S);
    const int op = kop >= 0 ? kop : st.op, policy = st.policy;
    const bool right = st.chain_right != 0;
    T r[W];
    bool any = false;
    if (op == kStepRelu) {
#pragma unroll
        for (int j = 0; j < W; j++) {
            r[j] = relu_select(v[j]);
            any |= base + j < n && (!finite_bits(v[j]) || (policy == kPolicyRejectSubnormal && subnormal(r[j])));
        }
    } else if (op == kStepReluBackward) {
#pragma unroll
        for (int j = 0; j < W; j++) {
            const T x = right ? o[j] : v[j], u = right ? v[j] : o[j];
            r[j] = strictly_positive(x) ? u : (T)0;
            any |= base + j < n && (!finite_bits(x) || !finite_bits(u) ||
                                    (policy == kPolicyRejectSubnormal && subnormal(r[j])));
        }
    } else {
#pragma unroll
        for (int j = 0; j < W; j++) {
            const T a = right ? o[j] : v[j], b = right ? v[j] : o[j];
            r[j] = chain_binary(op, a, b);
            any |= base + j < n && chain_suspect(op, a, b, r[j], policy);
        }
    }
    if (st.out)
        store_lanes<T, VEC>((T *)st.out, base, n, r);
    if (any && key == kNoFault) {
        LaneVals<T, W> lv, lo, lr;
#pragma unroll
        for (int j = 0; j < W; j++) {
            lv.x[j] = v[j];
            lo.x[j] = o[j];
            lr.x[j] = r[j];
        }
        if constexpr (kop >= 0)
            key = chain_first_fault_body<T, W>(op, policy, right, lv, lo, lr, base, n);
        else
            key = chain_first_fault<T, W>(op, policy, right, lv, lo, lr, base, n);
    }
#pragma unroll
    for (int j = 0; j < W; j++)
        v[j] = r[j];
}

// NS = c.steps, a template argument: a kernel for all four steps held every step's
// parameters and registers at once and spilled scalar registers into vector lanes (about 750
// lane reads; a two-step chain ran at half the speed of one checked binary op over the
// same bytes).
template <typename T, bool VEC, int NS, int SIG = -1>
__global__ __launch_bounds__(kEwThreads) void k_chain(ChainLaunch c, uint64_t n, NodeGate gate)
{
    static_assert(NS >= 1 && NS <= kChainMaxSteps && kChainMaxSteps == 4,
                  "one chain_step call per step below");
    if (wave_gate_closed(gate))
        return;
    constexpr int W = Lanes<T, VEC>::W;
    uint64_t k0 = kNoFault, k1 = kNoFault, k2 = kNoFault, k3 = kNoFault;
    PCU_EW_LOOP(W)
    {
        // Every operand is loaded before any step stores: no step reads a value stored in
        // this launch (the plan keeps chain members out of other operands), so the loads go
        // out together, one round trip, instead of one after each step's stores.
        T v[W], o0[W], o1[W], o2[W], o3[W];
        load_lanes<T, VEC>((const T *)c.head, base, n, v);
        chain_other<T, VEC, 0, SIG>(c, base, n, o0);
        if constexpr (NS > 1)
            chain_other<T, VEC, 1, SIG>(c, base, n, o1);
        if constexpr (NS > 2)
            chain_other<T, VEC, 2, SIG>(c, base, n, o2);
        if constexpr (NS > 3)
            chain_other<T, VEC, 3, SIG>(c, base, n, o3);
        chain_step<T, VEC, 0, SIG>(c, base, n, v, o0, k0);
        if constexpr (NS > 1)
            chain_step<T, VEC, 1, SIG>(c, base, n, v, o1, k1);
        if constexpr (NS > 2)
            chain_step<T, VEC, 2, SIG>(c, base, n, v, o2, k2);
        if constexpr (NS > 3)
            chain_step<T, VEC, 3, SIG>(c, base, n, v, o3, k3);
    }
    wave_record_fault(k0, c.step[0].fault, gate);
    if constexpr (NS > 1)
        wave_record_fault(k1, c.step[1].fault, NodeGate{gate.word, gate.node + 1});
    if constexpr (NS > 2)
        wave_record_fault(k2, c.step[2].fault, NodeGate{gate.word, gate.node + 2});
    if constexpr (NS > 3)
        wave_record_fault(k3, c.step[3].fault, NodeGate{gate.word, gate.node + 3});
}

// -------------------------------------------------------------------- SGD
// core/dialect/tensor/reference/strict_sgd/strict_sgd.rs:20-46: p = rate (x) g, then
// w' = w (-) p; ordinal 2i (Multiply) and 2i+1 (Subtract).

// Blocks [bid, ...) of nb blocks over one update.
template <typename T, bool VEC>
__device__ __forceinline__ void sgd_range(const T *w, const T *g, T rate, T *out, uint64_t n,
                                          int policy, unsigned long long *fault, NodeGate gate,
                                          uint64_t bid, uint64_t nb)
{
    if (wave_gate_closed(gate))
        return;
    constexpr int W = Lanes<T, VEC>::W;
    uint64_t key = kNoFault;
    const uint64_t stride = nb * kEwThreads * W;
    for (uint64_t base = (bid * kEwThreads + threadIdx.x) * W; base < n; base += stride) {
        T wv[W], gv[W], p[W], r[W];
        load_lanes<T, VEC>(w, base, n, wv);
        load_lanes<T, VEC>(g, base, n, gv);
        bool any = false;
#pragma unroll
        for (int j = 0; j < W; j++) {
            p[j] = rate * gv[j];
            r[j] = wv[j] - p[j];
            any |= base + j < n && (mul_suspect(rate, gv[j], p[j], policy) |
                                    add_suspect(wv[j], p[j], r[j], policy));
        }
        store_lanes<T, VEC>(out, base, n, r);
        if (any && key == kNoFault) {
#pragma unroll
            for (int j = 0; j < W; j++) {
                if (base + j >= n || key != kNoFault)
                    continue;
                const uint32_t km = classify_mul(rate, gv[j], p[j], policy);
                if (km != kOk) {
                    key = pack_fault(2 * (base + j), km);
                } else {
                    const uint32_t ks = classify_add(wv[j], p[j], r[j], policy);
                    if (ks != kOk)
                        key = pack_fault(2 * (base + j) + 1, ks);
                }
            }
        }
    }
    wave_record_fault(key, fault, gate);
}

template <typename T, bool VEC>
__global__ __launch_bounds__(kEwThreads) void k_sgd(const T *w,
                                                    const T *g, T rate,
                                                    T *out, uint64_t n, int policy,
                                                    unsigned long long *fault, NodeGate gate,
                                                    ProgramClose close)
{
    sgd_range<T, VEC>(w, g, rate, out, n, policy, fault, gate, blockIdx.x, gridDim.x);
    program_close_block(close);
}

// Two updates of one program in one launch: blocks [0, blocks0) take update 0, the rest
// update 1; each keeps its own fault word and gate.
template <typename T> struct SgdPairArgs {
    const T *w[2], *g[2];
    T *out[2];
    T rate[2];
    uint64_t n[2];
    unsigned long long *fault[2];
    NodeGate gate[2];
    unsigned blocks0;
};

template <typename T, bool VEC>
__global__ __launch_bounds__(kEwThreads) void k_sgd_pair(SgdPairArgs<T> a, int policy,
                                                         ProgramClose close)
{
    const bool first = blockIdx.x < a.blocks0;
    const int u = first ? 0 : 1;
    const uint64_t bid = first ? blockIdx.x : blockIdx.x - a.blocks0;
    const uint64_t nb = first ? a.blocks0 : gridDim.x - a.blocks0;
    sgd_range<T, VEC>(a.w[u], a.g[u], a.rate[u], a.out[u], a.n[u], policy, a.fault[u], a.gate[u],
                      bid, nb);
    program_close_block(close);
}

// -------------------------------------------------------------------- MSE
// core/dialect/tensor/reference/strict_mse/strict_mse.rs:22-59. Stage 1 (parallel):
// d = p (-) t and s = d (x) d per element, ordinals 3i and 3i+1. Stage 2 (one wave): the
// ordered sum total = total (+) s_i from +0 (ordinal 3i+2), then total (/) count
// (ordinal 3n). The sum is a dependent chain by contract; it stops before the first
// element whose Subtract or Multiply faulted.

// Ordered sum of the squares, exact and parallel. Every square is +0 or positive, so the
// running total never decreases. While the total stays inside one binade [2^E, 2^(E+1))
// (or below the smallest normal), it is m * u for an integer m and the binade's quantum u,
// and one rounded step total (+) s equals (m + r) * u where r is s/u rounded to the nearest
// integer, a tie going to the r that makes m + r even. So inside a binade the chain is a
// prefix sum of integers whose only coupling is the parity of m at each tie: a two-state
// automaton, which composes associatively and scans in parallel. What a run of squares adds from
// an even and from an odd m is read off two chains of plain adds, from the binade's first two
// values. The run holding the first element whose step would reach the binade's upper end is
// executed as real rounded hardware adds, checked like every other Add, and its total starts the
// next phase. Results equal the dependent chain of the contract bit for bit.

template <typename T> struct SumBits;
template <> struct SumBits<float> {
    using U = uint32_t;
    using C = uint32_t;                  // step counts: a binade holds 2^24 quanta at most
    static constexpr int kFrac = 23;     // stored fraction bits
    static constexpr int kQmin = -149;   // exponent of the smallest subnormal
    static constexpr uint32_t kExpAll = 0xff;
    static constexpr int kPer = 16;      // elements per thread of a full-chunk scan
    static constexpr C kBig = 1u << 25;  // count of a run that surely leaves the binade
    static constexpr C kCap = 1u << 30;  // saturation of prefix counts (past any crossing)
};
template <> struct SumBits<double> {
    using U = uint64_t;
    using C = uint64_t;
    static constexpr int kFrac = 52;
    static constexpr int kQmin = -1074;
    static constexpr uint32_t kExpAll = 0x7ff;
    static constexpr int kPer = 8;
    static constexpr C kBig = 1ull << 54;
    static constexpr C kCap = 1ull << 62;
};

// Threads of a chunk's scan; a chunk is kPer elements for each.
constexpr int kSumThreads = 512;
// Inputs of up to kMseSerialMax elements are summed by one wave (k_mse_serial).
constexpr uint64_t kMseSerialMax = 2048;
constexpr int kQuarters = 4; // parts of a chunk that the squares kernel sums on their own

template <typename T>
__device__ __forceinline__ typename SumBits<T>::C sat_add(typename SumBits<T>::C a,
                                                          typename SumBits<T>::C b)
{
    const typename SumBits<T>::C c = a + b; // a, b <= kCap: no wrap
    return c < SumBits<T>::kCap ? c : SumBits<T>::kCap;
}

// Effect of a run of steps as a function of the parity of m before it: the added count
// and the parity after it, for each starting parity (bit 0: start even, bit 1: start odd).
template <typename C> struct SumScanT {
    C r0, r1;
    uint32_t p;
};
template <typename T> using SumScan = SumScanT<typename SumBits<T>::C>;

template <typename T> __device__ __forceinline__ SumScan<T> scan_identity() { return SumScan<T>{0, 0, 2u}; }

template <typename T>
__device__ __forceinline__ SumScan<T> scan_compose(const SumScan<T> &a, const SumScan<T> &b)
{
    const uint32_t a0 = a.p & 1u, a1 = (a.p >> 1) & 1u;
    const uint32_t b0 = b.p & 1u, b1 = (b.p >> 1) & 1u;
    SumScan<T> c;
    c.r0 = sat_add<T>(a.r0, a0 ? b.r1 : b.r0);
    c.r1 = sat_add<T>(a.r1, a1 ? b.r1 : b.r0);
    c.p = (a0 ? b1 : b0) | ((a1 ? b1 : b0) << 1);
    return c;
}

// Cross-lane moves of a summary. DPP (a register read across lanes, no LDS): a lane
// whose source lies outside the pattern, or whose row the row mask leaves out, keeps old.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp_c(uint32_t old, uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, CTRL, ROW_MASK, 0xf, false);
}
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint64_t dpp_c(uint64_t old, uint64_t v)
{
    const uint32_t lo = dpp_c<CTRL, ROW_MASK>((uint32_t)old, (uint32_t)v);
    const uint32_t hi = dpp_c<CTRL, ROW_MASK>((uint32_t)(old >> 32), (uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}

template <typename T, int CTRL, int ROW_MASK>
__device__ __forceinline__ SumScan<T> scan_dpp(const SumScan<T> &v)
{
    const SumScan<T> id = scan_identity<T>();
    return SumScan<T>{dpp_c<CTRL, ROW_MASK>(id.r0, v.r0), dpp_c<CTRL, ROW_MASK>(id.r1, v.r1),
                      dpp_c<CTRL, ROW_MASK>(id.p, v.p)};
}

__device__ __forceinline__ uint32_t readlane_c(uint32_t v, int l) { return (uint32_t)__builtin_amdgcn_readlane((int)v, l); }
__device__ __forceinline__ uint64_t readlane_c(uint64_t v, int l)
{
    return ((uint64_t)readlane_c((uint32_t)(v >> 32), l) << 32) | readlane_c((uint32_t)v, l);
}

template <typename T>
__device__ __forceinline__ SumScan<T> scan_readlane(const SumScan<T> &v, int l)
{
    return SumScan<T>{readlane_c(v.r0, l), readlane_c(v.r1, l), readlane_c(v.p, l)};
}

template <typename T>
__device__ __forceinline__ SumScan<T> scan_shfl_up(const SumScan<T> &v, int d)
{
    return SumScan<T>{__shfl_up(v.r0, d, 64), __shfl_up(v.r1, d, 64), __shfl_up(v.p, d, 64)};
}

// DPP patterns of the wave scan: row_shr:1,2,4,8 inside each row of 16 lanes, then
// row_bcast:15 (lane 15 of rows 0 and 2 into rows 1 and 3) and row_bcast:31 (lane 31 into
// rows 2 and 3).
constexpr int kDppRowShr1 = 0x111, kDppRowShr2 = 0x112, kDppRowShr4 = 0x114, kDppRowShr8 = 0x118;
constexpr int kDppRowBcast15 = 0x142, kDppRowBcast31 = 0x143;

// Inclusive ordered composition over the 64 lanes of a wave.
template <typename T>
__device__ __forceinline__ SumScan<T> wave_scan_incl(SumScan<T> v)
{
    v = scan_compose<T>(scan_dpp<T, kDppRowShr1, 0xf>(v), v);
    v = scan_compose<T>(scan_dpp<T, kDppRowShr2, 0xf>(v), v);
    v = scan_compose<T>(scan_dpp<T, kDppRowShr4, 0xf>(v), v);
    v = scan_compose<T>(scan_dpp<T, kDppRowShr8, 0xf>(v), v);
    v = scan_compose<T>(scan_dpp<T, kDppRowBcast15, 0xa>(v), v);
    v = scan_compose<T>(scan_dpp<T, kDppRowBcast31, 0xc>(v), v);
    return v;
}

// Phase of a total given by its bits: quantum exponent, count m and the count at which
// the next binade starts.
template <typename T>
__device__ __forceinline__ void sum_phase(typename SumBits<T>::U bits, int &ue,
                                          typename SumBits<T>::C &m, typename SumBits<T>::C &mmax)
{
    using B = SumBits<T>;
    using C = typename B::C;
    const uint32_t e = (uint32_t)(bits >> B::kFrac) & B::kExpAll;
    if (e == 0) {
        ue = B::kQmin;
        m = (C)bits;
        mmax = (C)1 << B::kFrac;
    } else {
        ue = (int)e + B::kQmin - 1;
        m = ((C)bits & (((C)1 << B::kFrac) - 1)) | ((C)1 << B::kFrac);
        mmax = (C)1 << (B::kFrac + 1);
    }
}

template <typename T>
__device__ __forceinline__ typename SumBits<T>::U sum_bits(int ue, typename SumBits<T>::C m)
{
    using B = SumBits<T>;
    using U = typename B::U;
    if (ue == B::kQmin && m < ((typename B::C)1 << B::kFrac))
        return (U)m;
    return (U)(((U)(ue - B::kQmin) << B::kFrac) + (U)m);
}

template <typename T>
__device__ __forceinline__ T from_bits(typename SumBits<T>::U b);
template <>
__device__ __forceinline__ float from_bits<float>(uint32_t b) { return __uint_as_float(b); }
template <>
__device__ __forceinline__ double from_bits<double>(uint64_t b) { return __longlong_as_double((long long)b); }

// Whether 2^ue is the quantum of some binade.
template <typename T> __device__ __forceinline__ bool phase_valid(int ue)
{
    return ue >= SumBits<T>::kQmin && ue - SumBits<T>::kQmin + 1 < (int)SumBits<T>::kExpAll;
}

// Effect of the squares v (+0: none) on the quantum 2^ue. The count a run adds depends on the
// count before it only through its parity, so it is what two chains of rounded adds gain that
// start at the binade's first value and at the one after it: inside a binade the bits are the
// count (the subnormals share the quantum of the first normal binade, whose values stand in for
// them). A chain that leaves the binade has added more than any total in it can take. Two adds a
// square against some 40 instructions of integer steps: the summaries of 4096 x 1024 f32 squares
// took 15.9 us with those, 7.3 so.
template <typename T, int N>
__device__ __forceinline__ SumScan<T> run_summary(const T (&v)[N], int ue)
{
    using B = SumBits<T>;
    using U = typename B::U;
    const U even = (U)(ue - B::kQmin + 1) << B::kFrac, odd = even + 1, end = even + ((U)1 << B::kFrac);
    T t0 = from_bits<T>(even), t1 = from_bits<T>(odd);
#pragma unroll
    for (int j = 0; j < N; j++) {
        t0 = t0 + v[j];
        t1 = t1 + v[j];
    }
    const U b0 = (U)bits_of(t0), b1 = (U)bits_of(t1);
    SumScan<T> s;
    s.r0 = b0 < end ? b0 - even : B::kBig; // NaN and infinities lie past the end
    s.r1 = b1 < end ? b1 - odd : B::kBig;
    s.p = (uint32_t)(s.r0 & 1u) | ((uint32_t)((s.r1 + 1) & 1u) << 1);
    return s;
}

// ----------------------------------------------------- ordered sum: pipeline
// The squares are cut into chunks of 512*P elements (P = 16 for binary32, 8 for binary64).
//  A  k_mse_squares          the squares, and each quarter chunk's sum in binary64 (an
//                            estimate: order does not matter);
//  B  k_mse_chunk_prefix     the chunks' sums and their exclusive prefix: about where the
//                            running total stands at each chunk start (C's own work for
//                            up to 512 chunks);
//  C  k_mse_chunk_summaries  per chunk, in parallel, the summary (count added for an even
//                            and an odd start) of the whole chunk inside one binade, for
//                            the one or two binades the estimate allows;
//  D  k_mse_ordered_walk     one workgroup walks the chunks in order, 512 at a time: a scan
//                            of the summaries made for the running binade folds every chunk
//                            before the first one that has no such summary or reaches the
//                            binade's end. That chunk runs exactly: the run of 16 (8)
//                            squares holding the crossing is added square by square, checked
//                            like every other Add, and the runs after it fold from the
//                            prefixes made for the next binade; where several crossings
//                            share a chunk, one wave adds the squares one by one while they
//                            are dense, and elsewhere the workgroup scans windows sized from
//                            the chunk's estimate.
// The estimate only decides how fast the walk goes, never its value.

struct ChunkSummary {
    uint64_t r0, r1;   // count added starting from an even / odd count
    int32_t ue;        // quantum exponent the summary was made for (kNoPhase: none)
    uint32_t pad;
};
constexpr int32_t kNoPhase = INT32_MIN;
constexpr uint32_t kNoStep = 0xffffffffu;

template <typename T> __device__ __forceinline__ uint64_t sum_chunk_len() { return (uint64_t)kSumThreads * SumBits<T>::kPer; }

__device__ __forceinline__ uint64_t sum_limit(const unsigned long long *fault, uint64_t n)
{
    // Elements at or after the first Subtract/Multiply fault are never summed.
    const uint64_t w = __atomic_load_n(fault, __ATOMIC_RELAXED);
    return w == kNoFault ? n : (w >> 3) / 3;
}

// Quantum exponent of the binade a total of about x lies in.
template <typename T>
__device__ __forceinline__ int32_t phase_ue_of(double x)
{
    using B = SumBits<T>;
    const double min_normal = ldexp(1.0, B::kQmin + B::kFrac);
    if (!(x >= min_normal))
        return B::kQmin;
    int e;
    (void)frexp(x, &e); // x = f * 2^e, f in [1/2, 1): floor(log2 x) = e - 1
    return e - 1 - B::kFrac;
}

// Thread t's P elements of the chunk at base (elements at or past limit read as 0).
template <typename T>
__device__ __forceinline__ void load_chunk(const typename SumBits<T>::U *__restrict__ src,
                                           bool vec_ok, uint64_t base, uint64_t limit, int tid,
                                           typename SumBits<T>::U (&dst)[SumBits<T>::kPer])
{
    using U = typename SumBits<T>::U;
    constexpr int P = SumBits<T>::kPer;
    const uint64_t first = base + (uint64_t)tid * P;
    if (vec_ok && base + sum_chunk_len<T>() <= limit) {
        const uint4 *v = reinterpret_cast<const uint4 *>(src + first);
        constexpr int per16 = 16 / sizeof(U);
#pragma unroll
        for (int q = 0; q < P / per16; q++) {
            const uint4 x = v[q];
            const U *xs = reinterpret_cast<const U *>(&x);
#pragma unroll
            for (int j = 0; j < per16; j++)
                dst[q * per16 + j] = xs[j];
        }
    } else {
#pragma unroll
        for (int j = 0; j < P; j++)
            dst[j] = first + j < limit ? src[first + j] : (U)0;
    }
}

// Ordered composition over the workgroup: every thread gets the summary of all threads
// before it (excl) and of the whole workgroup (total).
template <typename T>
__device__ __forceinline__ void block_scan(const SumScan<T> &mine, int lane, int wave,
                                           SumScan<T> *wave_tot, SumScan<T> &excl,
                                           SumScan<T> &total)
{
    constexpr int kWaves = kSumThreads / 64;
    static_assert(kWaves <= 8, "the wave totals are scanned inside one DPP row");
    const SumScan<T> inc = wave_scan_incl<T>(mine);
    SumScan<T> lane_excl = scan_shfl_up<T>(inc, 1);
    if (lane == 0)
        lane_excl = scan_identity<T>();
    if (lane == 63)
        wave_tot[wave] = inc;
    __syncthreads();
    // Every wave scans the per-wave totals on the first lanes of its first row.
    SumScan<T> wt = lane < kWaves ? wave_tot[lane] : scan_identity<T>();
    wt = scan_compose<T>(scan_dpp<T, kDppRowShr1, 0xf>(wt), wt);
    wt = scan_compose<T>(scan_dpp<T, kDppRowShr2, 0xf>(wt), wt);
    wt = scan_compose<T>(scan_dpp<T, kDppRowShr4, 0xf>(wt), wt);
    total = scan_readlane<T>(wt, kWaves - 1);
    SumScan<T> before = scan_readlane<T>(wt, wave > 0 ? wave - 1 : 0);
    if (wave == 0)
        before = scan_identity<T>();
    excl = scan_compose<T>(before, lane_excl);
}

// A chunk staged in LDS for its exact run: element i sits at slot i + i / kPadEvery (one
// spare slot per 128 bytes), so that runs of 2..16 consecutive elements per thread spread
// over distinct banks.
template <typename T> struct ChunkLds {
    using U = typename SumBits<T>::U;
    static constexpr uint32_t kPadEvery = 128 / sizeof(U);
    static constexpr uint32_t kLen = kSumThreads * SumBits<T>::kPer;
    static constexpr uint32_t kSlots = kLen + kLen / kPadEvery;
    __device__ static __forceinline__ uint32_t slot(uint32_t i) { return i + i / kPadEvery; }
};

// Shared state of the ordered walk. The step slots are double-buffered by iteration: one
// is written during an iteration while the other is cleared for the next.
template <typename T> struct WalkShared {
    typename SumBits<T>::U vals[ChunkLds<T>::kSlots];
    SumScan<T> wave_tot[kSumThreads / 64];
    uint64_t m_first[2];             // count standing before the stopping chunk
    uint32_t first[2];               // stopping chunk of a batch (offset), kNoStep: none
    uint32_t at[2];                  // element after a window's crossing run, or after a
                                     // serial walk (offset); kNoStep: no crossing
    typename SumBits<T>::U total[2]; // total before that element
    int stop[2];                     // an Add faulted
    int first_cand[2];               // candidate summary the stopping chunk matched, or -1
    double mean[2];                  // the stopping chunk's mean square (an estimate)
    // Result of a chunk's run-prefix fold (written by the one thread holding the crossing).
    uint64_t run_m;
    int run_status, run_ue;
    uint32_t run_resume;
    uint64_t limit;
};

// Summary of elements [i0, min(i0 + PER, i1)) of the staged chunk on the quantum 2^ue.
template <typename T, int PER>
__device__ __forceinline__ SumScan<T> run_scan(const typename SumBits<T>::U *vals, uint32_t i0,
                                               uint32_t i1, int ue)
{
    T v[PER];
#pragma unroll
    for (int j = 0; j < PER; j++)
        v[j] = i0 + j < i1 ? from_bits<T>(vals[ChunkLds<T>::slot(i0 + j)]) : (T)0;
    return run_summary<T, PER>(v, ue);
}

template <typename T>
__device__ __forceinline__ SumScan<T> run_scan_per(const typename SumBits<T>::U *vals,
                                                   uint32_t per, uint32_t i0, uint32_t i1, int ue)
{
    constexpr int P = SumBits<T>::kPer;
    if (per == 1)
        return run_scan<T, 1>(vals, i0, i1, ue);
    if (per == 2)
        return run_scan<T, 2>(vals, i0, i1, ue);
    if (per == 4)
        return run_scan<T, 4>(vals, i0, i1, ue);
    if (P > 8 && per == 8)
        return run_scan<T, 8>(vals, i0, i1, ue);
    return run_scan<T, P>(vals, i0, i1, ue);
}

// Expected number of squares (at the chunk's mean square) until the running total leaves
// its binade: room quanta of 2^ue left.
__device__ __forceinline__ double expected_gap(double room, int ue, double mean)
{
    return mean > 0.0 ? ldexp(room, ue) / mean : INFINITY;
}

// Elements per thread of the next window: a power of two covering about twice the expected
// gap, from one element per thread up to the whole chunk.
template <typename T>
__device__ __forceinline__ uint32_t window_per(double gap)
{
    constexpr uint32_t P = SumBits<T>::kPer;
    const double span = 2.0 * gap / kSumThreads;
    uint32_t per = 1;
    while (per < P && (double)per < span)
        per <<= 1;
    return per;
}

// Below this expected gap (in squares) one wave folds the squares one by one with plain adds: a
// window costs 2.2 to 2.9 us, the time of about 500 such adds. The fold stops at the first binade whose
// expected gap reaches kSerialGap, or after kSerialMax squares (then a window runs next, whatever
// the estimate says).
constexpr double kSerialGap = 512.0;
constexpr uint32_t kSerialMax = 4096;

// `count` squares from global element `at` on, given by read(0 .. count - 1), added to `total` one
// by one with the exact add classifier: false when an Add faulted (recorded).
template <typename T, class F>
__device__ __forceinline__ bool fold_exact(T total, uint32_t count, uint64_t at, int policy,
                                                     unsigned long long *fault, const NodeGate &gate,
                                                     F read)
{
    for (uint32_t i = 0; i < count; i++) {
        const T s_i = read(i);
        const T nxt = total + s_i;
        const uint32_t kind = classify_add(total, s_i, nxt, policy);
        if (kind != kOk) {
            atomicMin(fault, (unsigned long long)pack_fault(3 * (at + i) + 2, kind));
            gate_record(gate);
            return false;
        }
        total = nxt;
    }
    return true;
}

// One thread's run of squares (those past its end +0, which change no total) added to `total`.
// The squares are finite and not negative, so a sum can only fault by overflowing (the total
// turns, and stays, infinite) or, under RejectSubnormal, by being subnormal: plain adds and that
// check, and only a run that trips it goes through the exact classifier. Returns false when an
// Add faulted (recorded).
template <typename T, class F>
__device__ __forceinline__ bool fold_run(const T (&v)[SumBits<T>::kPer], T &total, uint32_t count,
                                         uint64_t at, int policy, unsigned long long *fault,
                                         const NodeGate &gate, F read)
{
    T t = total;
    bool sub = false;
#pragma unroll
    for (int j = 0; j < SumBits<T>::kPer; j++) {
        t = t + v[j];
        sub |= subnormal(t);
    }
    if (!finite_bits(t) || (sub && policy == kPolicyRejectSubnormal))
        if (!fold_exact<T>(total, count, at, policy, fault, gate, read))
            return false;
    total = t;
    return true;
}

// t = t + (lane j's v) for j = 0 .. 63 in order. Each lane value goes through a scalar register,
// read four adds ahead (the ties keep that order: a read right before its add would be waited
// for). f sees every partial sum.
__device__ __forceinline__ void tie_scalar(uint32_t &x) { asm volatile("" : "+s"(x)); }
__device__ __forceinline__ void tie_scalar(uint64_t &x) { asm volatile("" : "+s"(x)); }

template <typename T, class F>
__device__ __forceinline__ T fold_lanes(T t, typename SumBits<T>::U v, F &&f)
{
    typename SumBits<T>::U q[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        q[j] = readlane_c(v, j);
        tie_scalar(q[j]);
    }
#pragma unroll
    for (int j = 0; j < 64; j++) {
        t = t + from_bits<T>(q[j & 3]);
        asm volatile("" : "+v"(t));
        f(t);
        if (j + 4 < 64) {
            q[j & 3] = readlane_c(v, j + 4);
            tie_scalar(q[j & 3]);
        }
    }
    return t;
}

// The serial fold (wave 0 alone; every value it keeps is uniform over the wave). Lane l holds
// square off + l, and each add takes its square from that lane through a scalar register, read
// while the add before it is in flight, so a square costs the latency of one dependent add, about
// 4.6 ns. The squares are finite and not negative, so a sum can only fault by overflowing (the
// total turns, and stays, infinite) or, under RejectSubnormal, by being subnormal: 64 squares are
// folded with plain adds and that check, and only 64 that trip it are folded again with the exact
// add classifier. Returns false when an Add faulted (recorded).
template <typename T>
__device__ bool serial_walk(const typename SumBits<T>::U *vals, uint64_t base, uint32_t len,
                            double mean, int policy, unsigned long long *fault,
                            const NodeGate &gate, int lane, uint32_t &off, int &ue,
                            typename SumBits<T>::C &m, typename SumBits<T>::C &mmax)
{
    using U = typename SumBits<T>::U;
    const uint32_t end = off + kSerialMax < len ? off + kSerialMax : len;
    const bool reject_sub = policy == kPolicyRejectSubnormal;
    T total = from_bits<T>(sum_bits<T>(ue, m));
    auto load = [&](uint32_t o) { // squares past `end` read as +0, which changes no total
        const uint32_t i = o + lane < end ? o + lane : end - 1;
        const U x = vals[ChunkLds<T>::slot(i)];
        return o + lane < end ? x : (U)0;
    };
    U v = load(off);
    while (off < end) {
        const uint32_t here = end - off < 64 ? end - off : 64;
        const U nx = load(off + here);
        T t = total;
        bool sub = false;
        if (reject_sub)
            t = fold_lanes<T>(total, v, [&](T x) { sub |= subnormal(x); });
        else
            t = fold_lanes<T>(total, v, [](T) {});
        if (!finite_bits(t) || sub) {
            bool ok = true;
            if (lane == 0)
                ok = fold_exact<T>(total, here, base + off, policy, fault, gate, [&](uint32_t i) {
                    return from_bits<T>(vals[ChunkLds<T>::slot(off + i)]);
                });
            if (__ballot(!ok))
                return false;
        }
        total = t;
        off += here;
        const int was = ue;
        sum_phase<T>((U)bits_of(total), ue, m, mmax);
        if (ue != was && expected_gap((double)(mmax - m), ue, mean) >= kSerialGap)
            break;
        v = nx;
    }
    return true;
}

// Exact fold of elements [start, len) of the chunk at base, staged in sh.vals (its barrier is
// here), from the phase (ue, m, mmax): by the serial walk where crossings are dense, elsewhere
// window by window, where the one thread whose run holds the window's first step to reach the
// binade's end adds its run square by square and the next window starts after it, in the new
// binade. Returns false when an Add faulted (recorded).
template <typename T>
__device__ bool exact_chunk(uint64_t base, uint32_t len, uint32_t start, double mean, int policy,
                            unsigned long long *fault, int &ue, typename SumBits<T>::C &m,
                            typename SumBits<T>::C &mmax, WalkShared<T> &sh, const NodeGate &gate)
{
    using U = typename SumBits<T>::U;
    using C = typename SumBits<T>::C;
    constexpr uint32_t P = SumBits<T>::kPer;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid == 0)
        sh.at[0] = sh.at[1] = kNoStep;
    __syncthreads();
    uint32_t off = start, per = 0; // per = 0: no window has run yet
    bool serial_ok = true;
    for (int it = 0; off < len; it++) {
        const int slot = it & 1;
        const double gap = expected_gap((double)(mmax - m), ue, mean);
        if (serial_ok && gap < kSerialGap) {
            if (wave == 0) {
                uint32_t o = off;
                int u = ue;
                C mm = m, mx = mmax;
                const bool ok = serial_walk<T>(sh.vals, base, len, mean, policy, fault, gate, lane,
                                               o, u, mm, mx);
                if (lane == 0) {
                    sh.stop[slot] = !ok;
                    sh.total[slot] = sum_bits<T>(u, mm);
                    sh.at[slot] = o;
                }
            }
            __syncthreads();
            const uint32_t next = sh.at[slot];
            const int stop = sh.stop[slot];
            const U tot = sh.total[slot];
            if (tid == 0)
                sh.at[slot ^ 1] = kNoStep;
            if (stop)
                return false;
            sum_phase<T>(tot, ue, m, mmax);
            serial_ok = next - off < kSerialMax;
            off = next;
            per = 0;
            continue;
        }
        // After a window without a crossing the next one is at least twice as long.
        const uint32_t want = window_per<T>(gap);
        per = per && 2 * per > want ? (2 * per < P ? 2 * per : P) : want;
        const uint32_t wend = off + per * kSumThreads < len ? off + per * kSumThreads : len;
        const uint32_t i0 = off + (uint32_t)tid * per;
        const uint32_t i1 = i0 + per < wend ? i0 + per : wend;
        const SumScan<T> mine = run_scan_per<T>(sh.vals, per, i0, i1, ue);
        SumScan<T> before, total;
        block_scan<T>(mine, lane, wave, sh.wave_tot, before, total);
        const uint32_t p0 = (uint32_t)(m & 1u);
        const C mt = sat_add<T>(m, p0 ? before.r1 : before.r0);
        const uint32_t pt = p0 ? (before.p >> 1) & 1u : before.p & 1u;
        // Counts only grow along the window, so exactly one run can start below the
        // binade's end and reach it.
        if (mt < mmax && sat_add<T>(mt, pt ? mine.r1 : mine.r0) >= mmax) {
            T v[P], tot_run = from_bits<T>(sum_bits<T>(ue, mt));
#pragma unroll
            for (uint32_t j = 0; j < P; j++)
                v[j] = i0 + j < i1 ? from_bits<T>(sh.vals[ChunkLds<T>::slot(i0 + j)]) : (T)0;
            const bool ok = fold_run<T>(v, tot_run, i1 - i0, base + i0, policy, fault, gate, [&](uint32_t i) {
                return from_bits<T>(sh.vals[ChunkLds<T>::slot(i0 + i)]);
            });
            sh.stop[slot] = !ok;
            sh.total[slot] = (U)bits_of(tot_run);
            sh.at[slot] = i1;
        }
        __syncthreads();
        const uint32_t at = sh.at[slot];
        const int stop = sh.stop[slot];
        const U tot = sh.total[slot];
        if (tid == 0)
            sh.at[slot ^ 1] = kNoStep;
        if (at == kNoStep) {
            m = sat_add<T>(m, p0 ? total.r1 : total.r0);
            off = wend;
            continue;
        }
        if (stop)
            return false;
        sum_phase<T>(tot, ue, m, mmax);
        off = at;
        per = 0;
        serial_ok = true;
    }
    return true;
}

// Summaries kept per chunk: the estimate's binade less and plus 1/512 of it (lo, hi) and,
// when the estimate says the chunk crosses a binade, the binade after hi (where the rest
// of the chunk lands after one crossing).
constexpr int kCands = 3;

template <typename T>
__device__ __forceinline__ SumScan<T> scan_of_summary(const ChunkSummary &c)
{
    using C = typename SumBits<T>::C;
    const C r0 = (C)c.r0, r1 = (C)c.r1;
    return SumScan<T>{r0, r1, (uint32_t)(r0 & 1u) | ((uint32_t)((r1 + 1) & 1u) << 1)};
}

// Run-prefix fold of the chunk at base whose summary `cand` (made for the running binade)
// reaches the binade's end. runs_c holds, per candidate, each thread run's exclusive prefix
// (run t = elements [P*t, P*t + P)). The run where the count reaches the end is the one
// whose prefixes straddle it; its thread adds the run's squares one by one (16 dependent adds,
// 0.1 us; stepping the automaton through them took about 3) and so lands in the new binade.
// The runs after it fold at once from the prefixes of a candidate made for the new binade:
// from parity q at the chunk start a candidate's prefix adds E(q) before run t and T(q) over
// the whole chunk, so the runs from t on add T(q) - E(q), for the q whose parity after E is
// the parity actually standing there. Every thread loads its squares and its prefixes of every
// candidate at once: one round trip to memory, which is most of the time (in a second one after
// the crossing is known, another). Returns 1 when the chunk is folded, 0 when an Add
// faulted (recorded), -1 when a second crossing (or a missing candidate) leaves elements
// [*resume, len) to the windowed path, with (ue, m, mmax) standing before element *resume.
template <typename T>
__device__ int run_prefix_chunk(const typename SumBits<T>::U *__restrict__ src,
                                const SumScan<T> *__restrict__ runs_c,
                                const ChunkSummary *__restrict__ summ_c, int cand, uint64_t base,
                                uint32_t len, int policy, unsigned long long *fault, int &ue,
                                typename SumBits<T>::C &m, typename SumBits<T>::C &mmax,
                                uint32_t &resume, WalkShared<T> &sh, const NodeGate &gate)
{
    using U = typename SumBits<T>::U;
    using C = typename SumBits<T>::C;
    constexpr uint32_t P = SumBits<T>::kPer;
    const int tid = threadIdx.x;
    U vals[P];
    load_chunk<T>(src, ((uintptr_t)src & 15u) == 0, base, base + len, tid, vals);
    ChunkSummary cs[kCands];
    SumScan<T> e0[kCands], e1[kCands];
    const int next = tid + 1 < kSumThreads ? tid + 1 : tid;
#pragma unroll
    for (int y = 0; y < kCands; y++) {
        cs[y] = summ_c[y];
        e0[y] = runs_c[(size_t)y * kSumThreads + tid];
        e1[y] = runs_c[(size_t)y * kSumThreads + next];
    }
    SumScan<T> E = e0[0], E1 = e1[0];
#pragma unroll
    for (int y = 0; y < kCands; y++) {
        if (next == tid)
            e1[y] = scan_of_summary<T>(cs[y]);
        if (y == cand) {
            E = e0[y];
            E1 = e1[y];
        }
    }
    const uint32_t p0 = (uint32_t)(m & 1u);
    const C mt = sat_add<T>(m, p0 ? E.r1 : E.r0), mt1 = sat_add<T>(m, p0 ? E1.r1 : E1.r0);
    // Counts only grow along the chunk: exactly one run starts below the end and reaches it.
    if (mt < mmax && mt1 >= mmax) {
        const uint32_t i0 = (uint32_t)tid * P, i1 = i0 + P < len ? i0 + P : len;
        T v[P], total = from_bits<T>(sum_bits<T>(ue, mt));
#pragma unroll
        for (uint32_t j = 0; j < P; j++)
            v[j] = from_bits<T>(vals[j]);
        const bool ok = fold_run<T>(v, total, i1 - i0, base + i0, policy, fault, gate,
                                    [&](uint32_t i) { return from_bits<T>(src[base + i0 + i]); });
        C mm, mx;
        int u, status = ok ? 1 : 0;
        sum_phase<T>((U)bits_of(total), u, mm, mx);
        if (ok && i1 < len) {
            // The runs after this one, from the prefixes of a candidate for the new binade.
            status = -1;
            const uint32_t pt = (uint32_t)(mm & 1u);
            bool found = false;
            SumScan<T> Ey = scan_identity<T>(), Ty = scan_identity<T>();
#pragma unroll
            for (int y = kCands - 1; y >= 0; y--)
                if (cs[y].ue == u) {
                    found = true;
                    Ey = e1[y];
                    Ty = scan_of_summary<T>(cs[y]);
                }
            const int q = (Ey.p & 1u) == pt ? 0 : (((Ey.p >> 1) & 1u) == pt ? 1 : -1);
            if (found && q >= 0) {
                const C tq = q ? Ty.r1 : Ty.r0, eq = q ? Ey.r1 : Ey.r0;
                if (tq < SumBits<T>::kCap && mm + (tq - eq) < mx) {
                    mm += tq - eq;
                    status = 1;
                }
            }
        }
        sh.run_status = status;
        sh.run_ue = u;
        sh.run_m = (uint64_t)mm;
        sh.run_resume = i1;
    }
    __syncthreads();
    const int status = sh.run_status;
    if (status == 0)
        return 0;
    sum_phase<T>(sum_bits<T>(sh.run_ue, (C)sh.run_m), ue, m, mmax);
    resume = sh.run_resume;
    return status;
}

// A: the squares, with the first faulting Subtract or Multiply, and beside them each quarter
// chunk's sum in binary64 (order does not matter: only an estimate, so what is not finite, at or
// after a fault, is left out). One quarter a workgroup, all of a thread's loads in flight at
// once; 12 bytes an element (f32) over memory bound it. A pass of its own over the squares for
// the sums took 4.6 us beside 14 at 4096 x 1024 f32.
template <typename T, bool VEC>
__global__ __launch_bounds__(kEwThreads) void k_mse_squares(const T *__restrict__ p,
                                                            const T *__restrict__ t,
                                                            T *__restrict__ sq, uint64_t n,
                                                            int policy,
                                                            double *__restrict__ quarter_sum,
                                                            unsigned long long *fault, NodeGate gate)
{
    if (block_gate_closed(gate))
        return;
    constexpr int W = Lanes<T, VEC>::W;
    constexpr int kQuarter = kSumThreads * SumBits<T>::kPer / kQuarters;
    constexpr int R = kQuarter / (kEwThreads * W);
    __shared__ double part[kEwThreads / 64];
    const uint64_t first = (uint64_t)blockIdx.x * kQuarter + threadIdx.x * W;
    uint64_t key = kNoFault;
    double acc = 0.0;
    T pv[R][W], tv[R][W];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint64_t base = first + (uint64_t)r * kEwThreads * W;
        if (base < n) {
            load_lanes<T, VEC>(p, base, n, pv[r]);
            load_lanes<T, VEC>(t, base, n, tv[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint64_t base = first + (uint64_t)r * kEwThreads * W;
        if (base >= n)
            break;
        T d[W], sv[W];
        bool any = false;
#pragma unroll
        for (int j = 0; j < W; j++) {
            d[j] = pv[r][j] - tv[r][j];
            sv[j] = d[j] * d[j];
            if (base + j < n) {
                any |= add_suspect(pv[r][j], tv[r][j], d[j], policy) |
                       mul_suspect(d[j], d[j], sv[j], policy);
                acc += finite_bits(sv[j]) ? (double)sv[j] : 0.0;
            }
        }
        // Ordinary stores: the ordered sum reads the squares next.
        store_lanes<T, VEC, false>(sq, base, n, sv);
        if (any && key == kNoFault) {
#pragma unroll
            for (int j = 0; j < W; j++) {
                if (base + j >= n || key != kNoFault)
                    continue;
                const uint32_t ks = classify_add(pv[r][j], tv[r][j], d[j], policy);
                if (ks != kOk) {
                    key = pack_fault(3 * (base + j), ks);
                } else {
                    const uint32_t km = classify_mul(d[j], d[j], sv[j], policy);
                    if (km != kOk)
                        key = pack_fault(3 * (base + j) + 1, km);
                }
            }
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        acc += __shfl_xor(acc, off, 64);
    if ((threadIdx.x & 63) == 0)
        part[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0)
        quarter_sum[blockIdx.x] = (part[0] + part[1]) + (part[2] + part[3]);
    wave_record_fault(key, fault, gate);
}

// B: chunk sums and their exclusive prefix (one workgroup; each thread a contiguous run).
constexpr int kPrefixThreads = 1024;
__global__ __launch_bounds__(kPrefixThreads) void k_mse_chunk_prefix(const double *__restrict__ quarter_sum,
                                                                     uint64_t chunks,
                                                                     double *__restrict__ chunk_sum,
                                                                     double *__restrict__ pre,
                                                                     NodeGate gate)
{
    if (block_gate_closed(gate))
        return;
    __shared__ double wave_sum[kPrefixThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint64_t per = (chunks + kPrefixThreads - 1) / kPrefixThreads;
    const uint64_t i0 = (uint64_t)tid * per;
    const uint64_t i1 = i0 + per < chunks ? i0 + per : chunks;
    double own = 0.0;
    for (uint64_t i = i0; i < i1; i++) {
        const double *q = quarter_sum + kQuarters * i;
        const double sum = (q[0] + q[1]) + (q[2] + q[3]);
        chunk_sum[i] = sum;
        own += sum;
    }
    double inc = own;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const double o = __shfl_up(inc, d, 64);
        if (lane >= d)
            inc += o;
    }
    if (lane == 63)
        wave_sum[wave] = inc;
    __syncthreads();
    double run = inc - own;
    for (int w = 0; w < wave; w++)
        run += wave_sum[w];
    for (uint64_t i = i0; i < i1; i++) {
        pre[i] = run;
        run += chunk_sum[i];
    }
}

// C: summary of chunk blockIdx.x for candidate blockIdx.y (0: the binade of the estimate
// less 1/512 of it; 1: plus 1/512, skipped when both agree; 2: the binade after candidate 1,
// only when the estimate says the chunk crosses), with every thread run's exclusive prefix.
// Up to kSumThreads chunks (chunk_pre null) each block sums the quarters before its chunk itself,
// four loads a thread at most, and the first block of a chunk stores its sum: 9.2 us at 512 chunks
// against 7.3 with a launch of 3.9 before it. With more chunks each block would read more.
template <typename T>
__global__ __launch_bounds__(kSumThreads) void k_mse_chunk_summaries(
    const T *__restrict__ sq, uint64_t n, const unsigned long long *fault,
    const double *__restrict__ quarter_sum, double *__restrict__ chunk_sum,
    const double *__restrict__ chunk_pre, ChunkSummary *__restrict__ summ,
    SumScan<T> *__restrict__ runs, NodeGate gate)
{
    if (block_gate_closed(gate))
        return;
    using U = typename SumBits<T>::U;
    constexpr int P = SumBits<T>::kPer;
    __shared__ SumScan<T> wave_tot[kSumThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint64_t c = blockIdx.x;
    const uint64_t limit = sum_limit(fault, n);
    double pre, own;
    if (chunk_pre != nullptr) {
        pre = chunk_pre[c];
        own = chunk_sum[c];
    } else {
        __shared__ double part[kSumThreads / 64];
        double q[kQuarters];
#pragma unroll
        for (int j = 0; j < kQuarters; j++) {
            const uint64_t i = (uint64_t)(kSumThreads * j + tid);
            q[j] = i < kQuarters * c ? quarter_sum[i] : 0.0;
        }
        const double *mine = quarter_sum + kQuarters * c;
        own = (mine[0] + mine[1]) + (mine[2] + mine[3]);
        if (blockIdx.y == 0 && tid == 0)
            chunk_sum[c] = own;
        double acc = (q[0] + q[1]) + (q[2] + q[3]);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1)
            acc += __shfl_xor(acc, off, 64);
        if (lane == 0)
            part[wave] = acc;
        __syncthreads();
        pre = 0.0;
#pragma unroll
        for (int w = 0; w < kSumThreads / 64; w++)
            pre += part[w];
    }
    const int32_t lo = phase_ue_of<T>(pre * (1.0 - 1.0 / 512)), hi = phase_ue_of<T>(pre * (1.0 + 1.0 / 512));
    const int32_t end = phase_ue_of<T>((pre + own) * (1.0 + 1.0 / 512));
    ChunkSummary *out = summ + kCands * c + blockIdx.y;
    const int ue = blockIdx.y == 0 ? lo : (blockIdx.y == 1 ? hi : hi + 1);
    if ((blockIdx.y == 1 && hi == lo) || (blockIdx.y == 2 && end <= lo) || !phase_valid<T>(ue)) {
        if (tid == 0)
            *out = ChunkSummary{0, 0, kNoPhase, 0};
        return;
    }
    const U *src = reinterpret_cast<const U *>(sq);
    U cur[P];
    const uint64_t base = c * sum_chunk_len<T>();
    load_chunk<T>(src, ((uintptr_t)sq & 15u) == 0, base, limit, tid, cur);
    T v[P];
#pragma unroll
    for (int j = 0; j < P; j++)
        v[j] = from_bits<T>(cur[j]);
    const SumScan<T> mine = run_summary<T, P>(v, ue);
    SumScan<T> excl, total;
    block_scan<T>(mine, lane, wave, wave_tot, excl, total);
    runs[(kCands * c + blockIdx.y) * kSumThreads + tid] = excl;
    if (tid == 0)
        *out = ChunkSummary{(uint64_t)total.r0, (uint64_t)total.r1, ue, 0};
}

// D: the ordered walk (one workgroup), then total (/) count.
template <typename T>
__device__ __forceinline__ void ordered_walk(const T *__restrict__ sq, uint64_t n, T count, int policy,
                                             T *__restrict__ out, unsigned long long *fault,
                                             const double *__restrict__ chunk_sum,
                                             const ChunkSummary *__restrict__ summ,
                                             const SumScan<T> *__restrict__ runs, const NodeGate &gate)
{
    if (block_gate_closed(gate))
        return;
    using U = typename SumBits<T>::U;
    using C = typename SumBits<T>::C;
    constexpr C kBig = SumBits<T>::kBig;
    __shared__ WalkShared<T> sh;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid == 0) {
        sh.limit = sum_limit(fault, n);
        sh.first[0] = sh.first[1] = kNoStep;
    }
    __syncthreads();
    const uint64_t limit = sh.limit;
    const U *src = reinterpret_cast<const U *>(sq);
    const uint64_t L = sum_chunk_len<T>();
    const uint64_t chunks = (limit + L - 1) / L;

    int ue;
    C m, mmax;
    sum_phase<T>((U)0, ue, m, mmax); // the total starts at +0
    // Batches of 512 chunks: thread t keeps the candidates of chunk b0 + t in registers, read
    // once a batch, and the batch is scanned again from the chunk after each stopping one.
    int it = 0;
    for (uint64_t b0 = 0; b0 < chunks; b0 += kSumThreads) {
        const uint64_t c = b0 + tid;
        int32_t cue[kCands];
        SumScan<T> cscan[kCands];
        const double csum = c < chunks ? chunk_sum[c] : 0.0;
#pragma unroll
        for (int y = 0; y < kCands; y++) {
            cue[y] = kNoPhase;
            cscan[y] = scan_identity<T>();
            if (c < chunks) {
                const ChunkSummary cs = summ[kCands * c + y];
                cue[y] = cs.ue;
                // Summary counts saturate at kCap, past any crossing: they fit C.
                cscan[y] = scan_of_summary<T>(cs);
            }
        }
        const uint64_t bend = b0 + kSumThreads < chunks ? b0 + kSumThreads : chunks;
        for (uint64_t c0 = b0; c0 < bend; it++) {
        const int slot = it & 1;
        SumScan<T> mine = scan_identity<T>();
        int cand = -1;
        if (c >= c0 && c < chunks) {
            // No summary for this binade: stop here.
            mine = SumScan<T>{kBig, kBig, 2u};
#pragma unroll
            for (int y = kCands - 1; y >= 0; y--)
                if (cue[y] == ue) {
                    cand = y;
                    mine = cscan[y];
                }
        }
        SumScan<T> before, total;
        block_scan<T>(mine, lane, wave, sh.wave_tot, before, total);
        const uint32_t p0 = (uint32_t)(m & 1u);
        const C mt = sat_add<T>(m, p0 ? before.r1 : before.r0);
        const uint32_t pt = p0 ? (before.p >> 1) & 1u : before.p & 1u;
        if (c >= c0 && c < chunks && mt < mmax && sat_add<T>(mt, pt ? mine.r1 : mine.r0) >= mmax) {
            sh.first[slot] = (uint32_t)tid;
            sh.m_first[slot] = (uint64_t)mt;
            sh.first_cand[slot] = cand;
            sh.mean[slot] = csum / (double)(c + 1 < chunks ? L : limit - c * L);
        }
        __syncthreads();
        const uint32_t first = sh.first[slot];
        const C m_first = (C)sh.m_first[slot];
        const int first_cand = sh.first_cand[slot];
        const double mean = sh.mean[slot];
        if (tid == 0)
            sh.first[slot ^ 1] = kNoStep;
        if (first == kNoStep) {
            m = sat_add<T>(m, p0 ? total.r1 : total.r0);
            c0 = bend;
            continue;
        }
        // Chunks before the stopping one fold; it runs exactly from the count before it: from
        // its run prefixes when it has a summary for this binade and the next binade is not
        // expected to end in the chunk's dense part too, and with the staged squares from
        // wherever that leaves off.
        m = m_first;
        const uint64_t cc = b0 + first;
        const uint64_t base = cc * L;
        const uint32_t len = (uint32_t)(base + L <= limit ? L : limit - base);
        uint32_t resume = 0;
        const bool dense = expected_gap((double)((C)1 << SumBits<T>::kFrac), ue + 1, mean) < kSerialGap;
        const int folded = first_cand < 0 || dense
                               ? -1
                               : run_prefix_chunk<T>(src, runs + kCands * cc * kSumThreads,
                                                     summ + kCands * cc, first_cand, base, len,
                                                     policy, fault, ue, m, mmax, resume, sh, gate);
        if (folded == 0)
            return;
        if (folded < 0) {
            U vals[SumBits<T>::kPer];
            load_chunk<T>(src, ((uintptr_t)src & 15u) == 0, base, base + len, tid, vals);
#pragma unroll
            for (uint32_t j = 0; j < (uint32_t)SumBits<T>::kPer; j++)
                sh.vals[ChunkLds<T>::slot(tid * SumBits<T>::kPer + j)] = vals[j];
            if (!exact_chunk<T>(base, len, resume, mean, policy, fault, ue, m, mmax, sh, gate))
                return;
        }
        c0 = cc + 1;
        }
    }
    if (limit < n || tid != 0)
        return;
    const T total = from_bits<T>(sum_bits<T>(ue, m));
    const T r = total / count;
    const uint32_t kind = classify_div(total, count, r, policy);
    if (kind != kOk) {
        atomicMin(fault, (unsigned long long)pack_fault(3 * n, kind));
        gate_record(gate);
    } else {
        *out = r;
    }
}

// A call of its own ends its program in this kernel (close).
template <typename T>
__global__ __launch_bounds__(kSumThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_mse_ordered_walk(
    const T *__restrict__ sq, uint64_t n, T count, int policy, T *__restrict__ out,
    unsigned long long *fault, const double *__restrict__ chunk_sum,
    const ChunkSummary *__restrict__ summ, const SumScan<T> *__restrict__ runs, NodeGate gate,
    ProgramClose close)
{
    ordered_walk<T>(sq, n, count, policy, out, fault, chunk_sum, summ, runs, gate);
    program_close_block(close);
}

// Inputs of at most kMseSerialMax elements, one workgroup. Its four waves form every difference and
// square in parallel into LDS (all of a thread's loads are issued before it computes) and find the
// first faulting Subtract or Multiply; then one wave folds the squares before that element in order,
// a chunk of 60 (binary64 30) at a time, every lane holding the chunk in registers and the next
// chunk's LDS reads in flight. A sum can only fault as in fold_run, so a chunk is folded with plain
// adds (REJECT_SUB: each partial total is kept and checked after) and again exactly only when that
// trips. The same results and first fault as below. What bounds it is the chain of adds, about
// 4.4 ns each and no barrier among them; the kernel of one chunk below pays some 250 ns more for 64
// of them and 2 us a window: whole calls, this one against that, binary32 300 squares 15.1 / 17.1 us,
// 512 16.2 / 18.6, 1024 18.9 / 21.7, 2000 23.6 / 24.2, 4096 45 / 42; binary64 512 18.0 / 20.2, 1024
// 21.4 / 23.9.
template <typename T, bool REJECT_SUB>
__device__ __forceinline__ void mse_serial(const T *__restrict__ p, const T *__restrict__ t, uint64_t n,
                                           T count, int policy, T *__restrict__ out,
                                           unsigned long long *fault, const NodeGate &gate)
{
    if (block_gate_closed(gate))
        return;
    constexpr int P = 16 / sizeof(T);              // squares per 16-byte LDS read
    constexpr int R = (int)(kMseSerialMax / 256);  // elements a thread
    __shared__ __align__(16) T sq[kMseSerialMax];
    __shared__ unsigned long long first_sm; // earliest Subtract or Multiply fault word
    const int tid = threadIdx.x;
    if (tid == 0)
        first_sm = kNoFault;
    T pv[R], tv[R];
#pragma unroll
    for (int j = 0; j < R; j++) {
        const uint64_t i = (uint64_t)tid + 256u * (uint64_t)j;
        if (i < n) {
            pv[j] = p[i];
            tv[j] = t[i];
        }
    }
    __syncthreads();
    uint64_t key = kNoFault;
    bool any = false; // a square other than +0
#pragma unroll
    for (int j = 0; j < R; j++) {
        const uint64_t i = (uint64_t)tid + 256u * (uint64_t)j;
        if (i < n) {
            const T d = pv[j] - tv[j];
            const T s = d * d;
            sq[i] = s;
            any |= !is_zero(s);
            if (key == kNoFault) {
                const uint32_t ks = classify_add(pv[j], tv[j], d, policy);
                if (ks != kOk) {
                    key = pack_fault(3 * i, ks);
                } else {
                    const uint32_t km = classify_mul(d, d, s, policy);
                    if (km != kOk)
                        key = pack_fault(3 * i + 1, km);
                }
            }
        }
    }
    if (key != kNoFault)
        atomicMin(&first_sm, (unsigned long long)key);
    any = __syncthreads_or(any);
    if (tid >= 64)
        return;
    const unsigned long long fsm = first_sm;
    // Elements summed; squares that are all +0 leave the total at +0.
    const uint64_t limit = fsm != kNoFault ? ((fsm >> 3) / 3) : (any ? n : 0);
    T total = (T)0;
    // The exact pass over squares i0 .. i0 + here - 1 from `total`: false when an Add faults
    // (recorded).
    auto exact = [&](uint64_t i0, uint32_t here) {
        bool ok = true;
        if (tid == 0)
            ok = fold_exact<T>(total, here, i0, policy, fault, gate, [&](uint32_t i) { return sq[i0 + i]; });
        return __ballot(!ok) == 0;
    };
    // A chunk is 15 LDS reads: with the next chunk's 15 reads issued before its adds, the wait for
    // this chunk (in-order LDS counter, at most 15 outstanding) leaves all of them in flight.
    constexpr int CH = 15 * P;
    auto load = [&](T (&v)[CH], uint64_t i0) {
#pragma unroll
        for (int q = 0; q < CH / P; q++)
            *reinterpret_cast<uint4 *>(&v[P * q]) = *reinterpret_cast<const uint4 *>(&sq[i0 + P * q]);
    };
    // Folds a whole chunk held in v; false when an Add faults (recorded).
    auto fold = [&](T (&v)[CH], uint64_t i0) __attribute__((always_inline)) {
        T sum = total;
        bool trip = false;
        if constexpr (!REJECT_SUB) {
#pragma unroll
            for (int j = 0; j < CH; j++)
                sum = sum + v[j];
        } else {
#pragma unroll
            for (int j = 0; j < CH; j++) {
                sum = sum + v[j];
                v[j] = sum;
            }
#pragma unroll
            for (int j = 0; j < CH; j++)
                trip |= subnormal(v[j]);
        }
        if ((!finite_bits(sum) || trip) && !exact(i0, CH))
            return false;
        total = sum;
        return true;
    };
    const uint64_t full = limit / CH * CH;
    T va[CH], vb[CH];
    if (full > 0)
        load(va, 0);
    for (uint64_t i0 = 0; i0 < full; i0 += 2 * CH) {
        const bool second = i0 + CH < full;
        if (second)
            load(vb, i0 + CH);
        if (!fold(va, i0))
            return;
        if (!second)
            break;
        if (i0 + 2 * CH < full)
            load(va, i0 + 2 * CH);
        if (!fold(vb, i0 + CH))
            return;
    }
    if (limit > full) {
        const uint32_t here = (uint32_t)(limit - full);
        T sum = total;
        bool trip = false;
        for (uint32_t j = 0; j < here; j++) {
            sum = sum + sq[full + j];
            trip |= REJECT_SUB && subnormal(sum);
        }
        if ((!finite_bits(sum) || trip) && !exact(full, here))
            return;
        total = sum;
    }
    if (tid != 0)
        return;
    const T r = total / count;
    const uint32_t kind = fsm != kNoFault ? kOk : classify_div(total, count, r, policy);
    if (fsm != kNoFault || kind != kOk) {
        atomicMin(fault, fsm != kNoFault ? fsm : (unsigned long long)pack_fault(3 * n, kind));
        gate_record(gate);
    } else {
        *out = r;
    }
}

template <typename T, bool REJECT_SUB>
__global__ __launch_bounds__(256) void k_mse_serial(const T *__restrict__ p, const T *__restrict__ t, uint64_t n,
                                                    T count, int policy, T *__restrict__ out,
                                                    unsigned long long *fault, NodeGate gate,
                                                    ProgramClose close)
{
    mse_serial<T, REJECT_SUB>(p, t, n, count, policy, out, fault, gate);
    program_close_block(close);
}

// Inputs of one chunk, one workgroup. Its waves form every difference and square in parallel into
// LDS (each thread issues all of its loads before it computes, so the inputs arrive in one round
// trip), find the first faulting Subtract or Multiply and estimate the mean; then the squares
// before that element fold as a chunk of the pipeline above does, from +0. The same results and
// first fault, in one launch and no scratch. What bounds it is the chain of phases: 512 or so
// dependent adds, then a window for each doubling of the total: 17 us at 4096 f32, where one wave
// adding all of the squares took 22.7.
template <typename T>
__device__ __forceinline__ void mse_one(const T *__restrict__ p, const T *__restrict__ t, uint64_t n,
                                        T count, int policy, T *__restrict__ out,
                                        unsigned long long *fault, const NodeGate &gate)
{
    if (block_gate_closed(gate))
        return;
    using U = typename SumBits<T>::U;
    using C = typename SumBits<T>::C;
    constexpr int P = SumBits<T>::kPer;
    __shared__ WalkShared<T> sh;
    __shared__ unsigned long long first_sm; // earliest Subtract or Multiply fault word
    __shared__ double part[kSumThreads / 64];
    const int tid = threadIdx.x;
    if (tid == 0)
        first_sm = kNoFault;
    T pv[P], tv[P];
#pragma unroll
    for (int j = 0; j < P; j++) {
        const uint64_t i = (uint64_t)tid + (uint64_t)(kSumThreads * j);
        if (i < n) {
            pv[j] = p[i];
            tv[j] = t[i];
        }
    }
    __syncthreads();
    uint64_t key = kNoFault;
    double acc = 0.0;
#pragma unroll
    for (int j = 0; j < P; j++) {
        const uint64_t i = (uint64_t)tid + (uint64_t)(kSumThreads * j);
        if (i < n) {
            const T d = pv[j] - tv[j];
            const T s = d * d;
            sh.vals[ChunkLds<T>::slot((uint32_t)i)] = (U)bits_of(s);
            acc += finite_bits(s) ? (double)s : 0.0;
            if (key == kNoFault) {
                const uint32_t ks = classify_add(pv[j], tv[j], d, policy);
                if (ks != kOk) {
                    key = pack_fault(3 * i, ks);
                } else {
                    const uint32_t km = classify_mul(d, d, s, policy);
                    if (km != kOk)
                        key = pack_fault(3 * i + 1, km);
                }
            }
        }
    }
    if (key != kNoFault)
        atomicMin(&first_sm, (unsigned long long)key);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        acc += __shfl_xor(acc, off, 64);
    if ((tid & 63) == 0)
        part[tid >> 6] = acc;
    __syncthreads();
    const unsigned long long fsm = first_sm;
    const uint64_t limit = fsm == kNoFault ? n : ((fsm >> 3) / 3); // elements summed
    double sum = 0.0;
#pragma unroll
    for (int w = 0; w < kSumThreads / 64; w++)
        sum += part[w];
    int ue;
    C m, mmax;
    sum_phase<T>((U)0, ue, m, mmax); // the total starts at +0
    if (!exact_chunk<T>(0, (uint32_t)limit, 0, sum / (double)n, policy, fault, ue, m, mmax, sh, gate))
        return;
    if (tid != 0)
        return;
    const T total = from_bits<T>(sum_bits<T>(ue, m));
    const T r = total / count;
    const uint32_t kind = fsm != kNoFault ? kOk : classify_div(total, count, r, policy);
    if (fsm != kNoFault || kind != kOk) {
        atomicMin(fault, fsm != kNoFault ? fsm : (unsigned long long)pack_fault(3 * n, kind));
        gate_record(gate);
    } else {
        *out = r;
    }
}

template <typename T>
__global__ __launch_bounds__(kSumThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_mse_one(
    const T *__restrict__ p, const T *__restrict__ t, uint64_t n, T count, int policy,
    T *__restrict__ out, unsigned long long *fault, NodeGate gate, ProgramClose close)
{
    mse_one<T>(p, t, n, count, policy, out, fault, gate);
    program_close_block(close);
}

// ------------------------------------------------------------- native compounds
// Explicitly permitted native compound arithmetic (Boundary + BackendDefined): no fault is
// classified; special values and subnormals flow through as the hardware produces them.

// SGD (backends/rocm/tensor/native_sgd/native_sgd.rs:100-145): the product rounded before
// the subtraction, or one fused multiply-add when contraction is permitted.
template <typename T, bool VEC, bool CONTRACT>
__global__ __launch_bounds__(kEwThreads) void k_native_sgd(const T *w,
                                                           const T *g, T rate,
                                                           T *out, uint64_t n, NodeGate gate)
{
    if (wave_gate_closed(gate))
        return;
    constexpr int W = Lanes<T, VEC>::W;
    PCU_EW_LOOP(W)
    {
        T wv[W], gv[W], r[W];
        load_lanes<T, VEC>(w, base, n, wv);
        load_lanes<T, VEC>(g, base, n, gv);
#pragma unroll
        for (int j = 0; j < W; j++) {
            if (CONTRACT) {
                r[j] = fma(-rate, gv[j], wv[j]);
            } else {
                const T p = rate * gv[j];
                r[j] = wv[j] - p;
            }
        }
        store_lanes<T, VEC>(out, base, n, r);
    }
}

// MSE (backends/rocm/tensor/native_loss/native_loss.rs, tensor.rs:5020-5070): rounded
// difference and square, a sum in the declared precision, times the rounded reciprocal
// count. The sum is a fixed-shape tree (per thread, wave, block, then over the blocks), so
// it repeats bit for bit from run to run.
template <typename T>
__device__ __forceinline__ T block_tree_sum(T v, T *part)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        v = v + __shfl_xor(v, off, 64);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
        part[wave] = v;
    __syncthreads();
    T total = (T)0;
    for (int w = 0; w < (int)(blockDim.x >> 6); w++)
        total = total + part[w];
    return total;
}

template <typename T, bool VEC>
__global__ __launch_bounds__(kEwThreads) void k_native_mse_partial(const T *__restrict__ p,
                                                                   const T *__restrict__ t,
                                                                   T *__restrict__ partial,
                                                                   uint64_t n, NodeGate gate)
{
    if (block_gate_closed(gate))
        return;
    __shared__ T part[kEwThreads / 64];
    constexpr int W = Lanes<T, VEC>::W;
    T acc = (T)0;
    PCU_EW_LOOP(W)
    {
        T pv[W], tv[W];
        load_lanes<T, VEC>(p, base, n, pv);
        load_lanes<T, VEC>(t, base, n, tv);
        T local = (T)0;
#pragma unroll
        for (int j = 0; j < W; j++) {
            const T d = pv[j] - tv[j];
            const T sq = d * d;
            local = local + (base + j < n ? sq : (T)0);
        }
        acc = acc + local;
    }
    const T total = block_tree_sum(acc, part);
    if (threadIdx.x == 0)
        partial[blockIdx.x] = total;
}

template <typename T>
__global__ __launch_bounds__(1024) void k_native_mse_final(const T *__restrict__ partial,
                                                           uint64_t blocks, T scale,
                                                           T *__restrict__ out, NodeGate gate)
{
    if (block_gate_closed(gate))
        return;
    __shared__ T part[16];
    T acc = (T)0;
    for (uint64_t i = threadIdx.x; i < blocks; i += 1024)
        acc = acc + partial[i];
    const T total = block_tree_sum(acc, part);
    if (threadIdx.x == 0)
        *out = total * scale;
}

// ================================================================ launchers

static inline bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

static inline unsigned grid_for(uint64_t work_items)
{
    // One work item per thread; beyond 2^24 blocks the kernels' loops take the rest.
    uint64_t blocks = (work_items + kEwThreads - 1) / kEwThreads;
    if (blocks > (1ull << 24))
        blocks = 1ull << 24;
    return blocks ? (unsigned)blocks : 1u;
}

template <typename T>
static hipError_t binary_t(hipStream_t s, int op, uint64_t n, const void *a, const void *b,
                           const void *b_value, void *out, int policy, unsigned long long *fault, NodeGate gate)
{
    const T *A = (const T *)a, *B = (const T *)b;
    T bv = b_value ? *(const T *)b_value : (T)0;
    bool uniform = b == nullptr;
    constexpr int Wd = Vec<T>::width;
    bool vec = aligned16(a) && aligned16(out) && (uniform || aligned16(b));
    unsigned grid = grid_for(vec ? (n + Wd - 1) / Wd : n);
#define PCU_LAUNCH_BINARY(OPC)                                                                      \
    if (uniform) {                                                                                  \
        if (vec) hipLaunchKernelGGL((k_binary<T, OPC, true, true>), dim3(grid), dim3(kEwThreads), 0, s, A, B, bv, (T *)out, n, policy, fault, gate); \
        else hipLaunchKernelGGL((k_binary<T, OPC, true, false>), dim3(grid), dim3(kEwThreads), 0, s, A, B, bv, (T *)out, n, policy, fault, gate); \
    } else {                                                                                        \
        if (vec) hipLaunchKernelGGL((k_binary<T, OPC, false, true>), dim3(grid), dim3(kEwThreads), 0, s, A, B, bv, (T *)out, n, policy, fault, gate); \
        else hipLaunchKernelGGL((k_binary<T, OPC, false, false>), dim3(grid), dim3(kEwThreads), 0, s, A, B, bv, (T *)out, n, policy, fault, gate); \
    }
    switch (op) {
    case kOpAdd: PCU_LAUNCH_BINARY(kOpAdd) break;
    case kOpSub: PCU_LAUNCH_BINARY(kOpSub) break;
    case kOpMul: PCU_LAUNCH_BINARY(kOpMul) break;
    default: PCU_LAUNCH_BINARY(kOpDiv) break;
    }
#undef PCU_LAUNCH_BINARY
    return hipGetLastError();
}

hipError_t launch_binary(hipStream_t s, int dtype, int op, uint64_t n, const void *a,
                         const void *b, const void *b_value, void *out, int policy,
                         unsigned long long *fault, NodeGate gate)
{
    if (n == 0)
        return hipSuccess;
    return dtype == 0 ? binary_t<float>(s, op, n, a, b, b_value, out, policy, fault, gate)
                      : binary_t<double>(s, op, n, a, b, b_value, out, policy, fault, gate);
}

template <typename T>
static hipError_t relu_t(hipStream_t s, uint64_t n, const void *x, void *out, int policy,
                         unsigned long long *fault, NodeGate gate)
{
    constexpr int Wd = Vec<T>::width;
    bool vec = aligned16(x) && aligned16(out);
    unsigned grid = grid_for(vec ? (n + Wd - 1) / Wd : n);
    if (vec)
        hipLaunchKernelGGL((k_relu<T, true>), dim3(grid), dim3(kEwThreads), 0, s, (const T *)x, (T *)out, n, policy, fault, gate);
    else
        hipLaunchKernelGGL((k_relu<T, false>), dim3(grid), dim3(kEwThreads), 0, s, (const T *)x, (T *)out, n, policy, fault, gate);
    return hipGetLastError();
}

template <typename T>
static hipError_t chain_t(hipStream_t s, uint64_t n, const ChainLaunch &c, NodeGate gate)
{
    constexpr int Wd = Vec<T>::width;
    bool vec = aligned16(c.head);
    for (int i = 0; i < c.steps; i++)
        vec = vec && aligned16(c.step[i].other) && aligned16(c.step[i].out);
    const unsigned grid = grid_for(vec ? (n + Wd - 1) / Wd : n);
    int sig = 0;
    for (int i = 0; i < c.steps && i < kChainMaxSteps; i++)
        sig |= c.step[i].op << (4 * i);
    const int key = c.steps * 2 + (vec ? 1 : 0);
    if (c.steps == 2 && sig == kSigSubMul) {
        if (vec) hipLaunchKernelGGL((k_chain<T, true, 2, kSigSubMul>), dim3(grid), dim3(kEwThreads), 0, s, c, n, gate);
        else hipLaunchKernelGGL((k_chain<T, false, 2, kSigSubMul>), dim3(grid), dim3(kEwThreads), 0, s, c, n, gate);
        return hipGetLastError();
    }
    if (c.steps == 2 && sig == kSigAddRelu) {
        if (vec) hipLaunchKernelGGL((k_chain<T, true, 2, kSigAddRelu>), dim3(grid), dim3(kEwThreads), 0, s, c, n, gate);
        else hipLaunchKernelGGL((k_chain<T, false, 2, kSigAddRelu>), dim3(grid), dim3(kEwThreads), 0, s, c, n, gate);
        return hipGetLastError();
    }
    if (c.steps == 3 && sig == kSigSubMulReluBack) {
        if (vec) hipLaunchKernelGGL((k_chain<T, true, 3, kSigSubMulReluBack>), dim3(grid), dim3(kEwThreads), 0, s, c, n, gate);
        else hipLaunchKernelGGL((k_chain<T, false, 3, kSigSubMulReluBack>), dim3(grid), dim3(kEwThreads), 0, s, c, n, gate);
        return hipGetLastError();
    }
    switch (key) {
    case 3: hipLaunchKernelGGL((k_chain<T, true, 1>), dim3(grid), dim3(kEwThreads), 0, s, c, n, gate); break;
    case 2: hipLaunchKernelGGL((k_chain<T, false, 1>), dim3(grid), dim3(kEwThreads), 0, s, c, n, gate); break;
    case 5: hipLaunchKernelGGL((k_chain<T, true, 2>), dim3(grid), dim3(kEwThreads), 0, s, c, n, gate); break;
    case 4: hipLaunchKernelGGL((k_chain<T, false, 2>), dim3(grid), dim3(kEwThreads), 0, s, c, n, gate); break;
    case 7: hipLaunchKernelGGL((k_chain<T, true, 3>), dim3(grid), dim3(kEwThreads), 0, s, c, n, gate); break;
    case 6: hipLaunchKernelGGL((k_chain<T, false, 3>), dim3(grid), dim3(kEwThreads), 0, s, c, n, gate); break;
    case 9: hipLaunchKernelGGL((k_chain<T, true, 4>), dim3(grid), dim3(kEwThreads), 0, s, c, n, gate); break;
    case 8: hipLaunchKernelGGL((k_chain<T, false, 4>), dim3(grid), dim3(kEwThreads), 0, s, c, n, gate); break;
    default: return hipErrorInvalidValue; // a chain has 1 to 4 steps
    }
    return hipGetLastError();
}

hipError_t launch_chain(hipStream_t s, int dtype, uint64_t n, const ChainLaunch &c, NodeGate gate)
{
    if (n == 0 || c.steps <= 0)
        return hipSuccess;
    return dtype == 0 ? chain_t<float>(s, n, c, gate) : chain_t<double>(s, n, c, gate);
}

hipError_t launch_relu(hipStream_t s, int dtype, uint64_t n, const void *x, void *out,
                       int policy, unsigned long long *fault, NodeGate gate)
{
    if (n == 0)
        return hipSuccess;
    return dtype == 0 ? relu_t<float>(s, n, x, out, policy, fault, gate)
                      : relu_t<double>(s, n, x, out, policy, fault, gate);
}

template <typename T>
static hipError_t relu_backward_t(hipStream_t s, uint64_t n, const void *x, const void *up,
                                  void *out, int policy, unsigned long long *fault, NodeGate gate)
{
    constexpr int Wd = Vec<T>::width;
    bool vec = aligned16(x) && aligned16(up) && aligned16(out);
    unsigned grid = grid_for(vec ? (n + Wd - 1) / Wd : n);
    if (vec)
        hipLaunchKernelGGL((k_relu_backward<T, true>), dim3(grid), dim3(kEwThreads), 0, s, (const T *)x, (const T *)up, (T *)out, n, policy, fault, gate);
    else
        hipLaunchKernelGGL((k_relu_backward<T, false>), dim3(grid), dim3(kEwThreads), 0, s, (const T *)x, (const T *)up, (T *)out, n, policy, fault, gate);
    return hipGetLastError();
}

hipError_t launch_relu_backward(hipStream_t s, int dtype, uint64_t n, const void *x,
                                const void *up, void *out, int policy,
                                unsigned long long *fault, NodeGate gate)
{
    if (n == 0)
        return hipSuccess;
    return dtype == 0 ? relu_backward_t<float>(s, n, x, up, out, policy, fault, gate)
                      : relu_backward_t<double>(s, n, x, up, out, policy, fault, gate);
}

template <typename T>
static hipError_t add_relu_t(hipStream_t s, uint64_t n, const void *a, const void *b,
                             const void *b_value, void *out, int policy,
                             unsigned long long *fault_add, unsigned long long *fault_relu, NodeGate gate)
{
    const T *A = (const T *)a, *B = (const T *)b;
    T bv = b_value ? *(const T *)b_value : (T)0;
    bool uniform = b == nullptr;
    constexpr int Wd = Vec<T>::width;
    bool vec = aligned16(a) && aligned16(out) && (uniform || aligned16(b));
    unsigned grid = grid_for(vec ? (n + Wd - 1) / Wd : n);
    if (uniform) {
        if (vec) hipLaunchKernelGGL((k_add_relu<T, true, true>), dim3(grid), dim3(kEwThreads), 0, s, A, B, bv, (T *)out, n, policy, fault_add, fault_relu, gate);
        else hipLaunchKernelGGL((k_add_relu<T, true, false>), dim3(grid), dim3(kEwThreads), 0, s, A, B, bv, (T *)out, n, policy, fault_add, fault_relu, gate);
    } else {
        if (vec) hipLaunchKernelGGL((k_add_relu<T, false, true>), dim3(grid), dim3(kEwThreads), 0, s, A, B, bv, (T *)out, n, policy, fault_add, fault_relu, gate);
        else hipLaunchKernelGGL((k_add_relu<T, false, false>), dim3(grid), dim3(kEwThreads), 0, s, A, B, bv, (T *)out, n, policy, fault_add, fault_relu, gate);
    }
    return hipGetLastError();
}

hipError_t launch_add_relu(hipStream_t s, int dtype, uint64_t n, const void *a, const void *b,
                           const void *b_value, void *out, int policy,
                           unsigned long long *fault_add, unsigned long long *fault_relu, NodeGate gate)
{
    if (n == 0)
        return hipSuccess;
    return dtype == 0 ? add_relu_t<float>(s, n, a, b, b_value, out, policy, fault_add, fault_relu, gate)
                      : add_relu_t<double>(s, n, a, b, b_value, out, policy, fault_add, fault_relu, gate);
}

// An SGD launch ends its program (ProgramClose) only on a grid of at most kCloseMaxBlocks
// workgroups: every workgroup takes one ticket on a single counter at its end, and the
// tickets queue behind one another (1024 of them made a 2^20-element update 15 -> 24 us).

template <typename T>
static hipError_t sgd_t(hipStream_t s, uint64_t n, const void *w, const void *g, T rate,
                        void *out, int policy, unsigned long long *fault, NodeGate gate,
                        ProgramClose close, bool *closed)
{
    constexpr int Wd = Vec<T>::width;
    bool vec = aligned16(w) && aligned16(g) && aligned16(out);
    unsigned grid = grid_for(vec ? (n + Wd - 1) / Wd : n);
    if (grid > kCloseMaxBlocks)
        close = ProgramClose{};
    if (closed)
        *closed = close.words != nullptr;
    if (vec)
        hipLaunchKernelGGL((k_sgd<T, true>), dim3(grid), dim3(kEwThreads), 0, s, (const T *)w, (const T *)g, rate, (T *)out, n, policy, fault, gate, close);
    else
        hipLaunchKernelGGL((k_sgd<T, false>), dim3(grid), dim3(kEwThreads), 0, s, (const T *)w, (const T *)g, rate, (T *)out, n, policy, fault, gate, close);
    return hipGetLastError();
}

hipError_t launch_sgd(hipStream_t s, int dtype, uint64_t n, const void *w, const void *g,
                      double rate, void *out, int policy, unsigned long long *fault, NodeGate gate,
                      ProgramClose close, bool *closed)
{
    if (closed)
        *closed = false;
    if (n == 0)
        return hipSuccess;
    return dtype == 0 ? sgd_t<float>(s, n, w, g, (float)rate, out, policy, fault, gate, close, closed)
                      : sgd_t<double>(s, n, w, g, rate, out, policy, fault, gate, close, closed);
}

template <typename T>
static hipError_t sgd_pair_t(hipStream_t s, const SgdJob &j0, const SgdJob &j1, int policy,
                             ProgramClose close, bool *closed)
{
    constexpr int Wd = Vec<T>::width;
    const SgdJob *j[2] = {&j0, &j1};
    bool vec = true;
    for (int u = 0; u < 2; u++)
        vec = vec && aligned16(j[u]->w) && aligned16(j[u]->g) && aligned16(j[u]->out);
    SgdPairArgs<T> a;
    unsigned blocks[2];
    for (int u = 0; u < 2; u++) {
        a.w[u] = (const T *)j[u]->w;
        a.g[u] = (const T *)j[u]->g;
        a.out[u] = (T *)j[u]->out;
        a.rate[u] = (T)j[u]->rate;
        a.n[u] = j[u]->n;
        a.fault[u] = j[u]->fault;
        a.gate[u] = j[u]->gate;
        // grid_for caps each at 2^24 blocks, so the sum fits a launch.
        blocks[u] = grid_for(vec ? (j[u]->n + Wd - 1) / Wd : j[u]->n);
    }
    a.blocks0 = blocks[0];
    const dim3 grid(blocks[0] + blocks[1]);
    if (grid.x > kCloseMaxBlocks)
        close = ProgramClose{};
    if (closed)
        *closed = close.words != nullptr;
    if (vec)
        hipLaunchKernelGGL((k_sgd_pair<T, true>), grid, dim3(kEwThreads), 0, s, a, policy, close);
    else
        hipLaunchKernelGGL((k_sgd_pair<T, false>), grid, dim3(kEwThreads), 0, s, a, policy, close);
    return hipGetLastError();
}

hipError_t launch_sgd_pair(hipStream_t s, int dtype, const SgdJob &j0, const SgdJob &j1, int policy,
                           ProgramClose close, bool *closed)
{
    if (closed)
        *closed = false;
    if (j0.n == 0 || j1.n == 0)
        return hipErrorInvalidValue;
    return dtype == 0 ? sgd_pair_t<float>(s, j0, j1, policy, close, closed)
                      : sgd_pair_t<double>(s, j0, j1, policy, close, closed);
}

// Scratch of one MSE call: the squares, then the quarter and chunk sums and the summaries.
static inline size_t round256(size_t b) { return (b + 255) & ~(size_t)255; }

template <typename T>
static size_t mse_chunks(uint64_t n)
{
    const uint64_t L = (uint64_t)kSumThreads * SumBits<T>::kPer;
    return (size_t)((n + L - 1) / L);
}

size_t mse_scratch_bytes(int dtype, uint64_t n)
{
    const size_t es = dtype == 0 ? 4 : 8;
    const size_t chunks = dtype == 0 ? mse_chunks<float>(n) : mse_chunks<double>(n);
    const size_t run_bytes = dtype == 0 ? sizeof(SumScan<float>) : sizeof(SumScan<double>);
    return round256(n * es) + round256(kQuarters * chunks * sizeof(double)) +
           2 * round256(chunks * sizeof(double)) +
           round256(kCands * chunks * sizeof(ChunkSummary)) +
           round256(kCands * chunks * kSumThreads * run_bytes);
}

template <typename T> struct MseScratch {
    T *squares;
    double *quarter_sum, *chunk_sum, *chunk_pre;
    ChunkSummary *summ;
    SumScan<T> *runs;
    size_t chunks;
    MseScratch(void *scratch, uint64_t n)
    {
        char *base = (char *)scratch;
        chunks = mse_chunks<T>(n);
        squares = (T *)base;
        quarter_sum = (double *)(base + round256(n * sizeof(T)));
        chunk_sum = (double *)((char *)quarter_sum + round256(kQuarters * chunks * sizeof(double)));
        chunk_pre = (double *)((char *)chunk_sum + round256(chunks * sizeof(double)));
        summ = (ChunkSummary *)((char *)chunk_pre + round256(chunks * sizeof(double)));
        runs = (SumScan<T> *)((char *)summ + round256(kCands * chunks * sizeof(ChunkSummary)));
    }
};

template <typename T>
static hipError_t mse_prepare_t(hipStream_t s, uint64_t n, const void *p, const void *t,
                                void *scratch, int policy, unsigned long long *fault, NodeGate gate)
{
    const MseScratch<T> m(scratch, n);
    const bool vec = aligned16(p) && aligned16(t) && aligned16(m.squares);
    const unsigned grid = (unsigned)(kQuarters * m.chunks);
    if (vec)
        hipLaunchKernelGGL((k_mse_squares<T, true>), dim3(grid), dim3(kEwThreads), 0, s, (const T *)p, (const T *)t, m.squares, n, policy, m.quarter_sum, fault, gate);
    else
        hipLaunchKernelGGL((k_mse_squares<T, false>), dim3(grid), dim3(kEwThreads), 0, s, (const T *)p, (const T *)t, m.squares, n, policy, m.quarter_sum, fault, gate);
    const bool prefix = m.chunks > kSumThreads;
    if (prefix)
        hipLaunchKernelGGL(k_mse_chunk_prefix, dim3(1), dim3(kPrefixThreads), 0, s, (const double *)m.quarter_sum, (uint64_t)m.chunks, m.chunk_sum, m.chunk_pre, gate);
    hipLaunchKernelGGL((k_mse_chunk_summaries<T>), dim3((unsigned)m.chunks, kCands), dim3(kSumThreads), 0, s, (const T *)m.squares, n, (const unsigned long long *)fault, (const double *)m.quarter_sum, m.chunk_sum, prefix ? (const double *)m.chunk_pre : nullptr, m.summ, m.runs, gate);
    return hipGetLastError();
}

template <typename T>
static hipError_t mse_walk_t(hipStream_t s, uint64_t n, void *scratch, T count, void *out,
                             int policy, unsigned long long *fault, NodeGate gate, ProgramClose close)
{
    const MseScratch<T> m(scratch, n);
    hipLaunchKernelGGL((k_mse_ordered_walk<T>), dim3(1), dim3(kSumThreads), 0, s, (const T *)m.squares, n, count, policy, (T *)out, fault, (const double *)m.chunk_sum, (const ChunkSummary *)m.summ, (const SumScan<T> *)m.runs, gate, close);
    return hipGetLastError();
}

hipError_t launch_mse_prepare(hipStream_t s, int dtype, uint64_t n, const void *p, const void *t,
                              void *scratch, int policy, unsigned long long *fault, NodeGate gate)
{
    if (n == 0)
        return hipErrorInvalidValue;
    return dtype == 0 ? mse_prepare_t<float>(s, n, p, t, scratch, policy, fault, gate)
                      : mse_prepare_t<double>(s, n, p, t, scratch, policy, fault, gate);
}

hipError_t launch_mse_walk(hipStream_t s, int dtype, uint64_t n, void *scratch, double count,
                           void *out, int policy, unsigned long long *fault, NodeGate gate,
                           ProgramClose close)
{
    if (n == 0)
        return hipErrorInvalidValue;
    return dtype == 0 ? mse_walk_t<float>(s, n, scratch, (float)count, out, policy, fault, gate, close)
                      : mse_walk_t<double>(s, n, scratch, count, out, policy, fault, gate, close);
}

uint64_t mse_one_max(int dtype)
{
    return (uint64_t)kSumThreads * (dtype == 0 ? SumBits<float>::kPer : SumBits<double>::kPer);
}

hipError_t launch_mse_one(hipStream_t s, int dtype, uint64_t n, const void *p, const void *t,
                          double count, void *out, int policy, unsigned long long *fault, NodeGate gate,
                          ProgramClose close)
{
    if (n == 0 || n > mse_one_max(dtype))
        return hipErrorInvalidValue;
    const bool reject = policy == kPolicyRejectSubnormal;
    if (n <= kMseSerialMax && dtype == 0 && reject)
        hipLaunchKernelGGL((k_mse_serial<float, true>), dim3(1), dim3(256), 0, s, (const float *)p, (const float *)t, n, (float)count, policy, (float *)out, fault, gate, close);
    else if (n <= kMseSerialMax && dtype == 0)
        hipLaunchKernelGGL((k_mse_serial<float, false>), dim3(1), dim3(256), 0, s, (const float *)p, (const float *)t, n, (float)count, policy, (float *)out, fault, gate, close);
    else if (n <= kMseSerialMax && reject)
        hipLaunchKernelGGL((k_mse_serial<double, true>), dim3(1), dim3(256), 0, s, (const double *)p, (const double *)t, n, count, policy, (double *)out, fault, gate, close);
    else if (n <= kMseSerialMax)
        hipLaunchKernelGGL((k_mse_serial<double, false>), dim3(1), dim3(256), 0, s, (const double *)p, (const double *)t, n, count, policy, (double *)out, fault, gate, close);
    else if (dtype == 0)
        hipLaunchKernelGGL((k_mse_one<float>), dim3(1), dim3(kSumThreads), 0, s, (const float *)p, (const float *)t, n, (float)count, policy, (float *)out, fault, gate, close);
    else
        hipLaunchKernelGGL((k_mse_one<double>), dim3(1), dim3(kSumThreads), 0, s, (const double *)p, (const double *)t, n, count, policy, (double *)out, fault, gate, close);
    return hipGetLastError();
}

// ------------------------------------------------------------ native launchers

template <typename T>
static hipError_t native_sgd_t(hipStream_t s, uint64_t n, const void *w, const void *g, T rate,
                               bool contracted, void *out, NodeGate gate)
{
    constexpr int Wd = Vec<T>::width;
    const bool vec = aligned16(w) && aligned16(g) && aligned16(out);
    const unsigned grid = grid_for(vec ? (n + Wd - 1) / Wd : n);
    const T *W = (const T *)w, *G = (const T *)g;
    T *O = (T *)out;
    if (vec && contracted) hipLaunchKernelGGL((k_native_sgd<T, true, true>), dim3(grid), dim3(kEwThreads), 0, s, W, G, rate, O, n, gate);
    else if (vec) hipLaunchKernelGGL((k_native_sgd<T, true, false>), dim3(grid), dim3(kEwThreads), 0, s, W, G, rate, O, n, gate);
    else if (contracted) hipLaunchKernelGGL((k_native_sgd<T, false, true>), dim3(grid), dim3(kEwThreads), 0, s, W, G, rate, O, n, gate);
    else hipLaunchKernelGGL((k_native_sgd<T, false, false>), dim3(grid), dim3(kEwThreads), 0, s, W, G, rate, O, n, gate);
    return hipGetLastError();
}

hipError_t launch_native_sgd(hipStream_t s, int dtype, uint64_t n, const void *w, const void *g,
                             double rate, bool contracted, void *out, NodeGate gate)
{
    if (n == 0)
        return hipSuccess;
    return dtype == 0 ? native_sgd_t<float>(s, n, w, g, (float)rate, contracted, out, gate)
                      : native_sgd_t<double>(s, n, w, g, rate, contracted, out, gate);
}

static uint64_t native_mse_blocks(int dtype, uint64_t n)
{
    const uint64_t w = dtype == 0 ? 4 : 2;
    return grid_for((n + w - 1) / w);
}

size_t native_mse_scratch_bytes(int dtype, uint64_t n)
{
    return (size_t)native_mse_blocks(dtype, n) * (dtype == 0 ? 4 : 8);
}

template <typename T>
static hipError_t native_mse_t(hipStream_t s, uint64_t n, const void *p, const void *t,
                               void *scratch, T scale, void *out, NodeGate gate)
{
    constexpr int Wd = Vec<T>::width;
    const bool vec = aligned16(p) && aligned16(t);
    const unsigned grid = grid_for(vec ? (n + Wd - 1) / Wd : n);
    if (vec)
        hipLaunchKernelGGL((k_native_mse_partial<T, true>), dim3(grid), dim3(kEwThreads), 0, s, (const T *)p, (const T *)t, (T *)scratch, n, gate);
    else
        hipLaunchKernelGGL((k_native_mse_partial<T, false>), dim3(grid), dim3(kEwThreads), 0, s, (const T *)p, (const T *)t, (T *)scratch, n, gate);
    hipLaunchKernelGGL((k_native_mse_final<T>), dim3(1), dim3(1024), 0, s, (const T *)scratch, (uint64_t)grid, scale, (T *)out, gate);
    return hipGetLastError();
}

hipError_t launch_native_mse(hipStream_t s, int dtype, uint64_t n, const void *p, const void *t,
                             void *scratch, double scale, void *out, NodeGate gate)
{
    if (n == 0)
        return hipErrorInvalidValue;
    return dtype == 0 ? native_mse_t<float>(s, n, p, t, scratch, (float)scale, out, gate)
                      : native_mse_t<double>(s, n, p, t, scratch, scale, out, gate);
}


// ------------------------------------------------------------ program end
// The fault words go to the host without a copy command: one workgroup copies them into
// coherent pinned memory, resets them (and opens the stage gate) for the next program, and
// then stores the program's sequence number, so the host waits on that one word instead of
// the stream.
__global__ __launch_bounds__(256) void k_program_publish(unsigned long long *words, uint64_t n,
                                                         unsigned long long value, unsigned int *gate,
                                                         unsigned long long *host_words,
                                                         unsigned long long *host_seq, uint64_t seq)
{
    for (uint64_t i = threadIdx.x; i < n; i += blockDim.x) {
        const unsigned long long w = words[i];
        __hip_atomic_store(&host_words[i], w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        words[i] = value;
    }
    if (threadIdx.x == 0)
        *gate = 0xffffffffu;
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0)
        __hip_atomic_store(host_seq, (unsigned long long)seq, __ATOMIC_RELEASE,
                           __HIP_MEMORY_SCOPE_SYSTEM);
}

hipError_t launch_program_publish(hipStream_t s, unsigned long long *words, uint64_t n,
                                  uint64_t value, unsigned int *gate,
                                  unsigned long long *host_words, unsigned long long *host_seq,
                                  uint64_t seq)
{
    hipLaunchKernelGGL(k_program_publish, dim3(1), dim3(256), 0, s, words, n,
                       (unsigned long long)value, gate, host_words, host_seq, seq);
    return hipGetLastError();
}

} // namespace pcu

