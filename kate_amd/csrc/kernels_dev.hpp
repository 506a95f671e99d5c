// kernels_dev.hpp -- device code shared by the kernel translation units
// (kernels.hip, pass_f64.hip, pass_f32.hip, batch_f64.hip, batch_f32.hip).
// Each unit instantiates only the templates it launches, so the pass and
// batch kernels of the two precisions compile in parallel.
//
// k_pass is the gate-group kernel: the replacement of Kate's
// executeGroupKernelSharedState + GPUGate::compute
// (HIPcode/simulator.hpp:143-218, HIPcode/GPUGate.hpp:21-203) and, with a
// permuted store, of its multi-GPU qubit swap (HIPcode/simulator.hpp:102-115).
// One workgroup owns one tile of 2^TB amplitudes:
//   1. load: 16 independent coalesced loads per thread (tile bits 0..TB-5
//      come from the thread index, so each wave reads whole runs of the
//      tile's low qubits) into an XOR-swizzled LDS tile;
//   2. micro-steps: each thread pulls the 16 amplitudes spanned by 4 tile
//      bits into registers, applies every gate of the step there (gate
//      coefficients are uniform, read through the scalar cache), writes them
//      back; one barrier per micro-step;
//   3. store: the same 16 coalesced runs, optionally to permuted positions.
// Complex arithmetic follows Kate's Complex class
// (backendagnosticcode/basic_host_types.hpp:43-45); the compiler may contract
// it into FMAs, so results agree with Kate's CPU path to rounding, not bits.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstdlib>

#include "kernels.hpp"

namespace kate {
namespace {

template <typename R>
struct alignas(2 * sizeof(R)) Cx {
    R re, im;
};

// Fused multiply-add written out: which product of an expression is fused
// is then fixed by the source, not by how the compiler contracts each
// inlined copy, so the direct and LDS paths of a step round identically.
template <typename R>
__device__ __forceinline__ R fmar(R a, R b, R c)
{
    if constexpr (sizeof(R) == 8) return __builtin_fma(a, b, c);
    else return __builtin_fmaf(a, b, c);
}

template <typename R>
__device__ __forceinline__ Cx<R> cmul(Cx<R> a, Cx<R> b)
{
    return Cx<R>{fmar(a.re, b.re, -(a.im * b.im)), fmar(a.re, b.im, a.im * b.re)};
}

template <typename R>
__device__ __forceinline__ Cx<R> cmac(Cx<R> acc, Cx<R> a, Cx<R> b)
{
    acc.re = fmar(-a.im, b.im, fmar(a.re, b.re, acc.re));
    acc.im = fmar(a.im, b.re, fmar(a.re, b.im, acc.im));
    return acc;
}

// XOR swizzle of the low W bits of an LDS element index with the next W bits,
// W = log2(elements per 256 B bank row): makes the 16-amplitude micro-step
// accesses of a wave land in distinct banks for every choice of tile bits
// inside the low 2W bits.
template <typename R>
__device__ __forceinline__ uint32_t swz(uint32_t j)
{
    constexpr uint32_t W = sizeof(R) == 8 ? 4 : 5;
    return j ^ ((j >> W) & ((1u << W) - 1u));
}

// Deterministic reductions: fixed butterfly within a wave, fixed order across waves.
__device__ __forceinline__ double wave_sum(double x)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off, 64);
    return x;
}

// Sum over the 256 threads of a block, fixed order; result valid in thread 0.
__device__ __forceinline__ double block_sum(double x, double* lds4)
{
    x = wave_sum(x);
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) lds4[w] = x;
    __syncthreads();
    return ((lds4[0] + lds4[1]) + (lds4[2] + lds4[3]));
}

// Deposit the low bits of s into the set bits of MASK (compile-time).
__host__ __device__ constexpr int dep(int mask, int s)
{
    int out = 0, k = 0;
    for (int b = 0; b < 4; b++)
        if ((mask >> b) & 1) {
            if ((s >> k) & 1) out |= 1 << b;
            k++;
        }
    return out;
}

__host__ __device__ constexpr int popc4(int m) { return (m & 1) + ((m >> 1) & 1) + ((m >> 2) & 1) + ((m >> 3) & 1); }

// ---- register ops on the N = 2^NB amplitudes of a micro-step --------------
//
// A micro-step holds N = 8 (NB = 3 micro bits) or N = 16 (NB = 4) amplitudes
// per thread; register index bit i is micro bit i.  Every op is a template
// on the array size, and apply_op instantiates only the codes whose bits
// exist for that size.

// Dense gate on the micro bits of MASK; matrix bit i <-> i-th lowest bit.
template <int MASK, typename R, int N>
__device__ __forceinline__ void op_dense(Cx<R> (&v)[N], const Cx<R>* __restrict__ m)
{
    constexpr int K = popc4(MASK);
    constexpr int D = 1 << K;
#pragma unroll
    for (int rest = 0; rest < N; rest++) {
        if (rest & MASK) continue;
        Cx<R> in[D];
#pragma unroll
        for (int s = 0; s < D; s++) in[s] = v[rest | dep(MASK, s)];
#pragma unroll
        for (int r = 0; r < D; r++) {
            Cx<R> acc = cmul(m[r * D], in[0]);
#pragma unroll
            for (int c = 1; c < D; c++) acc = cmac(acc, m[r * D + c], in[c]);
            v[rest | dep(MASK, r)] = acc;
        }
    }
}

template <int J, typename R, int N>
__device__ __forceinline__ void op_phase(Cx<R> (&v)[N], const Cx<R>* __restrict__ m)
{
    const Cx<R> d0 = m[0], d1 = m[1];
#pragma unroll
    for (int s = 0; s < N; s++) v[s] = cmul(((s >> J) & 1) ? d1 : d0, v[s]);
}

// Kate's Hadamard: a0' = (a0+a1)/sqrt2, a1' = a0' - a1*sqrt2 (GateComputing.hpp:77-78).
template <int J, typename R, int N>
__device__ __forceinline__ void op_h(Cx<R> (&v)[N])
{
    const R inv = (R)0.7071067811865475, s2 = (R)1.4142135623730951;
#pragma unroll
    for (int s = 0; s < N; s++) {
        if ((s >> J) & 1) continue;
        const Cx<R> a = v[s], b = v[s | (1 << J)];
        const Cx<R> n0{(a.re + b.re) * inv, (a.im + b.im) * inv};
        v[s] = n0;
        v[s | (1 << J)] = Cx<R>{fmar(-b.re, s2, n0.re), fmar(-b.im, s2, n0.im)};
    }
}

template <int T, int C, typename R, int N>
__device__ __forceinline__ void op_cnot(Cx<R> (&v)[N])
{
#pragma unroll
    for (int s = 0; s < N; s++) {
        if (((s >> C) & 1) == 0 || ((s >> T) & 1)) continue;
        const Cx<R> t = v[s];
        v[s] = v[s | (1 << T)];
        v[s | (1 << T)] = t;
    }
}

template <int A, int B, typename R, int N>
__device__ __forceinline__ void op_crk(Cx<R> (&v)[N], const Cx<R>* __restrict__ m)
{
    const Cx<R> ph = m[0];
#pragma unroll
    for (int s = 0; s < N; s++)
        if (((s >> A) & 1) && ((s >> B) & 1)) v[s] = cmul(v[s], ph);
}

template <int T, int C0, int C1, typename R, int N>
__device__ __forceinline__ void op_toff(Cx<R> (&v)[N])
{
#pragma unroll
    for (int s = 0; s < N; s++) {
        if (((s >> C0) & 1) == 0 || ((s >> C1) & 1) == 0 || ((s >> T) & 1)) continue;
        const Cx<R> t = v[s];
        v[s] = v[s | (1 << T)];
        v[s | (1 << T)] = t;
    }
}

// Independent 2x2 gates on every micro bit of MASK (one matrix per bit, in
// ascending bit order), applied one after the other.
template <int MASK, typename R, int N>
__device__ __forceinline__ void op_kron(Cx<R> (&v)[N], const Cx<R>* __restrict__ m)
{
    int k = 0;
    if (MASK & 1) op_dense<1>(v, m + 4 * k++);
    if (MASK & 2) op_dense<2>(v, m + 4 * k++);
    if (MASK & 4) op_dense<4>(v, m + 4 * k++);
    if constexpr (N > 8)
        if (MASK & 8) op_dense<8>(v, m + 4 * k++);
}

// Packed index of the bits of s selected by MASK (inverse of dep).
__host__ __device__ constexpr int ext(int mask, int s)
{
    int out = 0, k = 0;
    for (int b = 0; b < 4; b++)
        if ((mask >> b) & 1) {
            if ((s >> b) & 1) out |= 1 << k;
            k++;
        }
    return out;
}

// Kronecker product of 2x2 gates in Euler form on the micro bits of MASK:
// gate b is D1_b * RX_b * D2_b with RX_b = [[x, -iy], [-iy, x]] (x, y real),
// D1_b diagonal and D2_b = diag(1, q_b).  The rotations cost 4 FMA-class
// instructions per amplitude each (against 8 for a dense 2x2), and the
// diagonals of all bits are one multiply by a table entry indexed by the
// amplitude's MASK bits.  Coefficients (complex elements): (x_b, y_b) per
// bit in ascending order, the D1 table (2^K entries), then, with D2, the D2
// table (its entry 0 is 1 and is not applied).
template <int MASK, bool HAS_D2, typename R, int N>
__device__ __forceinline__ void op_ekron(Cx<R> (&v)[N], const Cx<R>* __restrict__ m)
{
    constexpr int K = popc4(MASK);
    if constexpr (HAS_D2) {
        const Cx<R>* __restrict__ t2 = m + K + (1 << K);
#pragma unroll
        for (int s = 0; s < N; s++)
            if (ext(MASK, s)) v[s] = cmul(t2[ext(MASK, s)], v[s]);
    }
    int k = 0;
#pragma unroll
    for (int b = 0; b < 4; b++) {
        if (!((MASK >> b) & 1)) continue;
        const R x = m[k].re, y = m[k].im;
        k++;
#pragma unroll
        for (int s = 0; s < N; s++) {
            if ((s >> b) & 1) continue;
            const Cx<R> a = v[s], c = v[s | (1 << b)];
            v[s] = Cx<R>{fmar(x, a.re, y * c.im), fmar(x, a.im, -(y * c.re))};
            v[s | (1 << b)] = Cx<R>{fmar(x, c.re, y * a.im), fmar(x, c.im, -(y * a.re))};
        }
    }
    const Cx<R>* __restrict__ t1 = m + K;
#pragma unroll
    for (int s = 0; s < N; s++) v[s] = cmul(t1[ext(MASK, s)], v[s]);
}

// OK_FKRON on every register bit: the rotations scaled to
// [[1, -it], [-it, 1]] cost 2 FMAs per amplitude per bit (one per output
// component), then one multiply by the table T (the scales, the D1
// diagonal); coefficients: (t_b, 0) per bit in ascending order, then T.
// The exchanged outputs of the flip mask are undone by the caller's store.
template <typename R, int N>
__device__ __forceinline__ void op_fkron(Cx<R> (&v)[N], const Cx<R>* __restrict__ m)
{
#pragma unroll
    for (int b = 0; (1 << b) < N; b++) {
        const R t = m[b].re;
#pragma unroll
        for (int s = 0; s < N; s++) {
            if ((s >> b) & 1) continue;
            const Cx<R> a = v[s], c = v[s | (1 << b)];
            v[s] = Cx<R>{fmar(t, c.im, a.re), fmar(-t, c.re, a.im)};
            v[s | (1 << b)] = Cx<R>{fmar(t, a.im, c.re), fmar(-t, a.re, c.im)};
        }
    }
    constexpr int K = N == 16 ? 4 : (N == 8 ? 3 : 2);
    const Cx<R>* __restrict__ t1 = m + K;
#pragma unroll
    for (int s = 0; s < N; s++) v[s] = cmul(t1[s], v[s]);
}

#define KATE_OPC(kind, var) (((kind) << 8) | (var))

template <typename R, int N>
__device__ __forceinline__ void apply_op(Cx<R> (&v)[N], uint32_t code, const Cx<R>* __restrict__ cf)
{
    switch (code) {
#define D(M) \
    case KATE_OPC(OK_DENSE, M): if constexpr ((M) < N) op_dense<M>(v, cf); break; \
    case KATE_OPC(OK_KRON, M): if constexpr ((M) < N) op_kron<M>(v, cf); break;
        D(1) D(2) D(3) D(4) D(5) D(6) D(7) D(8) D(9) D(10) D(11) D(12) D(13) D(14) D(15)
#undef D
#define E(M) \
    case KATE_OPC(OK_EKRON, M): if constexpr ((M) < N) op_ekron<M, false>(v, cf); break; \
    case KATE_OPC(OK_EKRON, (M) | 16): if constexpr ((M) < N) op_ekron<M, true>(v, cf); break;
        E(3) E(5) E(6) E(7) E(9) E(10) E(11) E(12) E(13) E(14) E(15)
#undef E
#define P(J) \
    case KATE_OPC(OK_PHASE, J): if constexpr ((1 << (J)) < N) op_phase<J>(v, cf); break; \
    case KATE_OPC(OK_H, J): if constexpr ((1 << (J)) < N) op_h<J>(v); break;
        P(0) P(1) P(2) P(3)
#undef P
#define CN(T, C) \
    case KATE_OPC(OK_CNOT, (T) * 4 + (C)): if constexpr ((1 << (T)) < N && (1 << (C)) < N) op_cnot<T, C>(v); break;
        CN(0, 1) CN(0, 2) CN(0, 3) CN(1, 0) CN(1, 2) CN(1, 3) CN(2, 0) CN(2, 1) CN(2, 3) CN(3, 0) CN(3, 1) CN(3, 2)
#undef CN
#define CR(A, B) \
    case KATE_OPC(OK_CRK, (A) * 4 + (B)): if constexpr ((1 << (A)) < N && (1 << (B)) < N) op_crk<A, B>(v, cf); break;
        CR(0, 1) CR(0, 2) CR(0, 3) CR(1, 2) CR(1, 3) CR(2, 3)
#undef CR
#define TF(T, A, B) \
    case KATE_OPC(OK_TOFF, (T) * 16 + (A) * 4 + (B)): \
        if constexpr ((1 << (T)) < N && (1 << (A)) < N && (1 << (B)) < N) op_toff<T, A, B>(v); \
        break;
        TF(0, 1, 2) TF(0, 1, 3) TF(0, 2, 3) TF(1, 0, 2) TF(1, 0, 3) TF(1, 2, 3)
        TF(2, 0, 1) TF(2, 0, 3) TF(2, 1, 3) TF(3, 0, 1) TF(3, 0, 2) TF(3, 1, 2)
#undef TF
    default:
        break;
    }
}

// The op set of passes the planner marks light (PassArgs::light): Euler-form
// Kronecker ops without a right diagonal, dense 1-qubit ops, phases,
// Hadamards and CNOTs -- what RX/RZ layers with CNOT ladders lower to.  A
// shorter decision tree than apply_op, and no multi-qubit dense op holding
// its inputs and outputs at once.
template <typename R, int N>
__device__ __forceinline__ void apply_op_light(Cx<R> (&v)[N], uint32_t code, const Cx<R>* __restrict__ cf)
{
    switch (code) {
#define D1(M) \
    case KATE_OPC(OK_DENSE, M): if constexpr ((M) < N) op_dense<M>(v, cf); break;
        D1(1) D1(2) D1(4) D1(8)
#undef D1
#define E(M) \
    case KATE_OPC(OK_EKRON, M): if constexpr ((M) < N) op_ekron<M, false>(v, cf); break;
        E(3) E(5) E(6) E(7) E(9) E(10) E(11) E(12) E(13) E(14) E(15)
#undef E
#define P(J) \
    case KATE_OPC(OK_PHASE, J): if constexpr ((1 << (J)) < N) op_phase<J>(v, cf); break; \
    case KATE_OPC(OK_H, J): if constexpr ((1 << (J)) < N) op_h<J>(v); break;
        P(0) P(1) P(2) P(3)
#undef P
#define CN(T, C) \
    case KATE_OPC(OK_CNOT, (T) * 4 + (C)): if constexpr ((1 << (T)) < N && (1 << (C)) < N) op_cnot<T, C>(v); break;
        CN(0, 1) CN(0, 2) CN(0, 3) CN(1, 0) CN(1, 2) CN(1, 3) CN(2, 0) CN(2, 1) CN(2, 3) CN(3, 0) CN(3, 1) CN(3, 2)
#undef CN
    default:
        break;
    }
}

// LDS index of tile index y under a layout (see MicroStep::cols).
template <int TB>
__device__ __forceinline__ uint32_t layout(uint32_t y, const uint16_t* __restrict__ cols)
{
    uint32_t p = 0;
#pragma unroll
    for (int b = 0; b < TB; b++)
        if ((y >> b) & 1u) p ^= cols[b];
    return p;
}

// One dense gate of any width on the LDS tile: every thread computes its
// 2^NB outputs from LDS, then (after a barrier) writes them.
template <typename R, int TB, int NB>
__device__ __forceinline__ void generic_dense(Cx<R>* tile, const MicroStep* __restrict__ msp,
                                              const Cx<R>* __restrict__ m)
{
    const MicroStep& ms = *msp;
    constexpr int NT = 1 << (TB - NB);
    constexpr int N = 1 << NB;
    const int k = ms.nbits;
    const uint32_t dim = 1u << k;
    uint32_t gmask = 0;
    for (int i = 0; i < k; i++) gmask |= 1u << ms.bits[i];
    Cx<R> out[N];
#pragma unroll
    for (int e = 0; e < N; e++) {
        const uint32_t j = (uint32_t)e * NT + threadIdx.x;
        uint32_t row = 0;
        for (int i = 0; i < k; i++) row |= ((j >> ms.bits[i]) & 1u) << i;
        const uint32_t base = layout<TB>(j & ~gmask, ms.cols);
        Cx<R> acc{0, 0};
        for (uint32_t c = 0; c < dim; c++) {
            uint32_t idx = base;
            for (int i = 0; i < k; i++)
                if ((c >> i) & 1u) idx ^= ms.cols[ms.bits[i]];
            acc = cmac(acc, m[row * dim + c], tile[swz<R>(idx)]);
        }
        out[e] = acc;
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < N; e++) tile[swz<R>(layout<TB>((uint32_t)e * NT + threadIdx.x, ms.cols))] = out[e];
}

// One dense 5-qubit gate on the LDS tile (an SK_GENERIC step of 5 bits):
// the tile splits into 2^(TB-5) groups of 32 amplitudes that the gate mixes.
// Lane l of a wave holds group l (mod the group count) and all threads of a
// wave compute the same rows, so the matrix entries are wave-uniform and
// come in through scalar loads, by columns from the transpose that the plan
// stores after the matrix.  Each thread streams its group's 32 amplitudes
// from LDS into its rows' accumulators and, after a barrier, writes them.
// Every row sums its products in generic_dense's order, so the results are
// bit for bit the same.
template <typename R, int TB, int NB>
__device__ __forceinline__ void dense5(Cx<R>* tile, const MicroStep* __restrict__ msp,
                                       const Cx<R>* __restrict__ m)
{
    constexpr int NT = 1 << (TB - NB);  // threads of the workgroup
    constexpr int G = 1 << (TB - 5);    // groups of 32 amplitudes
    constexpr int RPT = 32 * G / NT;    // rows per thread
    static_assert(NT % G == 0 && RPT >= 1, "each group needs a whole number of threads");
    const uint32_t tid = threadIdx.x;
    const uint32_t grp = tid % (uint32_t)G;
    uint32_t part = tid / (uint32_t)G;
    if constexpr (G >= 64) part = __builtin_amdgcn_readfirstlane(part);  // one part per wave
    uint32_t gmask = 0, oc[5];
#pragma unroll
    for (int i = 0; i < 5; i++) {
        gmask |= 1u << msp->bits[i];
        oc[i] = msp->cols[msp->bits[i]];
    }
    // the group's tile index: its bits on the non-gate tile bits, ascending
    uint32_t y = 0, g = grp;
#pragma unroll
    for (int b = 0; b < TB; b++)
        if (!((gmask >> b) & 1u)) {
            y |= (g & 1u) << b;
            g >>= 1;
        }
    const uint32_t base = layout<TB>(y, msp->cols);
    const uint32_t row0 = part * (uint32_t)RPT;
    const Cx<R>* __restrict__ mt = m + 1024 + row0;  // transpose: entry (row, c) at c * 32 + row
    Cx<R> acc[RPT];
#pragma unroll
    for (int r = 0; r < RPT; r++) acc[r] = Cx<R>{0, 0};
#pragma unroll 4
    for (int c = 0; c < 32; c++) {
        uint32_t idx = base;
#pragma unroll
        for (int i = 0; i < 5; i++)
            if ((c >> i) & 1) idx ^= oc[i];
        const Cx<R> x = tile[swz<R>(idx)];
#pragma unroll
        for (int r = 0; r < RPT; r++) acc[r] = cmac(acc[r], mt[c * 32 + r], x);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RPT; r++) {
        const uint32_t row = row0 + (uint32_t)r;
        uint32_t idx = base;
#pragma unroll
        for (int i = 0; i < 5; i++)
            if ((row >> i) & 1u) idx ^= oc[i];
        tile[swz<R>(idx)] = acc[r];
    }
}

// WIDE: kRegSteps instantiations run register steps only, kGateSteps ones also
// SK_MFMA steps, kAnySteps ones every kind, kValuSteps ones all but matrix-core
// steps; keeping the larger steps out of the common variants keeps their
// register counts at the waves per SIMD that LDS allows.
enum StepSet { kRegSteps = 0, kAnySteps = 1, kGateSteps = 2, kValuSteps = 3 };

typedef float f32x16 __attribute__((ext_vector_type(16)));

template <typename R>
__device__ __forceinline__ Cx<R>& lds_at(Cx<R>* tile, uint32_t byte_off);

template <typename R>
struct MfmaVec;
template <>
struct MfmaVec<double> {
    typedef double t __attribute__((ext_vector_type(4)));
};
template <>
struct MfmaVec<float> {
    typedef float t __attribute__((ext_vector_type(4)));
};

// 16x16 += 16x4 * 4x16, one entry of each operand per lane.
__device__ __forceinline__ MfmaVec<double>::t mfma_16x16x4(double a, double b, MfmaVec<double>::t c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ MfmaVec<float>::t mfma_16x16x4(float a, float b, MfmaVec<float>::t c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Dense K-qubit gate on the matrix cores, in the state's own precision.  The
// gate is a real 2D x 2D matrix (D = 2^K) in the embedding
// [[Mr, -Mi], [Mi, Mr]] and the tile the 2D x 2^(TB-K) right-hand side.  A
// wave owns blocks of 16 columns, which it reads and overwrites in place
// (no barrier inside the step), and takes all rows of them: each element of
// A is then loaded once per wave and used for all its column blocks.
// Contraction step 2t + p holds part p (re, im) of gate rows 4t + lane/16, so
// a lane's two operands of B are one amplitude, and the rows of A are ordered
// so that an amplitude's two parts come out in one lane: whole amplitudes are
// read from and written to LDS.  Row i of row block b is in lane group i % 4,
// element i / 4 (double), or lane group i / 4, element i % 4 (float).
// A is in lane order (add_gate_operand): two values per lane, the parts
// p = 0, 1, for each t and row block.
// Bound by the matrix cores in complex128 (K = 5: 8192 clocks of a CU's FP64
// peak per 12-qubit tile, its HBM traffic 6000) and about evenly by HBM in
// complex64.  26 qubits, 24 Haar gates, all passes: K = 5 complex128 13.1 ms
// (register blocks on the VALU, matrix rows by scalar loads) -> 5.5, complex64
// 3.80 (32x32x2 products, single components scattered to LDS, two waves per
// SIMD) -> 3.26; K = 4 (register ops) 2.34 -> 2.07 and 1.37 -> 1.10; 23 qubits,
// K = 6 (generic step) 36.7 -> 2.9 and 36.7 -> 1.0.
template <typename R, int TB, int NB, int K>
__device__ __forceinline__ void mfma_gate(Cx<R>* tile, const MicroStep* __restrict__ msp, const R* __restrict__ A)
{
    typedef typename MfmaVec<R>::t V4;
    constexpr int D = 1 << K, RB = 2 * D / 16, T = D / 4;
    constexpr int NW = (1 << (TB - NB)) / 64, CB = (1 << (TB - K)) / 16, CBW = CB / NW;
    static_assert(CBW >= 1 && CBW * NW == CB, "column blocks must split evenly over the waves");
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, q = lane >> 4;
    uint32_t gc[K];
#pragma unroll
    for (int i = 0; i < K; i++) gc[i] = swz<R>(msp->gcols[i]) * (uint32_t)sizeof(Cx<R>);
    // LDS byte offset of the lane's column in each block
    uint32_t col[CBW];
#pragma unroll
    for (int c = 0; c < CBW; c++) {
        const uint32_t j = (wave * CBW + c) * 16u + (lane & 15u);
        uint32_t l = 0;
#pragma unroll
        for (int i = 0; i < TB - K; i++)
            if ((j >> i) & 1u) l ^= msp->tcols[i];
        col[c] = swz<R>(l) * (uint32_t)sizeof(Cx<R>);
    }
    V4 acc[CBW][RB];
#pragma unroll
    for (int c = 0; c < CBW; c++)
#pragma unroll
        for (int b = 0; b < RB; b++) acc[c][b] = V4{0, 0, 0, 0};
    const uint32_t rd = ((q & 1u) ? gc[0] : 0u) ^ ((q & 2u) ? gc[1] : 0u);
    const Cx<R>* __restrict__ a2 = reinterpret_cast<const Cx<R>*>(A) + lane;
#pragma unroll 2
    for (int t = 0; t < T; t++) {
        uint32_t row = rd;
#pragma unroll
        for (int i = 2; i < K; i++)
            if ((t >> (i - 2)) & 1) row ^= gc[i];
        Cx<R> x[CBW];
#pragma unroll
        for (int c = 0; c < CBW; c++) x[c] = lds_at(tile, col[c] ^ row);
#pragma unroll
        for (int b = 0; b < RB; b++) {
            const Cx<R> a = a2[(t * RB + b) * 64];
#pragma unroll
            for (int c = 0; c < CBW; c++) acc[c][b] = mfma_16x16x4(a.re, x[c].re, acc[c][b]);
#pragma unroll
            for (int c = 0; c < CBW; c++) acc[c][b] = mfma_16x16x4(a.im, x[c].im, acc[c][b]);
        }
    }
    // rows of block b: double 8b + 4h + q, float 8b + 2q + h
    constexpr bool F64 = sizeof(R) == 8;
    const uint32_t wr = F64 ? rd : ((q & 1u) ? gc[1] : 0u) ^ ((q & 2u) ? gc[2] : 0u);
#pragma unroll
    for (int c = 0; c < CBW; c++)
#pragma unroll
        for (int b = 0; b < RB; b++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                uint32_t row = wr ^ (h ? (F64 ? gc[2] : gc[0]) : 0u);
#pragma unroll
                for (int i = 3; i < K; i++)
                    if ((b >> (i - 3)) & 1) row ^= gc[i];
                lds_at(tile, col[c] ^ row) = Cx<R>{acc[c][b][2 * h], acc[c][b][2 * h + 1]};
            }
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// A 4- or 5-qubit gate (complex64) with split-bf16 products: A = Ahi + Alo (split on the host),
// B = Bhi + Blo (split here), acc += Ahi Bhi + Ahi Blo + Alo Bhi on
// v_mfma_f32_32x32x16_bf16 (lane l holds contraction indices 8(l/32)..+7 of
// its row / column).  Eight consecutive contraction indices are four complex
// amplitudes of consecutive gate rows, read as four 8-byte LDS loads.
template <int TB, int K>
__device__ __forceinline__ void mfma_bf16(Cx<float>* tile, const MicroStep* __restrict__ msp,
                                          const uint32_t* __restrict__ A)
{
    constexpr int D = 1 << K;
    constexpr int RB = 2 * D / 32;
    constexpr int T = 2 * D / 16;
    constexpr int NW = (1 << (TB - 4)) / 64;
    constexpr int CB = (1 << (TB - K)) / 32;
    constexpr int CBW = CB / NW;
    static_assert(CBW >= 1 && CBW * NW == CB, "column blocks must split evenly over the waves");
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t half = (uint32_t)lane >> 5;
    u32x4 a[RB][T][2];
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int part = 0; part < 2; part++)
                a[rb][t][part] = *reinterpret_cast<const u32x4*>(A + ((size_t)((rb * T + t) * 2 + part) * 64 + lane) * 4);
    uint32_t gc[K];
#pragma unroll
    for (int i = 0; i < K; i++) gc[i] = msp->gcols[i];
    const uint32_t hbit = half ? gc[2] : 0u;
#pragma unroll
    for (int cbi = 0; cbi < CBW; cbi++) {
        const uint32_t col = (uint32_t)(wave * CBW + cbi) * 32u + (uint32_t)(lane & 31);
        uint32_t lq = 0;
#pragma unroll
        for (int j = 0; j < TB - K; j++)
            if ((col >> j) & 1u) lq ^= msp->tcols[j];
        f32x16 acc[RB];
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[rb][r] = 0.0f;
#pragma unroll
        for (int t = 0; t < T; t++) {
            uint32_t hi[4], lo[4];
#pragma unroll
            for (int jj = 0; jj < 4; jj++) {
                const int g = 8 * t + jj;  // plus 4*half
                uint32_t lp = lq ^ hbit;
#pragma unroll
                for (int i = 0; i < K; i++)
                    if (i != 2 && ((g >> i) & 1)) lp ^= gc[i];
                const Cx<float> x = tile[swz<float>(lp)];
                // x = hi + lo in bf16, both rounded to nearest even by the
                // packed conversion (re in the low half, im in the high half)
                const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x.re, x.im}, bf16x2));
                const f32x2 rest{x.re - __uint_as_float(h << 16), x.im - __uint_as_float(h & 0xFFFF0000u)};
                hi[jj] = h;
                lo[jj] = __builtin_bit_cast(uint32_t, __builtin_convertvector(rest, bf16x2));
            }
            const bf16x8 bh = __builtin_bit_cast(bf16x8, u32x4{hi[0], hi[1], hi[2], hi[3]});
            const bf16x8 bl = __builtin_bit_cast(bf16x8, u32x4{lo[0], lo[1], lo[2], lo[3]});
#pragma unroll
            for (int rb = 0; rb < RB; rb++) {
                const bf16x8 ah = __builtin_bit_cast(bf16x8, a[rb][t][0]);
                const bf16x8 al = __builtin_bit_cast(bf16x8, a[rb][t][1]);
                acc[rb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bh, acc[rb], 0, 0, 0);
                acc[rb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bl, acc[rb], 0, 0, 0);
                acc[rb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bh, acc[rb], 0, 0, 0);
            }
        }
        float* tf = reinterpret_cast<float*>(tile);
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int o0 = rb * 32 + 8 * (r / 4) + (r % 4);
                const int g0 = o0 % D;
                uint32_t lp = lq ^ hbit;
#pragma unroll
                for (int i = 0; i < K; i++)
                    if (i != 2 && ((g0 >> i) & 1)) lp ^= gc[i];
                tf[2 * swz<float>(lp) + (uint32_t)(o0 / D)] = acc[rb][r];
            }
    }
}

// State offset of the first amplitude of tile `blk`: its bits go to the
// non-tile qubits rest_pos[0..nrest).  Unrolled with constant indices so that
// every rest_pos[] read is a scalar load and the whole sum stays in SALU;
// a loop indexed by the run-time nrest turns each read into a dependent
// vector load.
__device__ __forceinline__ uint64_t rest_base(const PassArgs& pa, uint64_t blk)
{
    uint64_t base = 0;
    const int nrest = pa.nrest;
#pragma unroll
    for (int i = 0; i < kMaxQubits - 10; i++)
        if (i < nrest) base |= ((blk >> i) & 1ull) << pa.rest_pos[i];
    return base;
}

static_assert(offsetof(MicroStep, op0_code) == 2 && offsetof(MicroStep, coef) == 12 &&
                  offsetof(MicroStep, op_begin) == 4 && offsetof(MicroStep, op_count) == 8 &&
                  offsetof(MicroStep, pbyte) == 16 && offsetof(MicroStep, wbyte) == 32 &&
                  offsetof(MicroStep, wflip) == 48 && offsetof(MicroStep, tbyte) == 52 &&
                  offsetof(MicroStep, phase_coef) == 100,
              "step_addressing reads MicroStep as 32-bit words");

// Addressing of an SK_REG micro-step for this thread: op range, the LDS
// byte offsets o[] of the register bits and the thread's base offset b (all
// already swizzled: the swizzle is linear, so offsets combine by XOR).  The
// descriptor is read as 32-bit words at constant offsets (scalar loads).
template <int TB, int NB>
__device__ __forceinline__ void step_addressing(const MicroStep* __restrict__ msp, uint32_t tid, uint32_t& op_begin,
                                                uint32_t& op_count, uint32_t (&o)[4], uint32_t& b)
{
    const uint32_t* __restrict__ w = reinterpret_cast<const uint32_t*>(msp);
    op_begin = w[1];
    op_count = w[2];
#pragma unroll
    for (int k = 0; k < 4; k++) o[k] = w[4 + k];
    b = 0;
#pragma unroll
    for (int i = 0; i < TB - NB; i++)
        if ((tid >> i) & 1u) b ^= w[13 + i];
}

template <typename R>
__device__ __forceinline__ Cx<R>& lds_at(Cx<R>* tile, uint32_t byte_off)
{
    return *reinterpret_cast<Cx<R>*>(reinterpret_cast<char*>(tile) + byte_off);
}

// LDS offset of register amplitude s from the columns of the micro bits.
template <int NB>
__device__ __forceinline__ uint32_t reg_offset(int s, const uint32_t (&o)[4])
{
    uint32_t x = 0;
#pragma unroll
    for (int k = 0; k < NB; k++)
        if ((s >> k) & 1) x ^= o[k];
    return x;
}

// The micro-steps of one pass on the LDS tile (each thread holds 2^NB
// amplitudes of a step in registers); one barrier after each step.
// The ops of an SK_REG step on the thread's registers.  The first op comes
// with the step (no load that waits on the step); the others are read as
// 32-bit words: a 16-bit field would be a vector load (there are no 16-bit
// scalar loads), whose wait also drains every other vector memory operation
// of the wave.
// Returns the step's flip mask: the store writes register s where register
// s ^ flip belongs (non-zero only for a lone OK_FKRON op).
template <typename R, int N, bool LIGHT>
__device__ __forceinline__ uint32_t reg_step_ops(Cx<R> (&v)[N], const MicroStep* __restrict__ msp, uint32_t op_begin,
                                                 uint32_t op_count, const MicroOp* __restrict__ ops,
                                                 const Cx<R>* __restrict__ coef)
{
    const uint32_t w0 = reinterpret_cast<const uint32_t*>(msp)[0];
    const uint32_t code0 = w0 >> 16, coef0 = reinterpret_cast<const uint32_t*>(msp)[3];
    // the planner makes OK_FKRON only in light passes, as the lone op of a
    // step, on every register bit
    if constexpr (LIGHT) {
        if (op_count == 1 && (code0 >> 8) == OK_FKRON) {
            op_fkron<R, N>(v, coef + coef0);
            return (code0 >> 4) & (N - 1);
        }
    }
    // Light complex128 passes: the common step (RX/RZ layers), one Kronecker
    // op in Euler form on every register bit, is taken before the op switch
    // (in the complex64 kernels the extra path would cost occupancy).
    if constexpr (LIGHT && sizeof(R) == 8) {
        if (op_count == 1 && code0 == KATE_OPC(OK_EKRON, N - 1)) {
            op_ekron<N - 1, false>(v, coef + coef0);
            return 0;
        }
    }
    for (uint32_t o = 0; o < op_count; o++) {
        uint32_t code = code0, cofs = coef0;
        if (o) {
            const uint32_t* ow = reinterpret_cast<const uint32_t*>(ops + op_begin + o);
            code = ow[0] & 0xFFFFu;
            cofs = ow[1];
        }
        if constexpr (LIGHT) apply_op_light<R>(v, code, coef + cofs);
        else apply_op<R>(v, code, coef + cofs);
    }
    return 0;
}

// Amplitude at state offset `off` of the basis state that the first pass
// of an execute makes in registers instead of reading (PassArgs::synth_basis).
template <typename R>
__device__ __forceinline__ Cx<R> synth_amp(const PassArgs& pa, uint64_t off)
{
    return Cx<R>{off == pa.synth_index ? (R)1 : (R)0, (R)0};
}

// Amplitude at `off` in a run from |0...0>: zero without a read when the
// offset has a bit of a qubit that no gate has touched yet.
template <typename R>
__device__ __forceinline__ Cx<R> masked_load(const Cx<R>* __restrict__ state, const PassArgs& pa, uint64_t off)
{
    return (off & pa.zero_mask) ? Cx<R>{(R)0, (R)0} : state[off];
}

// State offset of register amplitude s of this thread for a direct step:
// the XOR of the columns of the set thread-index and register bits.
template <int TB, int NB>
__device__ __forceinline__ uint64_t direct_thread_offset(const uint64_t* __restrict__ g, uint32_t tid)
{
    uint64_t off = 0;
#pragma unroll
    for (int i = 0; i < TB - NB; i++)
        if ((tid >> i) & 1u) off ^= g[i];
    return off;
}

template <int NB>
__device__ __forceinline__ uint64_t direct_reg_offset(const uint64_t* __restrict__ g, int s)
{
    uint64_t off = 0;
#pragma unroll
    for (int k = 0; k < NB; k++)
        if ((s >> k) & 1) off ^= g[12 + k];
    return off;
}

template <typename R, int TB, int WIDE, int NB, bool LIGHT>
__device__ __forceinline__ void run_steps(const PassArgs& pa, Cx<R>* tile, const MicroStep* __restrict__ micro,
                                          const MicroOp* __restrict__ ops, const Cx<R>* __restrict__ coef,
                                          const uint32_t* __restrict__ raw, uint32_t m_begin, uint32_t m_end)
{
    constexpr int N = 1 << NB;
    const uint32_t tid = threadIdx.x;
    for (uint32_t mi = m_begin; mi < m_end; mi++) {
        const MicroStep* __restrict__ msp = micro + pa.micro_begin + mi;
        if ((reinterpret_cast<const uint32_t*>(msp)[0] & 0xFFu) == SK_REG) {
            uint32_t op_begin, op_count, oc[4], b;
            step_addressing<TB, NB>(msp, tid, op_begin, op_count, oc, b);
            Cx<R> v[N];
#pragma unroll
            for (int s = 0; s < N; s++) v[s] = lds_at(tile, b ^ reg_offset<NB>(s, oc));
            const uint32_t f = reg_step_ops<R, N, LIGHT>(v, msp, op_begin, op_count, ops, coef);
            const uint32_t bw = b ^ reg_offset<NB>((int)f, oc);
#pragma unroll
            for (int s = 0; s < N; s++) lds_at(tile, bw ^ reg_offset<NB>(s, oc)) = v[s];
        } else if constexpr (WIDE != kRegSteps && NB == 4) {
            if (WIDE == kGateSteps || (WIDE == kAnySteps && msp->kind == SK_MFMA)) {
                const R* operand = reinterpret_cast<const R*>(raw + msp->coef);
                if (msp->nbits == 5) mfma_gate<R, TB, NB, 5>(tile, msp, operand);
                else if (msp->nbits == 6) mfma_gate<R, TB, NB, 6>(tile, msp, operand);
                else mfma_gate<R, TB, NB, 4>(tile, msp, operand);
            } else if constexpr (WIDE != kGateSteps) {
                if (msp->kind == SK_MFMA_BF16) {
                    if constexpr (sizeof(R) == 4) {
                        if (msp->nbits == 5) mfma_bf16<TB, 5>(tile, msp, raw + msp->coef);
                        else mfma_bf16<TB, 4>(tile, msp, raw + msp->coef);
                    }
                } else if (msp->nbits == 5) {
                    dense5<R, TB, NB>(tile, msp, coef + msp->coef);
                } else {
                    generic_dense<R, TB, NB>(tile, msp, coef + msp->coef);
                }
            }
        } else if constexpr (WIDE != kRegSteps) {
            // (a 1024-thread workgroup is held to 128 VGPRs: too few for
            // dense5's 32 amplitudes in complex128)
            constexpr bool kDense5 = TB - NB <= 9;
            if (kDense5 && msp->nbits == 5) dense5<R, TB, NB>(tile, msp, coef + msp->coef);
            else generic_dense<R, TB, NB>(tile, msp, coef + msp->coef);
        }
        __syncthreads();
    }

}

// Store of one tile, reading it through its final layout: the same
// coalesced runs as the load, optionally to permuted positions (store_pos).
template <typename R, int TB, int NB>
__device__ __forceinline__ void store_tile(Cx<R>* __restrict__ state, const PassArgs& pa, uint64_t base,
                                           Cx<R>* tile)
{
    constexpr int N = 1 << NB;
    const uint32_t tid = threadIdx.x;
    {
        uint64_t tb = base;
        uint32_t lt = 0;
#pragma unroll
        for (int b = 0; b < TB - NB; b++) {
            tb |= (uint64_t)((tid >> b) & 1u) << pa.store_pos[b];
            if ((tid >> b) & 1u) lt ^= pa.store_byte[b];
        }
        uint64_t m[NB];
        uint32_t l[4] = {0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < NB; k++) {
            m[k] = 1ull << pa.store_pos[TB - NB + k];
            l[k] = pa.store_byte[TB - NB + k];
        }
#pragma unroll
        for (int i = 0; i < N; i++) {
            uint64_t off = tb;
#pragma unroll
            for (int k = 0; k < NB; k++)
                if ((i >> k) & 1) off += m[k];
            state[off] = lds_at(tile, lt ^ reg_offset<NB>(i, l));
        }
    }
}

// One tile of one pass: load, micro-steps, store.  `blk` is the tile index
// (its bits are the non-tile qubits rest_pos[]).  Each of the 2^(TB-NB)
// threads holds N = 2^NB amplitudes; the register bits are tile bits
// TB-NB..TB-1 when loading and storing.
// Store of a gate pass that also applies the trailing permutation of its
// circuit (PassArgs::scatter): store index u (thread bits, then register
// bits) reads LDS at the XOR of store_byte[k] over its set bits and writes
// `dst` at the XOR of out_tile[k] and of out_rest[i] over the set bits of
// the tile number; store index bits 0..low-1 are offset bits 0..low-1, so
// the writes are whole runs.
// Output offset of tile `blk` of an out-of-place pass: the XOR of
// out_rest[i] over the set bits of blk (scalar loads, SALU).
__device__ __forceinline__ uint64_t out_base(const PassArgs& pa, uint64_t blk, const ScatterArgs* __restrict__ sa)
{
    uint64_t ob = 0;
#pragma unroll
    for (int i = 0; i < kMaxQubits - 10; i++)
        if (i < pa.nrest && ((blk >> i) & 1ull)) ob ^= sa->out_rest[i];
    return ob;
}

template <typename R, int TB, int NB>
__device__ __forceinline__ void scatter_store(Cx<R>* __restrict__ dst, const PassArgs& pa, uint64_t blk, Cx<R>* tile,
                                              const ScatterArgs* __restrict__ sa)
{
    constexpr int N = 1 << NB;
    const uint32_t tid = threadIdx.x;
    sa += pa.scatter_idx;
    uint64_t ob = out_base(pa, blk, sa);
    uint32_t lt = 0;
#pragma unroll
    for (int b = 0; b < TB - NB; b++)
        if ((tid >> b) & 1u) {
            lt ^= pa.store_byte[b];
            ob ^= sa->out_tile[b];
        }
#pragma unroll
    for (int i = 0; i < N; i++) {
        uint32_t l = lt;
        uint64_t o = ob;
#pragma unroll
        for (int k = 0; k < NB; k++)
            if ((i >> k) & 1) {
                l ^= pa.store_byte[TB - NB + k];
                o ^= sa->out_tile[TB - NB + k];
            }
        dst[o] = lds_at(tile, l);
    }
}

// A step is a chain of scalar loads: its descriptor, its ops, their coefficients.
// After a kernel boundary (a fence, in a batch) they miss the XCD's L2, and a
// workgroup that shares its CU with at most one other waits for each, so the
// passes of small states and of batches (WARM) fetch what they read of the plan
// into L2 under the loads of the amplitudes, one vector load a line (20
// qubits, 10 layers, complex128: a call 260 -> 231 us; 256 complex64 circuits of
// 10-20 qubits 3.14 -> 3.07 ms).  Reading the lines into the scalar cache as well
// gained nothing there (234 us) and cost a pass of one tile 11 us.
constexpr uint32_t kWarmLine = 128;

// Starts fetching the first WL * NT lines of what the pass reads of the
// plan's pools into L2 and returns the words read: the caller consumes them
// (warm_done) once its amplitudes are on their way.
template <typename R, int NT, int WL>
__device__ __forceinline__ void warm_plan(const PassArgs& pa, const MicroStep* __restrict__ micro,
                                          const MicroOp* __restrict__ ops, const Cx<R>* __restrict__ coef,
                                          const uint32_t* __restrict__ raw, uint32_t (&x)[WL])
{
    // every pool starts at a line and holds whole words: the line of a word
    // of a range starts inside the pool
    const char* base[4] = {reinterpret_cast<const char*>(micro), reinterpret_cast<const char*>(coef),
                           reinterpret_cast<const char*>(ops), reinterpret_cast<const char*>(raw)};
    const uint64_t begin[4] = {(uint64_t)pa.micro_begin * sizeof(MicroStep), (uint64_t)pa.coef_begin * sizeof(Cx<R>),
                               (uint64_t)pa.ops_begin * sizeof(MicroOp), (uint64_t)pa.raw_begin * 4u};
    const uint64_t end[4] = {(uint64_t)(pa.micro_begin + pa.micro_count) * sizeof(MicroStep),
                             (uint64_t)pa.coef_end * sizeof(Cx<R>), (uint64_t)pa.ops_end * sizeof(MicroOp),
                             (uint64_t)pa.raw_end * 4u};
    uint32_t total = 0, first[4];
    uint64_t from[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        first[r] = total;
        from[r] = begin[r] / kWarmLine;
        if (end[r] > begin[r]) total += (uint32_t)((end[r] - 1) / kWarmLine - from[r]) + 1u;
    }
#pragma unroll
    for (int i = 0; i < WL; i++) {
        // (micro_count > 0: at least one line)
        const uint32_t want = threadIdx.x + (uint32_t)(i * NT), l = want < total ? want : total - 1u;
        const char* p = base[0] + kWarmLine * (from[0] + l);
#pragma unroll
        for (int r = 1; r < 4; r++)
            if (l >= first[r]) p = base[r] + kWarmLine * (from[r] + (l - first[r]));
        x[i] = *reinterpret_cast<const uint32_t*>(p);
    }
}

template <int WL>
__device__ __forceinline__ void warm_done(const uint32_t (&x)[WL])
{
#pragma unroll
    for (int i = 0; i < WL; i++) asm volatile("" ::"v"(x[i]));
}

template <typename R, int TB, int WIDE, int NB, bool LIGHT, bool WARM>
__device__ __forceinline__ void tile_pass(Cx<R>* __restrict__ state, const PassArgs& pa, uint64_t blk, Cx<R>* tile,
                                          const MicroStep* __restrict__ micro, const MicroOp* __restrict__ ops,
                                          const Cx<R>* __restrict__ coef, const uint32_t* __restrict__ raw,
                                          Cx<R>* __restrict__ dst, const ScatterArgs* __restrict__ sa)
{
    constexpr int NT = 1 << (TB - NB);
    constexpr int N = 1 << NB;
    const uint32_t tid = threadIdx.x;

    const uint64_t base = rest_base(pa, blk);
    uint32_t m_begin = 0, m_end = pa.micro_count;
    constexpr int WL = NT < 128 ? 2 : 1;
    uint32_t warm[WL] = {};
    if constexpr (WARM)
        if (pa.micro_count) warm_plan<R, NT, WL>(pa, micro, ops, coef, raw, warm);

    if (pa.fuse_first) {
        // direct first step: HBM -> registers -> ops -> LDS in the step's layout
        const MicroStep* __restrict__ msp = micro + pa.micro_begin;
        uint32_t op_begin, op_count, oc[4], b;
        step_addressing<TB, NB>(msp, tid, op_begin, op_count, oc, b);
        const uint64_t gt = base ^ direct_thread_offset<TB, NB>(pa.first_g, tid);
        Cx<R> v[N];
        if (pa.synth_basis) {
#pragma unroll
            for (int s = 0; s < N; s++) v[s] = synth_amp<R>(pa, gt ^ direct_reg_offset<NB>(pa.first_g, s));
        } else if (pa.zero_mask) {
#pragma unroll
            for (int s = 0; s < N; s++) v[s] = masked_load(state, pa, gt ^ direct_reg_offset<NB>(pa.first_g, s));
        } else {
#pragma unroll
            for (int s = 0; s < N; s++) v[s] = state[gt ^ direct_reg_offset<NB>(pa.first_g, s)];
        }
        if constexpr (WARM) warm_done(warm);
        const uint32_t f = reg_step_ops<R, N, LIGHT>(v, msp, op_begin, op_count, ops, coef);
        m_begin = 1;
        if (pa.micro_count == 1 && pa.fuse_last) {
            // the store of one thread can hit an amplitude that another
            // thread of the tile loads (the final layout moves amplitudes
            // between threads): every load of the tile has completed (its
            // value was used above) once all threads pass this barrier
            __syncthreads();
            Cx<R>* __restrict__ out = pa.scatter ? dst : state;
            const uint64_t ob = pa.scatter ? out_base(pa, blk, sa + pa.scatter_idx) : base;
            const uint64_t gs = ob ^ direct_thread_offset<TB, NB>(pa.last_g, tid) ^
                                direct_reg_offset<NB>(pa.last_g, (int)f);
#pragma unroll
            for (int s = 0; s < N; s++) out[gs ^ direct_reg_offset<NB>(pa.last_g, s)] = v[s];
            return;
        }
        const uint32_t bw = b ^ reg_offset<NB>((int)f, oc);
#pragma unroll
        for (int s = 0; s < N; s++) lds_at(tile, bw ^ reg_offset<NB>(s, oc)) = v[s];
    } else {   // load
        uint64_t tb = base;
#pragma unroll
        for (int b = 0; b < TB - NB; b++) tb |= (uint64_t)((tid >> b) & 1u) << pa.load_pos[b];
        uint64_t m[NB];
#pragma unroll
        for (int k = 0; k < NB; k++) m[k] = 1ull << pa.load_pos[TB - NB + k];
        Cx<R> r[N];
        if (pa.synth_basis) {
#pragma unroll
            for (int i = 0; i < N; i++) {
                uint64_t off = tb;
#pragma unroll
                for (int k = 0; k < NB; k++)
                    if ((i >> k) & 1) off += m[k];
                r[i] = synth_amp<R>(pa, off);
            }
        } else if (pa.zero_mask) {
#pragma unroll
            for (int i = 0; i < N; i++) {
                uint64_t off = tb;
#pragma unroll
                for (int k = 0; k < NB; k++)
                    if ((i >> k) & 1) off += m[k];
                r[i] = masked_load(state, pa, off);
            }
        } else {
#pragma unroll
            for (int i = 0; i < N; i++) {
                uint64_t off = tb;
#pragma unroll
                for (int k = 0; k < NB; k++)
                    if ((i >> k) & 1) off += m[k];
                r[i] = state[off];
            }
        }
        if constexpr (WARM) warm_done(warm);
        const uint32_t tsw = swz<R>(tid) * (uint32_t)sizeof(Cx<R>);
#pragma unroll
        for (int i = 0; i < N; i++) lds_at(tile, tsw ^ (swz<R>((uint32_t)i * NT) * (uint32_t)sizeof(Cx<R>))) = r[i];
    }
    __syncthreads();

    if (pa.fuse_last) m_end--;
    run_steps<R, TB, WIDE, NB, LIGHT>(pa, tile, micro, ops, coef, raw, m_begin, m_end);
    if (pa.fuse_last) {
        // direct last step: LDS in the step's layout -> registers -> ops -> HBM
        const MicroStep* __restrict__ msp = micro + pa.micro_begin + m_end;
        uint32_t op_begin, op_count, oc[4], b;
        step_addressing<TB, NB>(msp, tid, op_begin, op_count, oc, b);
        Cx<R> v[N];
#pragma unroll
        for (int s = 0; s < N; s++) v[s] = lds_at(tile, b ^ reg_offset<NB>(s, oc));
        const uint32_t f = reg_step_ops<R, N, LIGHT>(v, msp, op_begin, op_count, ops, coef);
        // an out-of-place pass writes the other buffer, at its own tile base
        Cx<R>* __restrict__ out = pa.scatter ? dst : state;
        const uint64_t ob = pa.scatter ? out_base(pa, blk, sa + pa.scatter_idx) : base;
        const uint64_t gs = ob ^ direct_thread_offset<TB, NB>(pa.last_g, tid) ^
                            direct_reg_offset<NB>(pa.last_g, (int)f);
#pragma unroll
        for (int s = 0; s < N; s++) out[gs ^ direct_reg_offset<NB>(pa.last_g, s)] = v[s];
    } else if (pa.scatter) {
        scatter_store<R, TB, NB>(dst, pa, blk, tile, sa);
    } else {
        store_tile<R, TB, NB>(state, pa, base, tile);
    }
}

// Waves per SIMD that the LDS tiles of one CU (160 KiB) allow.
template <typename R, int TB, int NB>
constexpr int kLdsWavesPerSimd =
    (163840 / ((1 << TB) * 2 * (int)sizeof(R))) * ((1 << (TB - NB)) / 64) / 4;

// Minimum waves per SIMD the register allocation must allow: two for
// complex128 16-amplitude threads (their 64 KiB LDS tiles allow two per CU),
// for the other light variants and the complex64 gate variant (176 VGPRs left
// it two waves) as many as their LDS tiles allow, at most four; the compiler's own choice otherwise.
template <typename R, int TB, int WIDE, int NB, bool LIGHT>
constexpr int kPassWavesPerEU =
    (sizeof(R) == 8 && NB == 4) ? 2
                                : (LIGHT || WIDE == kGateSteps ? (kLdsWavesPerSimd<R, TB, NB> < 1 ? 1
                                            : (kLdsWavesPerSimd<R, TB, NB> > 4 ? 4 : kLdsWavesPerSimd<R, TB, NB>))
                                         : 1);

// LIGHT: the pass's ops are all in the light set (apply_op_light).
template <typename R, int TB, int WIDE, int NB, bool LIGHT, bool WARM = false>
__global__ __launch_bounds__(1 << (TB - NB)) __attribute__((amdgpu_waves_per_eu(kPassWavesPerEU<R, TB, WIDE, NB, LIGHT>)))
void k_pass(Cx<R>* __restrict__ state, PassArgs pa,
                                                         const MicroStep* __restrict__ micro,
                                                         const MicroOp* __restrict__ ops,
                                                         const Cx<R>* __restrict__ coef,
                                                         const uint32_t* __restrict__ raw,
                                                         Cx<R>* __restrict__ dst,
                                                         const ScatterArgs* __restrict__ sa)
{
    __shared__ Cx<R> tile[1 << TB];
    tile_pass<R, TB, WIDE, NB, LIGHT, WARM>(state, pa, blockIdx.x, tile, micro, ops, coef, raw, dst, sa);
}

// ---- streamed passes -----------------------------------------------------------
//
// k_stream runs the passes of programs of 1-qubit, CNOT and CRk gates whose CRk
// gates make it the cheaper form (PassArgs::stream; the planner's streams_pay).
// Each register step is a stream of three ops -- a rotation along any register
// direction, a 16-entry diagonal, a phase of the thread -- and writes its
// registers back through a linear map, so CNOTs inside a step cost nothing
// and diagonal gates collect into one product.  A CRk needs only one of its
// qubits in registers: the other one's value is a bit of the thread index or of
// the tile's offset, and the phases of all of them are one factor per
// register bit, looked up in 16-entry tables.  The 300 CRk of a 25-qubit QFT
// then fit the 3 passes its Hadamards need (14 with both qubits in registers:
// 5.05 -> 1.33 ms complex128; a copy of the state is 0.2 ms a pass).  Bound by
// the latency of the ops' operands with two workgroups of four waves per CU:
// scalar loads of rotations and diagonals (their cache lines are fetched ahead
// of the step: 45 % of a step waited on them), table lookups (read one op ahead).

// [[1, -it], [-it, 1]] on every pair (s, s ^ D) in place; the member with the
// lowest bit of D set comes out divided by 1 + t^2 (u = t / (1 + t^2)).
template <int D, typename R>
__device__ __forceinline__ void rotate(Cx<R> (&v)[16], R t, R u)
{
    constexpr int LOW = D & -D;
#pragma unroll
    for (int s = 0; s < 16; s++) {
        if (s & LOW) continue;
        v[s].re = fmar(t, v[s ^ D].im, v[s].re);
        v[s].im = fmar(-t, v[s ^ D].re, v[s].im);
        v[s ^ D].re = fmar(u, v[s].im, v[s ^ D].re);
        v[s ^ D].im = fmar(-u, v[s].re, v[s ^ D].im);
    }
}

// Registers with parity(s & M) ^ P times h.
template <int M, int P, typename R>
__device__ __forceinline__ void phase(Cx<R> (&v)[16], Cx<R> h)
{
#pragma unroll
    for (int s = 0; s < 16; s++)
        if ((popc4(s & M) & 1) ^ P) v[s] = cmul(h, v[s]);
}

// The ops of a streamed step, their codes four to a word.  `pt`: the thread
// tables of its SC_PHASE ops (NT: bits of the thread index), read one op
// ahead; `tile_phase`: the tile's factors of the same ops.
template <typename R, int NT>
__device__ __forceinline__ void stream_ops(Cx<R> (&v)[16], const uint32_t* __restrict__ codes,
                                           const Cx<R>* __restrict__ cf, const Cx<R>* __restrict__ pt,
                                           const Cx<R>* tile_phase, uint32_t phases)
{
    constexpr int G = (NT + 3) / 4;
    Cx<R> pre[G];
    uint32_t left = phases;
    auto fetch = [&] {
        if (!left) return;
        left--;
#pragma unroll
        for (int g = 0; g < G; g++) pre[g] = pt[16 * g + ((threadIdx.x >> (4 * g)) & 15u)];
        pt += 16 * G;
    };
    fetch();
    uint32_t cw = codes[0], next = codes[1], n = 0;
    for (;;) {
        const uint32_t code = cw & 0xFFu;
        if (code == SC_END) return;
        cw >>= 8;
        if ((++n & 3u) == 0) {
            cw = next;
            next = codes[(n >> 2) + 1];
        }
        switch (code) {
#define RO(D) \
    case D: rotate<D>(v, cf[0].re, cf[0].im); cf++; break;
            RO(1) RO(2) RO(3) RO(4) RO(5) RO(6) RO(7) RO(8) RO(9) RO(10) RO(11) RO(12) RO(13) RO(14) RO(15)
#undef RO
        case SC_DIAG:
#pragma unroll
            for (int s = 0; s < 16; s++) v[s] = cmul(cf[s], v[s]);
            cf += 16;
            break;
        case SC_LAYER:
            rotate<1>(v, cf[0].re, cf[0].im);
            rotate<2>(v, cf[1].re, cf[1].im);
            rotate<4>(v, cf[2].re, cf[2].im);
            rotate<8>(v, cf[3].re, cf[3].im);
#pragma unroll
            for (int s = 0; s < 16; s++) v[s] = cmul(cf[4 + s], v[s]);
            cf += 20;
            break;
        default: {
            Cx<R> h = *tile_phase++;
#pragma unroll
            for (int g = 0; g < G; g++) h = cmul(pre[g], h);
            fetch();
            switch (code - SC_PHASE) {
#define PH(M) \
    case M: phase<M, 0>(v, h); break; \
    case (M) + 16: phase<M, 1>(v, h); break;
                PH(1) PH(2) PH(3) PH(4) PH(5) PH(6) PH(7) PH(8) PH(9) PH(10) PH(11) PH(12) PH(13) PH(14) PH(15)
#undef PH
            default: __builtin_unreachable();
            }
            break;
        }
        }
    }
}

// All ones if bit i of x is set.
__device__ __forceinline__ uint32_t bit_mask(uint32_t x, int i) { return (uint32_t)((int32_t)(x << (31 - i)) >> 31); }

__device__ __forceinline__ uint64_t bit_select(uint32_t x, int i, uint64_t y)
{
    const uint32_t m = bit_mask(x, i);
    return ((uint64_t)(m & (uint32_t)(y >> 32)) << 32) | (m & (uint32_t)y);
}

constexpr uint32_t kTouchLines = 8;

// A streamed step's scalar words and this thread's LDS offset in it, loaded
// one step ahead.
struct StreamStep {
    uint32_t codes, phase, coef, phase_coef, lines;  // lines: 64-byte lines of the step's coefficients
    uint32_t r[4], w[4], flip;  // LDS byte offsets of the register bits as read and as written
    uint32_t base;
};

template <int TB, int NB>
__device__ __forceinline__ StreamStep load_stream_step(const MicroStep* __restrict__ ms, uint32_t tid)
{
    const uint32_t* __restrict__ w = reinterpret_cast<const uint32_t*>(ms);
    StreamStep st;
    st.codes = w[1];
    st.phase = w[2];
    st.phase_coef = w[25];
    st.coef = w[3];
    st.lines = w[0] >> 16;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        st.r[k] = w[4 + k];
        st.w[k] = w[8 + k];
    }
    st.flip = w[12];
    st.base = 0;
#pragma unroll
    for (int i = 0; i < TB - NB; i++) st.base ^= bit_mask(tid, i) & w[13 + i];
    return st;
}

// Waves per SIMD: what the LDS tiles allow.
template <typename R, int TB>
constexpr int kStreamWavesPerEU = kLdsWavesPerSimd<R, TB, 4> > 4 ? 4 : kLdsWavesPerSimd<R, TB, 4>;

template <typename R, int TB, bool WARM>
__global__ __launch_bounds__(1 << (TB - 4)) __attribute__((amdgpu_waves_per_eu(kStreamWavesPerEU<R, TB>)))
void k_stream(const Cx<R>* state, PassArgs pa, const MicroStep* __restrict__ micro,
              const uint32_t* __restrict__ codes, const Phase* __restrict__ phases,
              const Cx<R>* __restrict__ coef, Cx<R>* out, const ScatterArgs* __restrict__ sa)
{
    constexpr int NB = 4, N = 1 << NB, NT = 1 << (TB - NB);
    __shared__ Cx<R> tile[1 << TB];
    __shared__ Cx<R> tile_phase[kTilePhases];
    const uint32_t tid = threadIdx.x;
    const uint64_t blk = blockIdx.x, base = rest_base(pa, blk);
    const MicroStep* __restrict__ ms = micro + pa.micro_begin;
    constexpr int WL = NT < 128 ? 2 : 1;
    uint32_t warm[WL] = {};
    if constexpr (WARM)
        if (pa.micro_count) warm_plan<R, NT, WL>(pa, micro, (const MicroOp*)codes, coef, codes, warm);
    Cx<R> v[N];
    {
        // the first step's amplitudes straight into its registers, or the
        // tile in load order
        uint64_t tb = base, g[NB];
        if (pa.fuse_first) {
#pragma unroll
            for (int i = 0; i < TB - NB; i++) tb ^= bit_select(tid, i, pa.first_g[i]);
#pragma unroll
            for (int k = 0; k < NB; k++) g[k] = pa.first_g[12 + k];
        } else {
#pragma unroll
            for (int b = 0; b < TB - NB; b++) tb ^= bit_select(tid, b, 1ull << pa.load_pos[b]);
#pragma unroll
            for (int k = 0; k < NB; k++) g[k] = 1ull << pa.load_pos[TB - NB + k];
        }
        auto offset = [&](int s) {
            uint64_t off = tb;
#pragma unroll
            for (int k = 0; k < NB; k++)
                if ((s >> k) & 1) off ^= g[k];
            return off;
        };
        if (pa.synth_basis) {
#pragma unroll
            for (int s = 0; s < N; s++) v[s] = synth_amp<R>(pa, offset(s));
        } else if (pa.zero_mask) {
#pragma unroll
            for (int s = 0; s < N; s++) v[s] = masked_load(state, pa, offset(s));
        } else {
#pragma unroll
            for (int s = 0; s < N; s++) v[s] = state[offset(s)];
        }
    }
    if constexpr (WARM) warm_done(warm);
    // the tile's factors of the pass's phases, one thread each, while the
    // amplitudes come in
    for (uint32_t p = tid; p < pa.phase_count; p += NT) {
        const Phase* __restrict__ ph = phases + pa.phase_begin + p;
        Cx<R> h{(R)1, (R)0};
        const uint32_t groups = ph->groups;
        for (uint32_t g = 0; g < groups; g++) {
            const uint32_t w = ph->pos[g];
            uint32_t e = 0;
#pragma unroll
            for (int i = 0; i < 4; i++) e |= (uint32_t)((base >> ((w >> (8 * i)) & 63u)) & 1ull) << i;
            h = cmul(coef[ph->coef + 16 * g + e], h);
        }
        tile_phase[p] = h;
    }
    if (!pa.fuse_first) {
        const uint32_t tsw = swz<R>(tid) * (uint32_t)sizeof(Cx<R>);
#pragma unroll
        for (int i = 0; i < N; i++) lds_at(tile, tsw ^ (swz<R>((uint32_t)i * NT) * (uint32_t)sizeof(Cx<R>))) = v[i];
    }
    if (!pa.fuse_first || pa.phase_count) __syncthreads();
    StreamStep st;
    if (pa.micro_count) st = load_stream_step<TB, NB>(ms, tid);
    for (uint32_t mi = 0; mi < pa.micro_count; mi++) {
        // the lines of the step's coefficients, fetched into the scalar cache
        // under the LDS reads
        uint32_t touched = 0;
        {
            const char* __restrict__ p = reinterpret_cast<const char*>(coef + st.coef);
#pragma unroll
            for (uint32_t i = 0; i < kTouchLines; i++)
                touched ^= *reinterpret_cast<const uint32_t*>(p + 64 * (i < st.lines ? i : st.lines - 1));
        }
        if (mi || !pa.fuse_first) {
#pragma unroll
            for (int s = 0; s < N; s++) v[s] = lds_at(tile, st.base ^ reg_offset<NB>(s, st.r));
        }
        asm volatile("" ::"s"(touched));
        const uint32_t next_phase = mi + 1 < pa.micro_count ? reinterpret_cast<const uint32_t*>(ms + mi + 1)[2] : pa.phase_count;
        stream_ops<R, TB - NB>(v, codes + st.codes, coef + st.coef, coef + st.phase_coef, tile_phase + st.phase,
                               next_phase - st.phase);
        if (mi + 1 == pa.micro_count) {
            if (pa.fuse_last) break;
        }
        const uint32_t wb = st.base ^ st.flip;
        uint32_t w[4];
#pragma unroll
        for (int k = 0; k < 4; k++) w[k] = st.w[k];
        // the next step's words come in under the LDS writes
        if (mi + 1 < pa.micro_count) st = load_stream_step<TB, NB>(ms + mi + 1, tid);
#pragma unroll
        for (int s = 0; s < N; s++) lds_at(tile, wb ^ reg_offset<NB>(s, w)) = v[s];
        __syncthreads();
    }
    uint64_t tb = pa.scatter ? out_base(pa, blk, sa + pa.scatter_idx) : base, g[NB];
    if (pa.fuse_last) {
        // in place, a one-step pass stores where other threads of the tile
        // load: every load has completed once all threads pass this barrier
        if (pa.micro_count == 1) __syncthreads();
        tb ^= pa.last_xor;
#pragma unroll
        for (int i = 0; i < TB - NB; i++) tb ^= bit_select(tid, i, pa.last_g[i]);
#pragma unroll
        for (int k = 0; k < NB; k++) g[k] = pa.last_g[12 + k];
    } else {
        uint32_t rbase = 0, r[4];
#pragma unroll
        for (int b = 0; b < TB - NB; b++) {
            rbase ^= bit_mask(tid, b) & pa.store_byte[b];
            tb ^= bit_select(tid, b, pa.scatter ? sa[pa.scatter_idx].out_tile[b] : 1ull << pa.store_pos[b]);
        }
#pragma unroll
        for (int k = 0; k < NB; k++) {
            r[k] = pa.store_byte[TB - NB + k];
            g[k] = pa.scatter ? sa[pa.scatter_idx].out_tile[TB - NB + k] : 1ull << pa.store_pos[TB - NB + k];
        }
#pragma unroll
        for (int s = 0; s < N; s++) v[s] = lds_at(tile, rbase ^ reg_offset<NB>(s, r));
    }
#pragma unroll
    for (int s = 0; s < N; s++) {
        uint64_t off = tb;
#pragma unroll
        for (int k = 0; k < NB; k++)
            if ((s >> k) & 1) off ^= g[k];
        out[off] = v[s];
    }
}

template <typename R, int TB, bool WARM>
int stream_t(void* state, const PassArgs& pa, const DevPlan& dp, hipStream_t s)
{
    hipLaunchKernelGGL((k_stream<R, TB, WARM>), dim3(1u << pa.nrest), dim3(1 << (TB - 4)), 0, s, (const Cx<R>*)state, pa,
                       dp.micro, dp.raw, dp.phases, (const Cx<R>*)dp.coef, (Cx<R>*)(pa.scatter ? dp.dst : state), dp.scatter);
    return (int)hipGetLastError();
}

template <typename R, bool WARM>
int stream_r(int tile_bits, void* state, const PassArgs& pa, const DevPlan& dp, hipStream_t s)
{
    if (pa.micro_bits != 4 || (pa.scatter && (!dp.dst || !dp.scatter)) || pa.phase_count > kTilePhases ||
        (pa.phase_count && !dp.phases))
        return (int)hipErrorInvalidValue;
    // the planner streams only plans whose tile size it chose: 12 qubits, 10 or
    // 11 for states that small (13 only in complex64 plans of nothing but light
    // passes)
    switch (tile_bits) {
    case 10: return stream_t<R, 10, WARM>(state, pa, dp, s);
    case 11: return stream_t<R, 11, WARM>(state, pa, dp, s);
    case 12: return stream_t<R, 12, WARM>(state, pa, dp, s);
    default: return (int)hipErrorInvalidValue;
    }
}

// ---- many circuits in one persistent launch ---------------------------------
//
// Tasks are (circuit, pass, tile), queued by pass level, then circuit, then
// tile.  A workgroup takes the next task; a task of pass p > 0 first waits
// until every tile of its circuit's pass p-1 is done.  Tasks are taken in
// queue order and only wait on earlier ones, which running workgroups hold,
// so the queue always drains; the wait is still bounded, and a wait that
// runs out sets *err instead of spinning on.
// complex64 register-step batch kernels are held to 128 VGPRs (4 waves per
// SIMD): with 137 the 8-wave workgroups of 13-bit tiles ran one per CU.
template <typename R, int WIDE>
constexpr int kBatchWavesPerEU = (sizeof(R) == 4 && !WIDE) ? 4 : 1;

template <typename R, int TB, int WIDE, int NB>
__global__ __launch_bounds__(1 << (TB - NB)) __attribute__((amdgpu_waves_per_eu(kBatchWavesPerEU<R, WIDE>)))
void k_batch(Cx<R>* __restrict__ states,
                                                         const uint64_t* __restrict__ circ_off,
                                                         const BatchTask* __restrict__ tasks, uint32_t ntasks,
                                                         uint32_t* __restrict__ next, uint32_t* __restrict__ done,
                                                         const PassArgs* __restrict__ passes,
                                                         const MicroStep* __restrict__ micro,
                                                         const MicroOp* __restrict__ ops,
                                                         const Cx<R>* __restrict__ coef,
                                                         const uint32_t* __restrict__ raw, uint32_t* __restrict__ err)
{
    __shared__ Cx<R> tile[1 << TB];
    __shared__ uint32_t s_task;
    // One thread-0 block per iteration, between two barriers: it counts the
    // task just finished and fetches the next one.  Two separate thread-0
    // blocks (count at the end of an iteration, fetch at the start of the
    // next) sit side by side across the back edge with no barrier between
    // them; the compiler merges them into a thread-0-only path around the
    // loop head and leaves the other lanes of wave 0 circling an inner loop
    // that re-reads the old task index forever.  The index is also read
    // with readfirstlane so that the exit test is a scalar branch.
    //
    // Cross-workgroup visibility costs one agent-scope release (before a
    // finished task is counted) and one agent-scope acquire (after a wait),
    // both by thread 0: on this GPU they write back / invalidate the whole
    // L2 of the XCD (and the CU's L1), which every wave of the workgroup
    // shares, so one wave's fence covers the workgroup once the barrier
    // after the tile has drained every wave's stores.  (Fencing in every
    // thread made the batch four times slower.)
    uint32_t finished = 0xFFFFFFFFu;
    for (;;) {
        if (threadIdx.x == 0) {
            if (finished != 0xFFFFFFFFu) {
                __threadfence();
                __builtin_amdgcn_s_waitcnt(0);  // the L2 write-back has finished
                atomicAdd(done + finished, 1u);
            }
            s_task = atomicAdd(next, 1u);
        }
        __syncthreads();
        const uint32_t t = __builtin_amdgcn_readfirstlane(s_task);
        if (t >= ntasks) break;
        const BatchTask task = tasks[t];
        if (task.wait_pass != 0xFFFFFFFFu) {
            if (threadIdx.x == 0) {
                uint32_t spins = 0;
                while (__hip_atomic_load(done + task.wait_pass, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <
                       task.wait_count) {
                    __builtin_amdgcn_s_sleep(4);
                    if (++spins > (1u << 20)) {
                        atomicOr(err, 1u);
                        break;
                    }
                }
                __threadfence();
                __builtin_amdgcn_s_waitcnt(0);  // the cache invalidation has finished
            }
            __syncthreads();
        }
        tile_pass<R, TB, WIDE, NB, false, true>(states + circ_off[task.circuit], passes[task.pass], task.tile, tile, micro, ops,
                                          coef, raw, nullptr, nullptr);
        // every wave's stores of this tile have completed (each wave drains
        // its memory counters; a workgroup-scope barrier alone does not wait
        // for global stores) before thread 0 fences and counts the task, and
        // every wave has read s_task before thread 0 overwrites it
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        // the last pass of a circuit is read only after this launch ends:
        // no task waits on it, so it is neither fenced nor counted
        finished = task.signal ? task.pass : 0xFFFFFFFFu;
    }
}

template <typename R, int TB, int NB>
int pass_t(void* state, int nq_int, const PassArgs& pa, const DevPlan& dp, hipStream_t s)
{
    // one workgroup per tile; a run from |0...0> may list fewer rest qubits
    (void)nq_int;
    const unsigned grid = 1u << pa.nrest;
    if (pa.has_wide == kGateSteps) {
        if constexpr (NB == 4)
            hipLaunchKernelGGL((k_pass<R, TB, kGateSteps, NB, false>), dim3(grid), dim3(1 << (TB - NB)), 0, s,
                               (Cx<R>*)state, pa, dp.micro, dp.ops, (const Cx<R>*)dp.coef, dp.raw, (Cx<R>*)dp.dst,
                               dp.scatter);
        else
            return (int)hipErrorInvalidValue;
    } else if (pa.has_wide)
        hipLaunchKernelGGL((k_pass<R, TB, kAnySteps, NB, false>), dim3(grid), dim3(1 << (TB - NB)), 0, s, (Cx<R>*)state,
                           pa, dp.micro, dp.ops, (const Cx<R>*)dp.coef, dp.raw, (Cx<R>*)dp.dst, dp.scatter);
    else if (pa.light)
        hipLaunchKernelGGL((k_pass<R, TB, kRegSteps, NB, true>), dim3(grid), dim3(1 << (TB - NB)), 0, s, (Cx<R>*)state,
                           pa, dp.micro, dp.ops, (const Cx<R>*)dp.coef, dp.raw, (Cx<R>*)dp.dst, dp.scatter);
    else
        hipLaunchKernelGGL((k_pass<R, TB, kRegSteps, NB, false>), dim3(grid), dim3(1 << (TB - NB)), 0, s, (Cx<R>*)state,
                           pa, dp.micro, dp.ops, (const Cx<R>*)dp.coef, dp.raw, (Cx<R>*)dp.dst, dp.scatter);
    return (int)hipGetLastError();
}

// complex128 runs 3- or 4-bit micro-steps, complex64 4-bit ones.
template <typename R, int TB>
int pass_nb(void* state, int nq_int, const PassArgs& pa, const DevPlan& dp, hipStream_t s)
{
    if constexpr (sizeof(R) == 8)
        if (pa.micro_bits == 3) return pass_t<R, TB, 3>(state, nq_int, pa, dp, s);
    if (pa.micro_bits != 4) return (int)hipErrorInvalidValue;
    return pass_t<R, TB, 4>(state, nq_int, pa, dp, s);
}

template <typename R>
int pass_r(int tile_bits, void* state, int nq_int, const PassArgs& pa, const DevPlan& dp, hipStream_t s)
{
    switch (tile_bits) {
    case 10: return pass_nb<R, 10>(state, nq_int, pa, dp, s);
    case 11: return pass_nb<R, 11>(state, nq_int, pa, dp, s);
    case 12: return pass_nb<R, 12>(state, nq_int, pa, dp, s);
    case 13: return pass_nb<R, 13>(state, nq_int, pa, dp, s);
    default: return (int)hipErrorInvalidValue;
    }
}

// Passes of register steps with 16 amplitudes per thread, the plan fetched
// ahead.
template <typename R, int TB>
int warm_t(void* state, const PassArgs& pa, const DevPlan& dp, hipStream_t s)
{
    const dim3 grid(1u << pa.nrest), block(1 << (TB - 4));
    if (pa.light)
        hipLaunchKernelGGL((k_pass<R, TB, kRegSteps, 4, true, true>), grid, block, 0, s, (Cx<R>*)state, pa,
                           dp.micro, dp.ops, (const Cx<R>*)dp.coef, dp.raw, (Cx<R>*)dp.dst, dp.scatter);
    else
        hipLaunchKernelGGL((k_pass<R, TB, kRegSteps, 4, false, true>), grid, block, 0, s, (Cx<R>*)state, pa,
                           dp.micro, dp.ops, (const Cx<R>*)dp.coef, dp.raw, (Cx<R>*)dp.dst, dp.scatter);
    return (int)hipGetLastError();
}

template <typename R>
int warm_r(int tile_bits, void* state, const PassArgs& pa, const DevPlan& dp, hipStream_t s)
{
    if (pa.stream) return stream_r<R, true>(tile_bits, state, pa, dp, s);
    switch (tile_bits) {
    case 10: return warm_t<R, 10>(state, pa, dp, s);
    case 11: return warm_t<R, 11>(state, pa, dp, s);
    case 12: return warm_t<R, 12>(state, pa, dp, s);
    case 13: return warm_t<R, 13>(state, pa, dp, s);
    default: return (int)hipErrorInvalidValue;
    }
}

template <typename R, int TB, int WIDE, int NB>
int batch_t(const BatchArgs& a, hipStream_t s)
{
    hipLaunchKernelGGL((k_batch<R, TB, WIDE, NB>), dim3(a.grid), dim3(1 << (TB - NB)), 0, s, (Cx<R>*)a.states,
                       a.circ_off, a.tasks, a.ntasks, a.next, a.done, a.passes, a.dp.micro, a.dp.ops,
                       (const Cx<R>*)a.dp.coef, a.dp.raw, a.err);
    return (int)hipGetLastError();
}

template <typename R, int TB, int WIDE>
int batch_nb(const BatchArgs& a, hipStream_t s)
{
    if constexpr (sizeof(R) == 8)
        if (a.micro_bits == 3) return batch_t<R, TB, WIDE, 3>(a, s);
    if (a.micro_bits != 4) return (int)hipErrorInvalidValue;
    // A complex128 batch plans no matrix-core steps.  With their accumulators
    // its kernels of 10- and 11-qubit tiles hold 318 registers, one wave per
    // SIMD, without 254, two (256 circuits of 13-15 qubits with 8 dense
    // 5-qubit gates each: 2.22 and 1.97 ms, 1.11 and 0.96 ms).  Those of 12
    // qubits run one wave either way, and 8 % slower without (0.87, 0.94 ms).
    constexpr int kSteps = sizeof(R) == 8 && WIDE && TB <= 11 ? (int)kValuSteps : WIDE;
    return batch_t<R, TB, kSteps, 4>(a, s);
}

template <typename R, int WIDE>
int batch_w(const BatchArgs& a, hipStream_t s)
{
    switch (a.tile_bits) {
    case 10: return batch_nb<R, 10, WIDE>(a, s);
    case 11: return batch_nb<R, 11, WIDE>(a, s);
    case 12: return batch_nb<R, 12, WIDE>(a, s);
    case 13: return batch_nb<R, 13, WIDE>(a, s);
    default: return (int)hipErrorInvalidValue;
    }
}

}  // namespace
}  // namespace kate
