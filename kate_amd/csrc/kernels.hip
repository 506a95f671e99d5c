// kernels.hip -- initialisation, reduction and batch-driver kernels and the
// launchers of every kernel (the pass and batch kernels themselves are
// instantiated in pass_f64.hip, pass_f32.hip, batch_f64.hip, batch_f32.hip).
#include "kernels_dev.hpp"
#include "kernels_inst.hpp"

namespace kate {
namespace {


// Fills n words with v (a kernel, so that it can sit in a captured graph).
__global__ __launch_bounds__(256) void k_fill_u32(uint32_t* __restrict__ p, uint64_t n, uint32_t v)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

// |0...0> for every circuit of a batch.
template <typename R>
__global__ __launch_bounds__(256) void k_batch_init(Cx<R>* __restrict__ states, uint64_t total,
                                                    const uint64_t* __restrict__ circ_off, uint32_t count)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride)
        states[i] = Cx<R>{(R)0, (R)0};
}

template <typename R>
__global__ __launch_bounds__(256) void k_batch_ones(Cx<R>* __restrict__ states, const uint64_t* __restrict__ circ_off,
                                                    uint32_t count)
{
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c < count) states[circ_off[c]] = Cx<R>{(R)1, (R)0};
}

// <Z_q> and norms of a batch, level 1: workgroup w reduces the amplitudes
// [tile << kZBlockBits, ...) of circuit item.circuit to {sum |a|^2, and for
// each of the low kZBlockBits index bits the sum over the amplitudes with
// that bit set} (FP64, fixed order).  Bound by the read of the states: one
// workgroup per circuit, as this was first split, left a 20-qubit circuit to
// one CU (256 complex64 circuits of 10-20 qubits: 2.82 ms, 240 MB; blocks of
// 2^14 amplitudes and a sum over blocks: 0.09 ms).
template <typename R>
__global__ __launch_bounds__(256) void k_batch_z(const Cx<R>* __restrict__ states, const uint64_t* __restrict__ circ_off,
                                                 const int32_t* __restrict__ nq_int, const ZItem* __restrict__ items,
                                                 double* __restrict__ part)
{
    constexpr int H = kZBlockBits - 8;  // index bits of the loops
    const uint32_t tid = threadIdx.x;
    const ZItem item = items[blockIdx.x];
    const Cx<R>* __restrict__ st = states + circ_off[item.circuit] + ((uint64_t)item.tile << kZBlockBits);
    const int bits = nq_int[item.circuit];
    const uint32_t iters = 1u << ((bits < kZBlockBits ? bits : kZBlockBits) - 8);
    double val[1 + H + 8];
#pragma unroll
    for (int q = 0; q < 1 + H; q++) val[q] = 0.0;
#pragma unroll 4
    for (uint32_t it = 0; it < iters; it++) {
        const Cx<R> a = st[(it << 8) | tid];
        const double p = (double)a.re * (double)a.re + (double)a.im * (double)a.im;
        val[0] += p;
#pragma unroll
        for (int q = 0; q < H; q++)
            if ((it >> q) & 1u) val[1 + q] += p;
    }
#pragma unroll
    for (int q = 0; q < 8; q++) val[1 + H + q] = ((tid >> q) & 1u) ? val[0] : 0.0;
    __shared__ double wpart[4][1 + H + 8];
#pragma unroll
    for (int j = 0; j < 1 + H + 8; j++) {
        const double s = wave_sum(val[j]);
        if ((tid & 63u) == 0) wpart[tid >> 6][j] = s;
    }
    __syncthreads();
    if (tid < 1 + H + 8) {
        // row: total, bits 0..7 (threads), bits 8.. (loop)
        const int at = tid == 0 ? 0 : (tid <= (uint32_t)H ? (int)tid + 8 : (int)tid - H);
        part[(uint64_t)blockIdx.x * kZRow + at] =
            (wpart[0][tid] + wpart[1][tid]) + (wpart[2][tid] + wpart[3][tid]);
    }
}

// Level 2, one workgroup per circuit: wave w takes the sums of qubits w, w+4,
// ... over the circuit's blocks (an index bit above the block's is a bit of
// the block number), lanes over the blocks.
__global__ __launch_bounds__(256) void k_batch_zfin(const double* __restrict__ part, const uint32_t* __restrict__ first,
                                                    const int32_t* __restrict__ nq, const int64_t* __restrict__ zoff,
                                                    double* __restrict__ z, double* __restrict__ norms)
{
    const uint32_t c = blockIdx.x, lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    const uint32_t r0 = first[c], rows = first[c + 1] - r0;
    const int n = nq[c];
    double total = 0.0;
    for (uint32_t r = lane; r < rows; r += 64) total += part[(uint64_t)(r0 + r) * kZRow];
    total = wave_sum(total);
    for (int q = (int)w; q < n; q += 4) {
        double s1 = 0.0;
        for (uint32_t r = lane; r < rows; r += 64) {
            const double* row = part + (uint64_t)(r0 + r) * kZRow;
            if (q < kZBlockBits) s1 += row[1 + q];
            else if ((r >> (q - kZBlockBits)) & 1u) s1 += row[0];
        }
        s1 = wave_sum(s1);
        if (lane == 0) z[zoff[c] + q] = (total - 2.0 * s1) / total;
    }
    if (threadIdx.x == 0) norms[c] = total;
}

// ---- initialisation --------------------------------------------------------

template <typename R>
__global__ __launch_bounds__(256) void k_init_basis(Cx<R>* __restrict__ st, uint64_t n, uint64_t index)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        st[i] = Cx<R>{(R)(i == index ? 1 : 0), (R)0};
}

// Product state (initialize_probastate, HIPcode/simulator.hpp:26-38).  A
// workgroup writes blocks of 4096 amplitudes (the state is padded to that): the products over index bits
// 0-5 and 6-11 come from two 64-entry tables it makes once, the product over
// the higher bits once per block, so an amplitude costs two multiplications
// instead of one per qubit and the kernel is bound by its writes (25 qubits
// complex128: 0.41 -> 0.10 ms; 28 qubits complex64: 3.43 -> 0.38 ms).
template <typename R>
__global__ __launch_bounds__(256) void k_init_product(Cx<R>* __restrict__ st, uint64_t n, int nq,
                                                       const double* __restrict__ f)
{
    __shared__ Cx<double> lo[64], mid[64];
    const uint32_t tid = threadIdx.x;
    auto times = [&](Cx<double> a, int j, uint64_t bit) {  // qubit j's factor
        const double* c = f + 2 * (bit * (uint64_t)nq + (uint64_t)j);
        return Cx<double>{a.re * c[0] - a.im * c[1], a.re * c[1] + a.im * c[0]};
    };
    if (tid < 128) {
        const int first = tid < 64 ? 0 : 6;
        Cx<double> a{1.0, 0.0};
#pragma unroll
        for (int j = 0; j < 6; j++) a = times(a, first + j, (tid >> j) & 1u);  // nq >= 12
        if (tid < 64) lo[tid] = a;
        else mid[tid - 64] = a;
    }
    __syncthreads();
    for (uint64_t b = blockIdx.x; (b << 12) < n; b += gridDim.x) {
        Cx<double> h{1.0, 0.0};
#pragma unroll 4
        for (int j = 12; j < nq; j++) h = times(h, j, (b >> (j - 12)) & 1ull);
#pragma unroll 4
        for (int it = 0; it < 16; it++) {
            const uint32_t i = ((uint32_t)it << 8) | tid;
            const Cx<double> x = lo[i & 63u], y = mid[i >> 6];
            const Cx<double> p{x.re * y.re - x.im * y.im, x.re * y.im + x.im * y.re};
            st[(b << 12) + i] = Cx<R>{(R)(p.re * h.re - p.im * h.im), (R)(p.re * h.im + p.im * h.re)};
        }
    }
}

template <typename R>
__global__ __launch_bounds__(256) void k_scale(Cx<R>* __restrict__ st, uint64_t n, double f)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        Cx<R> a = st[i];
        st[i] = Cx<R>{(R)((double)a.re * f), (R)((double)a.im * f)};
    }
}

// ---- deterministic reductions ------------------------------------------------

// State offsets of index bits for a read through a GF(2)-linear map: the
// amplitude of index i is at the XOR of col[] over the set bits of i (a state
// whose last permutation passes have not run yet).
struct GatherMap {
    uint64_t col[kMaxQubits];
};

// Kate's amplitude sums: sum_x a_x and, for every index bit q, the sum over
// the x with bit q set, in two launches whatever the size.  Level 1: block b
// of G = gridDim.x (a power of two) reads the 4096-amplitude chunks b + i*G,
// 16 loads in flight per thread.  Index bits: 0-7 thread, 8-11 load, then
// log2(G) bits of b, then the bits of i.  Per chunk each thread adds its 16
// amplitudes to the total, the four load-bit sums and, uniformly over the
// block, the sums of the set bits of i; the thread bits and the waves are
// reduced once per block.  Column c of the sums is part[c * G + b]: 0 the
// total, 1-8 the thread bits, 9-12 the load bits, 13.. the bits of i.
// Bound by the read (proba_state call, 30 qubits complex128: 17.2 GB in 3.29
// -> 2.86 ms, 6.0 TB/s; 28 qubits complex64 0.86 -> 0.39 ms) or, up to about
// 22 qubits, by its two launches (20 qubits 48 -> 24 us): a workgroup per
// chunk that reduced 26 values for 4096 amplitudes, and levels of 256 rows
// reduced value by value in one workgroup, cost more than the loads.
constexpr int kSumCols = 13 + kSumIterBits;

template <typename R, bool GATHER>
__global__ __launch_bounds__(256) void k_ampsums(const Cx<R>* __restrict__ st, uint64_t chunks, GatherMap gm,
                                                 double* __restrict__ part)
{
    const uint32_t tid = threadIdx.x, G = gridDim.x;
    constexpr int V = 5 + kSumIterBits;
    double vr[V], vi[V];  // total, 4 load bits, bits of i
#pragma unroll
    for (int j = 0; j < V; j++) vr[j] = vi[j] = 0.0;
    uint64_t tbase = 0;
    if constexpr (GATHER) {
#pragma unroll
        for (int j = 0; j < 8; j++)
            if ((tid >> j) & 1u) tbase ^= gm.col[j];
    }
    uint32_t i = 0;
    for (uint64_t c = blockIdx.x; c < chunks; c += G, i++) {
        Cx<R> a[16];
        uint64_t gbase = tbase;
        if constexpr (GATHER) {
            for (int j = 0; (c >> j) != 0; j++)
                if ((c >> j) & 1ull) gbase ^= gm.col[12 + j];
        }
#pragma unroll
        for (int it = 0; it < 16; it++) {
            uint64_t off = (c << 12) + ((uint64_t)it << 8) + tid;
            if constexpr (GATHER) {
                off = gbase;
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if ((it >> j) & 1) off ^= gm.col[8 + j];
            }
            a[it] = st[off];
        }
        double cr = 0, ci = 0;
#pragma unroll
        for (int it = 0; it < 16; it++) {
            const double re = (double)a[it].re, im = (double)a[it].im;
            cr += re;
            ci += im;
#pragma unroll
            for (int j = 0; j < 4; j++)
                if ((it >> j) & 1) {
                    vr[1 + j] += re;
                    vi[1 + j] += im;
                }
        }
        vr[0] += cr;
        vi[0] += ci;
#pragma unroll
        for (int j = 0; j < kSumIterBits; j++)
            if ((i >> j) & 1u) {
                vr[5 + j] += cr;
                vi[5 + j] += ci;
            }
    }
    __shared__ double wpart[4][2 * (V + 8)];
    const uint32_t w = tid >> 6;
#pragma unroll
    for (int j = 0; j < V + 6; j++) {
        double re, im;
        if (j < V) {
            re = vr[j];
            im = vi[j];
        } else {  // thread bit j - V
            const bool on = (tid >> (j - V)) & 1u;
            re = on ? vr[0] : 0.0;
            im = on ? vi[0] : 0.0;
        }
        re = wave_sum(re);
        im = wave_sum(im);
        if ((tid & 63u) == 0) {
            wpart[w][2 * j] = re;
            wpart[w][2 * j + 1] = im;
            if (j == 0) {  // thread bits 6 and 7 are the wave number
                wpart[w][2 * (V + 6)] = (w & 1u) ? re : 0.0;
                wpart[w][2 * (V + 6) + 1] = (w & 1u) ? im : 0.0;
                wpart[w][2 * (V + 7)] = (w & 2u) ? re : 0.0;
                wpart[w][2 * (V + 7) + 1] = (w & 2u) ? im : 0.0;
            }
        }
    }
    __syncthreads();
    if (tid < 2 * (V + 8)) {
        const double s = (wpart[0][tid] + wpart[1][tid]) + (wpart[2][tid] + wpart[3][tid]);
        const int j = (int)tid >> 1;
        const int col = j == 0 ? 0 : (j < V ? j + 8 : j - V + 1);
        if (G > 1 || col <= 12) part[2 * ((uint64_t)col * G + blockIdx.x) + (tid & 1u)] = s;
    }
}

// Level 2: workgroup 0 adds the total's column, workgroup 1 + q the column of
// index bit q (or, for a bit of the block number, the totals of the blocks
// with it set).
__global__ __launch_bounds__(256) void k_ampsums_fin(const double* __restrict__ part, uint32_t G, int gbits,
                                                     double* __restrict__ out)
{
    __shared__ double lds[4];
    const int q = (int)blockIdx.x - 1;
    const int bbit = (q >= 12 && q < 12 + gbits) ? q - 12 : -1;
    const int col = q < 0 || bbit >= 0 ? 0 : (q < 12 ? q + 1 : q - 12 - gbits + 13);
    const double* __restrict__ p = part + 2 * (uint64_t)col * G;
    double re = 0, im = 0;
#pragma unroll 4
    for (uint32_t r = threadIdx.x; r < G; r += 256) {
        const bool on = bbit < 0 || ((r >> bbit) & 1u);
        re += on ? p[2 * (uint64_t)r] : 0.0;
        im += on ? p[2 * (uint64_t)r + 1] : 0.0;
    }
    re = block_sum(re, lds);
    im = block_sum(im, lds);
    if (threadIdx.x == 0) {
        out[2 * blockIdx.x] = re;
        out[2 * blockIdx.x + 1] = im;
    }
}

// Walsh-Hadamard transform of 16 values over their 4 index bits.
__device__ __forceinline__ void wht16(double (&v)[16])
{
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
        for (int s = 0; s < 16; s++) {
            if ((s >> b) & 1) continue;
            const double x = v[s], y = v[s | (1 << b)];
            v[s] = x + y;
            v[s | (1 << b)] = x - y;
        }
}

struct ZMaskArg {
    uint64_t m[kZMasks];
};

// Z strings: sum_x |a_x|^2 (-1)^popcount(x & mask) for up to kZMasks masks in
// one read of the state.  Each 4096-amplitude chunk is transformed by a
// Walsh-Hadamard transform of |a|^2 (three 16-point steps in registers with
// two exchanges through LDS: 12 additions per amplitude), after which the sum
// of a mask over the chunk is one entry, mask & 4095, with the sign of the
// mask on the chunk's number; thread j keeps mask j's sum.  The cost no
// longer depends on the number of masks, and the kernel is bound by the read
// (41 masks, 28 qubits complex64: three reads of 16 signed sums each 2.09 ms,
// this 0.40 ms, 5.4 TB/s; 20 qubits 137 -> 21 us a call).  LDS: 32 KiB, XOR swizzle of the low 4 index bits with
// the next 4, so each exchange's 16 lanes hit 16 distinct 8-byte slots.
template <typename R>
__global__ __launch_bounds__(256) void k_zwht(const Cx<R>* __restrict__ st, uint64_t chunks, ZMaskArg mk, int m,
                                              double* __restrict__ part)
{
    __shared__ double w[4096];
    const uint32_t tid = threadIdx.x, lo = tid & 15u, hi = tid >> 4;
    const uint64_t mask = tid < (uint32_t)m ? mk.m[tid & (kZMasks - 1)] : 0ull;
    const uint32_t mlow = (uint32_t)mask & 4095u;
    double acc = 0.0;
    for (uint64_t c = blockIdx.x; c < chunks; c += gridDim.x) {
        double v[16];
#pragma unroll
        for (int it = 0; it < 16; it++) {
            const Cx<R> a = st[(c << 12) + ((uint64_t)it << 8) + tid];
            v[it] = (double)a.re * (double)a.re + (double)a.im * (double)a.im;
        }
        wht16(v);  // index bits 8..11
#pragma unroll
        for (int r = 0; r < 16; r++) w[((uint32_t)r << 8) | (hi << 4) | (lo ^ hi)] = v[r];
        __syncthreads();
        // index bits 0..3: this thread holds indices (hi, lo, r)
#pragma unroll
        for (int r = 0; r < 16; r++) v[r] = w[(hi << 8) | (lo << 4) | ((uint32_t)r ^ lo)];
        wht16(v);
#pragma unroll
        for (int r = 0; r < 16; r++) w[(hi << 8) | (lo << 4) | ((uint32_t)r ^ lo)] = v[r];
        __syncthreads();
        // index bits 4..7: indices (hi, r, lo)
#pragma unroll
        for (int r = 0; r < 16; r++) v[r] = w[(hi << 8) | ((uint32_t)r << 4) | (lo ^ (uint32_t)r)];
        wht16(v);
#pragma unroll
        for (int r = 0; r < 16; r++) w[(hi << 8) | ((uint32_t)r << 4) | (lo ^ (uint32_t)r)] = v[r];
        __syncthreads();
        if (tid < (uint32_t)m) {
            const double x = w[(mlow & ~15u) | ((mlow ^ (mlow >> 4)) & 15u)];
            acc += (__popcll((c << 12) & mask) & 1) ? -x : x;
        }
        __syncthreads();
    }
    if (tid < (uint32_t)m) part[(uint64_t)tid * gridDim.x + blockIdx.x] = acc;
}

// Level 2: workgroup j adds the G partial sums of mask j.
__global__ __launch_bounds__(256) void k_rows_fin(const double* __restrict__ part, uint32_t G, double* __restrict__ out)
{
    __shared__ double lds[4];
    const double* __restrict__ p = part + (uint64_t)blockIdx.x * G;
    double a = 0.0;
#pragma unroll 4
    for (uint32_t r = threadIdx.x; r < G; r += 256) a += p[r];
    a = block_sum(a, lds);
    if (threadIdx.x == 0) out[blockIdx.x] = a;
}

// Level 0 of <a|b> = sum conj(a_i) b_i (FP64): a block reduces 4096
// amplitude pairs to {re, im, |a|^2, |b|^2}.
// Also folds max |a_i - b_i| into *maxabs (bits of a non-negative double,
// which order like the values; the max does not depend on the order).
template <typename RA, typename RB>
__global__ __launch_bounds__(256) void k_overlap0(const Cx<RA>* __restrict__ a, const Cx<RB>* __restrict__ b,
                                                  double* __restrict__ part, unsigned long long* __restrict__ maxabs)
{
    __shared__ double lds[4];
    const uint64_t base = (uint64_t)blockIdx.x << 12;
    double re = 0, im = 0, na = 0, nb = 0, mx = 0;
#pragma unroll
    for (int it = 0; it < 16; it++) {
        const uint64_t i = base + ((uint64_t)it << 8) + threadIdx.x;
        const Cx<RA> x = a[i];
        const Cx<RB> y = b[i];
        const double xr = x.re, xi = x.im, yr = y.re, yi = y.im;
        re += xr * yr + xi * yi;
        im += xr * yi - xi * yr;
        na += xr * xr + xi * xi;
        nb += yr * yr + yi * yi;
        const double dr = xr - yr, di = xi - yi;
        mx = fmax(mx, sqrt(dr * dr + di * di));
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off, 64));
    if ((threadIdx.x & 63) == 0) atomicMax(maxabs, (unsigned long long)__double_as_longlong(mx));
    double* out = part + (uint64_t)blockIdx.x * 4;
    double v = block_sum(re, lds);
    if (threadIdx.x == 0) out[0] = v;
    v = block_sum(im, lds);
    if (threadIdx.x == 0) out[1] = v;
    v = block_sum(na, lds);
    if (threadIdx.x == 0) out[2] = v;
    v = block_sum(nb, lds);
    if (threadIdx.x == 0) out[3] = v;
}

// rows[count][W] -> out[ceil(count/4096)][W] by fixed-order block sums.
__global__ __launch_bounds__(256) void k_rowsum(const double* __restrict__ rows, uint64_t count, int W,
                                                double* __restrict__ out)
{
    __shared__ double lds[4];
    const uint64_t r0 = (uint64_t)blockIdx.x << 12;
    for (int w = 0; w < W; w++) {
        double a = 0.0;
        for (int i = 0; i < 16; i++) {
            const uint64_t r = r0 + ((uint64_t)i << 8) + threadIdx.x;
            if (r < count) a += rows[r * W + w];
        }
        const double s = block_sum(a, lds);
        if (threadIdx.x == 0) out[(uint64_t)blockIdx.x * W + w] = s;
    }
}

// Calibration: the pass's tiles read and written back in place with no
// arithmetic (every amplitude once each way, the load positions of the
// pass, 2^(TB-4) threads of 16 registers, no LDS).  `one` is 1 at run time,
// so the stores cannot be elided.
template <typename R, int TB>
__global__ __launch_bounds__(1 << (TB - 4)) void k_copy_tile(Cx<R>* __restrict__ state, PassArgs pa, R one)
{
    constexpr int NB = 4;
    const uint32_t tid = threadIdx.x;
    uint64_t tb = rest_base(pa, blockIdx.x);
#pragma unroll
    for (int b = 0; b < TB - NB; b++) tb |= (uint64_t)((tid >> b) & 1u) << pa.load_pos[b];
    uint64_t off[1 << NB];
    Cx<R> v[1 << NB];
#pragma unroll
    for (int i = 0; i < (1 << NB); i++) {
        uint64_t o = tb;
#pragma unroll
        for (int k = 0; k < NB; k++)
            if ((i >> k) & 1) o |= 1ull << pa.load_pos[TB - NB + k];
        off[i] = o;
        v[i] = state[o];
    }
#pragma unroll
    for (int i = 0; i < (1 << NB); i++) state[off[i]] = Cx<R>{v[i].re * one, v[i].im * one};
}

// Out-of-place permutation pass (Plan::scatter_pass): tile `blk` of `src`
// (load_pos / rest_pos, read in runs as in k_pass, made from a basis state
// or read through the zero qubits in a run from |0...0>) goes to LDS; then
// store index u (thread bits, then register bits) reads LDS at the XOR of
// store_byte[k] over its set bits and writes dst at the XOR of out_tile[k]
// and of out_rest[i] over the set bits of blk.  Store index bits 0..low-1
// are state offset bits 0..low-1, so each wave writes whole runs.
template <typename R, int TB>
__global__ __launch_bounds__(1 << (TB - 4)) void k_scatter(const Cx<R>* __restrict__ src, Cx<R>* __restrict__ dst,
                                                          PassArgs pa, const ScatterArgs* __restrict__ sa)
{
    constexpr int NB = 4, N = 1 << NB, NT = 1 << (TB - NB);
    __shared__ Cx<R> tile[1 << TB];
    const uint32_t tid = threadIdx.x;
    const uint64_t blk = blockIdx.x;
    uint64_t tb = rest_base(pa, blk);
#pragma unroll
    for (int b = 0; b < TB - NB; b++) tb |= (uint64_t)((tid >> b) & 1u) << pa.load_pos[b];
    Cx<R> r[N];
#pragma unroll
    for (int i = 0; i < N; i++) {
        uint64_t off = tb;
#pragma unroll
        for (int k = 0; k < NB; k++)
            if ((i >> k) & 1) off |= 1ull << pa.load_pos[TB - NB + k];
        r[i] = pa.synth_basis ? synth_amp<R>(pa, off) : ((off & pa.zero_mask) ? Cx<R>{(R)0, (R)0} : src[off]);
    }
    const uint32_t tsw = swz<R>(tid) * (uint32_t)sizeof(Cx<R>);
#pragma unroll
    for (int i = 0; i < N; i++) lds_at(tile, tsw ^ (swz<R>((uint32_t)i * NT) * (uint32_t)sizeof(Cx<R>))) = r[i];
    __syncthreads();
    scatter_store<R, TB, NB>(dst, pa, blk, tile, sa);
}

template <typename R>
int scatter_r(int tile_bits, const void* src, void* dst, const PassArgs& pa, const ScatterArgs* sa, hipStream_t s)
{
    const unsigned grid = 1u << pa.nrest;
    switch (tile_bits) {
#define SC(TB) case TB: hipLaunchKernelGGL((k_scatter<R, TB>), dim3(grid), dim3(1 << (TB - 4)), 0, s, \
                                           (const Cx<R>*)src, (Cx<R>*)dst, pa, sa); break;
        SC(10) SC(11) SC(12) SC(13)
#undef SC
    default: return (int)hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
}

template <typename R>
int copy_tile_r(int tile_bits, void* state, const PassArgs& pa, hipStream_t s)
{
    const unsigned grid = 1u << pa.nrest;
    switch (tile_bits) {
#define CT(TB) case TB: hipLaunchKernelGGL((k_copy_tile<R, TB>), dim3(grid), dim3(1 << (TB - 4)), 0, s, (Cx<R>*)state, pa, (R)1); break;
        CT(10) CT(11) CT(12) CT(13)
#undef CT
    default: return (int)hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
}

inline unsigned grid_for(uint64_t n)
{
    const uint64_t b = (n + 255) / 256;
    return (unsigned)(b < 65536 ? (b ? b : 1) : 65536);
}

}  // namespace

int launch_batch(int dtype, const BatchArgs& a, void* stream)
{
    hipStream_t s = (hipStream_t)stream;
    const uint64_t nw = (uint64_t)a.npasses + 2;  // done[] + next + err
    hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(nw)), dim3(256), 0, s, a.done, (uint64_t)a.npasses, 0u);
    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(256), 0, s, a.next, (uint64_t)1, 0u);
    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(256), 0, s, a.err, (uint64_t)1, 0u);
    if (dtype == 0) {
        hipLaunchKernelGGL(k_batch_init<double>, dim3(grid_for(a.total_amps)), dim3(256), 0, s, (Cx<double>*)a.states,
                           a.total_amps, a.circ_off, a.count);
        hipLaunchKernelGGL(k_batch_ones<double>, dim3((a.count + 255) / 256), dim3(256), 0, s, (Cx<double>*)a.states,
                           a.circ_off, a.count);
        int e = launch_batch_kernel_f64(a, s);
        if (e) return e;
        hipLaunchKernelGGL(k_batch_z<double>, dim3(a.nzitems), dim3(256), 0, s, (const Cx<double>*)a.states, a.circ_off,
                           a.nq_int, a.zitems, a.zpart);
    } else {
        hipLaunchKernelGGL(k_batch_init<float>, dim3(grid_for(a.total_amps)), dim3(256), 0, s, (Cx<float>*)a.states,
                           a.total_amps, a.circ_off, a.count);
        hipLaunchKernelGGL(k_batch_ones<float>, dim3((a.count + 255) / 256), dim3(256), 0, s, (Cx<float>*)a.states,
                           a.circ_off, a.count);
        int e = launch_batch_kernel_f32(a, s);
        if (e) return e;
        hipLaunchKernelGGL(k_batch_z<float>, dim3(a.nzitems), dim3(256), 0, s, (const Cx<float>*)a.states, a.circ_off,
                           a.nq_int, a.zitems, a.zpart);
    }
    hipLaunchKernelGGL(k_batch_zfin, dim3(a.count), dim3(256), 0, s, a.zpart, a.zfirst, a.nq, a.zoff, a.z, a.norms);
    return (int)hipGetLastError();
}

int launch_overlap(int dtype_a, const void* a, int dtype_b, const void* b, int nq_int, double* d_scratch,
                   double* d_out, void* stream)
{
    hipStream_t s = (hipStream_t)stream;
    if (nq_int < 12) return (int)hipErrorInvalidValue;
    const uint64_t chunks = 1ull << (nq_int - 12);
    double* x = chunks == 1 ? d_out : d_scratch;
    double* y = d_scratch + chunks * 4 + 64;
    const dim3 g((unsigned)chunks), t(256);
    unsigned long long* mx = reinterpret_cast<unsigned long long*>(d_out + 4);
    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, s, reinterpret_cast<uint32_t*>(mx), (uint64_t)2, 0u);
    if (dtype_a == 0 && dtype_b == 0)
        hipLaunchKernelGGL((k_overlap0<double, double>), g, t, 0, s, (const Cx<double>*)a, (const Cx<double>*)b, x, mx);
    else if (dtype_a == 0)
        hipLaunchKernelGGL((k_overlap0<double, float>), g, t, 0, s, (const Cx<double>*)a, (const Cx<float>*)b, x, mx);
    else if (dtype_b == 0)
        hipLaunchKernelGGL((k_overlap0<float, double>), g, t, 0, s, (const Cx<float>*)a, (const Cx<double>*)b, x, mx);
    else
        hipLaunchKernelGGL((k_overlap0<float, float>), g, t, 0, s, (const Cx<float>*)a, (const Cx<float>*)b, x, mx);
    uint64_t rows = chunks;
    while (rows > 1) {
        const uint64_t blocks = (rows + 4095) / 4096;
        double* dst = blocks == 1 ? d_out : y;
        hipLaunchKernelGGL(k_rowsum, dim3((unsigned)blocks), dim3(256), 0, s, x, rows, 4, dst);
        rows = blocks;
        std::swap(x, y);
    }
    return (int)hipGetLastError();
}

// Passes that fetch the plan ahead: register steps on at most 512 tiles, two a
// CU, the early passes of a run from |0...0> among them (20 qubits, 10 layers: 260
// us a call without, 249 with passes of 2 to 512 tiles, 231 with those of one
// tile too; a program of one such pass, 10 qubits, 111 and 112 us).  More
// tiles find the plan in the caches and hide what they wait for (the same
// prologue in every launch: 27-qubit brickwork complex128 41.7 -> 42.7 ms,
// 28-qubit layered circuit complex64 20.0 -> 20.3 ms).
static bool warm_pass(const PassArgs& pa)
{
    return pa.nrest <= 9 && pa.micro_count > 0 && pa.micro_bits == 4 && !pa.has_wide;
}

int launch_pass(int dtype, int tile_bits, void* state, int nq_int, const PassArgs& pa, const DevPlan& dp, void* stream)
{
    if (pa.tile_bits != tile_bits || nq_int < tile_bits || nq_int - tile_bits > 31 || pa.nrest > nq_int - tile_bits)
        return (int)hipErrorInvalidValue;
    if (warm_pass(pa))
        return dtype == 0 ? launch_warm_f64(tile_bits, state, pa, dp, stream)
                          : launch_warm_f32(tile_bits, state, pa, dp, stream);
    if (pa.stream)
        return dtype == 0 ? launch_stream_f64(tile_bits, state, pa, dp, stream)
                          : launch_stream_f32(tile_bits, state, pa, dp, stream);
    if (dtype == 0) return launch_pass_f64(tile_bits, state, nq_int, pa, dp, stream);
    return launch_pass_f32(tile_bits, state, nq_int, pa, dp, stream);
}

int launch_scatter(int dtype, int tile_bits, const void* src, void* dst, const PassArgs& pa, const ScatterArgs* sa,
                   void* stream)
{
    if (!pa.scatter || pa.tile_bits != tile_bits || !sa || !dst) return (int)hipErrorInvalidValue;
    if (dtype == 0) return scatter_r<double>(tile_bits, src, dst, pa, sa, (hipStream_t)stream);
    return scatter_r<float>(tile_bits, src, dst, pa, sa, (hipStream_t)stream);
}

int launch_copy_tiles(int dtype, int tile_bits, void* state, int nq_int, const PassArgs& pa, void* stream)
{
    if (pa.tile_bits != tile_bits || nq_int < tile_bits || nq_int - tile_bits > 31 || pa.nrest > nq_int - tile_bits)
        return (int)hipErrorInvalidValue;
    if (dtype == 0) return copy_tile_r<double>(tile_bits, state, pa, (hipStream_t)stream);
    return copy_tile_r<float>(tile_bits, state, pa, (hipStream_t)stream);
}

int launch_init_basis(int dtype, void* state, int nq_int, uint64_t index, void* stream)
{
    const uint64_t n = 1ull << nq_int;
    if (dtype == 0)
        hipLaunchKernelGGL(k_init_basis<double>, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream,
                           (Cx<double>*)state, n, index);
    else
        hipLaunchKernelGGL(k_init_basis<float>, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream,
                           (Cx<float>*)state, n, index);
    return (int)hipGetLastError();
}

int launch_init_product(int dtype, void* state, int nq_int, const double* d_factors, void* stream)
{
    const uint64_t n = 1ull << nq_int;
    if (nq_int < 12) return (int)hipErrorInvalidValue;
    const dim3 g((unsigned)std::min<uint64_t>(n >> 12, 4096));
    if (dtype == 0)
        hipLaunchKernelGGL(k_init_product<double>, g, dim3(256), 0, (hipStream_t)stream,
                           (Cx<double>*)state, n, nq_int, d_factors);
    else
        hipLaunchKernelGGL(k_init_product<float>, g, dim3(256), 0, (hipStream_t)stream,
                           (Cx<float>*)state, n, nq_int, d_factors);
    return (int)hipGetLastError();
}

int launch_scale(int dtype, void* state, int nq_int, double factor, void* stream)
{
    const uint64_t n = 1ull << nq_int;
    if (dtype == 0)
        hipLaunchKernelGGL(k_scale<double>, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, (Cx<double>*)state,
                           n, factor);
    else
        hipLaunchKernelGGL(k_scale<float>, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, (Cx<float>*)state, n,
                           factor);
    return (int)hipGetLastError();
}

namespace {

// log2 of the level-1 workgroups of the amplitude and Z sums: a chunk each up
// to 2^11 workgroups (eight per CU), then up to 16 chunks each, then more
// workgroups (30 qubits complex128: a fixed grid of 2^11 left the last of its
// three rounds over the chip two thirds full).
int sum_grid_bits(int nq_int)
{
    const int cbits = nq_int - 12;
    if (cbits <= 11) return cbits;
    return std::max(11, cbits - kSumIterBits);
}

}  // namespace

uint64_t reduce_scratch_doubles(int nq_int)
{
    // the level-1 sums, and the rows of the overlap (4 per 4096 amplitudes
    // and 4 per 4096 rows)
    const uint64_t chunks = 1ull << (nq_int > 12 ? nq_int - 12 : 0);
    const uint64_t g = 1ull << sum_grid_bits(std::max(nq_int, 12));
    return std::max<uint64_t>(g * std::max(2 * kSumCols, kZMasks), chunks * 5) + 4096;
}

int launch_amp_sums(int dtype, const void* state, int nq_int, double* d_scratch, double* d_out, void* stream,
                    const uint64_t* gather_cols)
{
    hipStream_t s = (hipStream_t)stream;
    if (nq_int < 12 || nq_int > kMaxQubits) return (int)hipErrorInvalidValue;
    const uint64_t chunks = 1ull << (nq_int - 12);
    const int gbits = sum_grid_bits(nq_int);
    const dim3 g(1u << gbits), t(256);
    double* part = gbits ? d_scratch : d_out;  // one workgroup's columns are the result
    GatherMap gm{};
    if (gather_cols) {
        const uint64_t lim = (1ull << nq_int) - 1ull;
        for (int q = 0; q < nq_int; q++) {
            if (gather_cols[q] & ~lim) return (int)hipErrorInvalidValue;  // offsets stay inside the state
            gm.col[q] = gather_cols[q];
        }
    }
#define AS(R, GA) hipLaunchKernelGGL((k_ampsums<R, GA>), g, t, 0, s, (const Cx<R>*)state, chunks, gm, part)
    if (dtype == 0) {
        if (gather_cols) AS(double, true);
        else AS(double, false);
    } else {
        if (gather_cols) AS(float, true);
        else AS(float, false);
    }
#undef AS
    if (gbits) hipLaunchKernelGGL(k_ampsums_fin, dim3((unsigned)nq_int + 1), t, 0, s, d_scratch, 1u << gbits, gbits, d_out);
    return (int)hipGetLastError();
}

int launch_zsums(int dtype, const void* state, int nq_int, const uint64_t* masks, int count, double* d_scratch,
                 double* d_out, void* stream)
{
    hipStream_t s = (hipStream_t)stream;
    if (nq_int < 12 || nq_int > kMaxQubits || count < 1 || count > kZMasks) return (int)hipErrorInvalidValue;
    const uint64_t chunks = 1ull << (nq_int - 12);
    const uint32_t G = 1u << sum_grid_bits(nq_int);
    ZMaskArg mk{};
    std::copy(masks, masks + count, mk.m);
    double* part = G == 1 ? d_out : d_scratch;
    if (dtype == 0)
        hipLaunchKernelGGL(k_zwht<double>, dim3(G), dim3(256), 0, s, (const Cx<double>*)state, chunks, mk, count, part);
    else
        hipLaunchKernelGGL(k_zwht<float>, dim3(G), dim3(256), 0, s, (const Cx<float>*)state, chunks, mk, count, part);
    if (G > 1) hipLaunchKernelGGL(k_rows_fin, dim3((unsigned)count), dim3(256), 0, s, d_scratch, G, d_out);
    return (int)hipGetLastError();
}

}  // namespace kate
