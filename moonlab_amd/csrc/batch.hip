// batch.hip -- one persistent launch that simulates thousands of small,
// uneven circuits.
//
// Each 256-thread workgroup takes the next circuit from an atomic work queue
// (the host orders it longest-first) and runs it start to finish as passes of
// the Pauli-rotation engine (frame_device.h: 16 tile amplitudes per thread in
// registers, LDS only for layout changes):
//   * n <= tile bits (12): the whole state is one tile that never leaves the
//     registers; HBM sees only the program and the results.
//   * n > 12: the state lives in the workgroup's HBM slot and every pass
//     streams it in 2^12-amplitude tiles, the next tile's loads issued before
//     the current tile's rotations.
// Observables are read from the registers and accumulated per thread over all
// tiles of a circuit; one block reduction at its end.
//
// Bound: at two workgroups per CU (64 KiB of LDS each) the rotations' FP64
// FMAs and LDS exchanges for small circuits, slot traffic for large ones.
// The engine before it (1024 threads, one LDS sweep and barrier per op or
// pair of qubits, observables eight at a time) took 83 ms for 4096 ansatz
// instances of 8..18 qubits and 178 us for 193 of 12 qubits; this one takes
// 7.8 ms and 53 us, with 108 (complex128) and 128 (complex64) of its 256
// vector registers' values spilled: the interpreter's fixed registers and the
// measurement share one kernel.
// Workgroups never wait on each other; every workgroup exits when the queue
// is empty, so the grid always drains.
//
// Reference counterparts: the CPU VQE loop (src/algorithms/vqe.c:764-781,
// 1287-1350, 2156-2257) and the one-block-per-search batch kernel
// (src/optimization/gpu/backends/gpu_cuda.cu:350).
#include <hip/hip_runtime.h>

#include <limits.h>

#include <atomic>

#include "batch_device.h"
#include "frame_device.h"
#include "sv_device.h"
#include "sv_internal.h"

namespace mlx {
namespace {

constexpr int NT = kBatchThreads;
constexpr int NW = NT / 64;
constexpr int kMaxObs = 1 + kBatchMaxQubits + (kBatchMaxQubits - 1) + kBatchMaxQubits;

__device__ __forceinline__ double wsum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// The tile's LDS: layout changes and pair reads of amplitudes, later the CDF
// of a tile (one padding double per 16).
struct Shared {
    double2  tile[1 << kBatchMaxTileBits];   // 64 KiB
    double   red[NW][kMaxObs];               // per-wave partials
    double   res[8];                         // block_reduce results
    int      next;
    int      last_nz;
};

// Block reduction of v[0..nv): wave butterflies, then waves summed in order.
// Result j lands in out[j] (for j < nv) on every thread after the call.
template <typename S>
__device__ __forceinline__ void block_reduce(S &sh, double *v, int nv, double *out)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int j = 0; j < nv; j++) {
        const double s = wsum(v[j]);
        if (lane == 0) sh.red[wave][j] = s;
    }
    __syncthreads();
    if ((int)threadIdx.x < nv) {
        double s = 0.0;
        for (int w = 0; w < NW; w++) s += sh.red[w][threadIdx.x];
        out[threadIdx.x] = s;
    }
    __syncthreads();
}

template <typename R>
__device__ __forceinline__ double p2(const cplx_t<R> &x)
{
    const double r = (double)x.x, i = (double)x.y;
    return fmar(r, r, i * i);
}

__device__ __forceinline__ int bit_of(int32_t code, int l, uint64_t base)
{
    // code >= 0: local tile bit; code < 0 (and not INT32_MIN): global qubit -1 - code
    if (code == INT32_MIN) return 0;
    return code >= 0 ? (l >> code) & 1 : (int)((base >> (-1 - code)) & 1ull);
}

template <typename R, int STRIDE>
__device__ void apply_op(cplx_t<R> *t, int T, const BOp &op, uint64_t base)
{
    if ((base & op.cg) != op.cg) return;          // a global control is 0 for this whole tile
    const int tid = threadIdx.x;
    if (op.kind == BOP_MAT1) {
        const R m0 = (R)op.m[0], m1 = (R)op.m[1], m2 = (R)op.m[2], m3 = (R)op.m[3];
        const R m4 = (R)op.m[4], m5 = (R)op.m[5], m6 = (R)op.m[6], m7 = (R)op.m[7];
        const int half = T >> 1;
        for (int p = tid; p < half; p += STRIDE) {
            const int i0 = (int)ins0((uint64_t)p, op.lq), i1 = i0 | (1 << op.lq);
            if ((i0 & (int)op.cl) != (int)op.cl) continue;
            const cplx_t<R> a = t[i0], b = t[i1];
            cplx_t<R> x, y;
            x.x = fmar(m0, a.x, -(m1 * a.y)) + fmar(m2, b.x, -(m3 * b.y));
            x.y = fmar(m0, a.y, m1 * a.x) + fmar(m2, b.y, m3 * b.x);
            y.x = fmar(m4, a.x, -(m5 * a.y)) + fmar(m6, b.x, -(m7 * b.y));
            y.y = fmar(m4, a.y, m5 * a.x) + fmar(m6, b.y, m7 * b.x);
            t[i0] = x;
            t[i1] = y;
        }
    } else if (op.kind == BOP_XPERM) {
        const int half = T >> 1;
        for (int p = tid; p < half; p += STRIDE) {
            const int i0 = (int)ins0((uint64_t)p, op.lq), i1 = i0 | (1 << op.lq);
            if ((i0 & (int)op.cl) != (int)op.cl) continue;
            const cplx_t<R> a = t[i0];
            t[i0] = t[i1];
            t[i1] = a;
        }
    } else if (op.kind == BOP_DIAG) {
        MLX_DIAG4(R, op);
        for (int l = tid; l < T; l += STRIDE) {
            if ((l & (int)op.cl) != (int)op.cl) continue;
            const int k = (bit_of(op.lq2, l, base) << 1) | bit_of(op.lq, l, base);
            t[l] = cmul(t[l], pick4(k, dr0, dr1, dr2, dr3), pick4(k, di0, di1, di2, di3));
        }
    } else {   // BOP_SWAP
        const int b1 = 1 << op.lq, b2 = 1 << op.lq2;
        for (int l = tid; l < T; l += STRIDE) {
            if ((l & b1) && !(l & b2) && (l & (int)op.cl) == (int)op.cl) {
                const int j = (l ^ b1) | b2;
                const cplx_t<R> x = t[l];
                t[l] = t[j];
                t[j] = x;
            }
        }
    }
}

// 2x2 on the register pair (j, j | 1 << P) of a segment, the arithmetic of
// apply_op's BOP_MAT1 term by term.
template <typename R, int NR, int P>
__device__ __forceinline__ void seg_mat1(cplx_t<R> (&v)[1 << NR], const BOp &op, const int (&idx)[1 << NR])
{
    const R m0 = (R)op.m[0], m1 = (R)op.m[1], m2 = (R)op.m[2], m3 = (R)op.m[3];
    const R m4 = (R)op.m[4], m5 = (R)op.m[5], m6 = (R)op.m[6], m7 = (R)op.m[7];
#pragma unroll
    for (int j = 0; j < (1 << NR); j++) {
        if (j & (1 << P)) continue;
        if ((idx[j] & (int)op.cl) != (int)op.cl) continue;
        const cplx_t<R> a = v[j], b = v[j | (1 << P)];
        cplx_t<R> x, y;
        x.x = fmar(m0, a.x, -(m1 * a.y)) + fmar(m2, b.x, -(m3 * b.y));
        x.y = fmar(m0, a.y, m1 * a.x) + fmar(m2, b.y, m3 * b.x);
        y.x = fmar(m4, a.x, -(m5 * a.y)) + fmar(m6, b.x, -(m7 * b.y));
        y.y = fmar(m4, a.y, m5 * a.x) + fmar(m6, b.y, m7 * b.x);
        v[j] = x;
        v[j | (1 << P)] = y;
    }
}

// controlled X on register bit P (apply_op's BOP_XPERM)
template <typename R, int NR, int P>
__device__ __forceinline__ void seg_xperm(cplx_t<R> (&v)[1 << NR], const BOp &op, const int (&idx)[1 << NR])
{
#pragma unroll
    for (int j = 0; j < (1 << NR); j++) {
        if (j & (1 << P)) continue;
        if ((idx[j] & (int)op.cl) != (int)op.cl) continue;
        const cplx_t<R> a = v[j];
        v[j] = v[j | (1 << P)];
        v[j | (1 << P)] = a;
    }
}

// exchange of register bits P1 / P2 (apply_op's BOP_SWAP)
template <typename R, int NR, int P1, int P2>
__device__ __forceinline__ void seg_swap(cplx_t<R> (&v)[1 << NR], const BOp &op, const int (&idx)[1 << NR])
{
#pragma unroll
    for (int j = 0; j < (1 << NR); j++) {
        if (!(j & (1 << P1)) || (j & (1 << P2))) continue;
        if ((idx[j] & (int)op.cl) != (int)op.cl) continue;
        const int k = (j ^ (1 << P1)) | (1 << P2);
        const cplx_t<R> x = v[j];
        v[j] = v[k];
        v[k] = x;
    }
}

// A segment: nops ops whose non-diagonal targets lie in the NR local bits
// rq.  Each thread gathers the 2^NR amplitudes of one group from LDS,
// applies all ops in registers and writes them back: one LDS round trip and
// one barrier for the whole segment instead of one per op.
template <typename R, int STRIDE, int NR>
__device__ __forceinline__ void apply_segment(cplx_t<R> *t, int T, const BOp *ops, int nops, uint32_t packed,
                                              uint64_t base)
{
    int rq[NR];
#pragma unroll
    for (int i = 0; i < NR; i++) rq[i] = (int)((packed >> (5 * i)) & 31u);
    const int groups = T >> NR;
    for (int g = threadIdx.x; g < groups; g += STRIDE) {
        int gb = g;
#pragma unroll
        for (int i = 0; i < NR; i++) gb = (int)ins0((uint64_t)gb, rq[i]);
        int idx[1 << NR];
        cplx_t<R> v[1 << NR];
#pragma unroll
        for (int j = 0; j < (1 << NR); j++) {
            idx[j] = gb;
#pragma unroll
            for (int i = 0; i < NR; i++)
                if (j & (1 << i)) idx[j] |= 1 << rq[i];
            v[j] = t[idx[j]];
        }
        for (int k = 0; k < nops; k++) {
            const BOp &op = ops[k];
            if ((base & op.cg) != op.cg) continue;   // a global control is 0 for this whole tile
            if (op.kind == BOP_DIAG) {
                MLX_DIAG4(R, op);
#pragma unroll
                for (int j = 0; j < (1 << NR); j++) {
                    if ((idx[j] & (int)op.cl) != (int)op.cl) continue;
                    const int d = (bit_of(op.lq2, idx[j], base) << 1) | bit_of(op.lq, idx[j], base);
                    v[j] = cmul(v[j], pick4(d, dr0, dr1, dr2, dr3), pick4(d, di0, di1, di2, di3));
                }
            } else if (op.kind == BOP_MAT1) {
                const int p = op.lq == rq[0] ? 0 : (NR > 2 && op.lq != rq[1]) ? 2 : 1;
                if (p == 0) seg_mat1<R, NR, 0>(v, op, idx);
                else if (p == 1) seg_mat1<R, NR, 1>(v, op, idx);
                else seg_mat1<R, NR, (NR > 2 ? 2 : 1)>(v, op, idx);
            } else if (op.kind == BOP_XPERM) {
                const int p = op.lq == rq[0] ? 0 : (NR > 2 && op.lq != rq[1]) ? 2 : 1;
                if (p == 0) seg_xperm<R, NR, 0>(v, op, idx);
                else if (p == 1) seg_xperm<R, NR, 1>(v, op, idx);
                else seg_xperm<R, NR, (NR > 2 ? 2 : 1)>(v, op, idx);
            } else {   // BOP_SWAP of the register bits of lq and lq2
                const int p1 = op.lq == rq[0] ? 0 : (NR > 2 && op.lq != rq[1]) ? 2 : 1;
                const int p2 = op.lq2 == rq[0] ? 0 : (NR > 2 && op.lq2 != rq[1]) ? 2 : 1;
                if (p1 == 0 && p2 == 1) seg_swap<R, NR, 0, 1>(v, op, idx);
                else if (p1 == 1 && p2 == 0) seg_swap<R, NR, 1, 0>(v, op, idx);
                else if (NR > 2) {
                    constexpr int L = NR > 2 ? 2 : 1;
                    if (p1 == 0 && p2 == 2) seg_swap<R, NR, 0, L>(v, op, idx);
                    else if (p1 == 2 && p2 == 0) seg_swap<R, NR, L, 0>(v, op, idx);
                    else if (p1 == 1 && p2 == 2) seg_swap<R, NR, 1, L>(v, op, idx);
                    else if (p1 == 2 && p2 == 1) seg_swap<R, NR, L, 1>(v, op, idx);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < (1 << NR); j++) t[idx[j]] = v[j];
    }
}

// Run a pass's op list on the tile in LDS: segment headers send their ops
// through registers, other ops run one by one.  Every step ends with a
// workgroup barrier (LDS only when the caller overlaps global traffic).
template <typename R, int STRIDE, int NR, bool LDS_ONLY>
__device__ __forceinline__ void run_pass_ops(cplx_t<R> *t, int T, const BOp *ops, int nops, uint64_t base)
{
    for (int k = 0; k < nops;) {
        const BOp &op = ops[k];
        if (op.kind == BOP_SEG) {
            apply_segment<R, STRIDE, NR>(t, T, ops + k + 1, op.lq, op.cl, base);
            k += 1 + op.lq;
        } else {
            apply_op<R, STRIDE>(t, T, op, base);
            k++;
        }
        if (LDS_ONLY) lds_barrier();
        else __syncthreads();
    }
}

__device__ __forceinline__ uint64_t tile_base(uint64_t t, const BPass &p)
{
    for (int b = 0; b < p.nbits; b++) t = ins0(t, p.qubits[b]);
    return t;
}

// A tile as the batch kernel walks it: the thread holds tile indices tid +
// 2^(nb-4) j (IO layout); byte offsets into the circuit's slot (2^24
// amplitudes at most, so 32 bits hold them).
struct BatchTile {
    uint32_t tid;        // of the thread's index bits
    uint32_t reg[4];     // of register bit i (tile bit nb - 4 + i)
};

template <typename R>
__device__ __forceinline__ BatchTile batch_tile(uint64_t mask, int nb, int tid)
{
    constexpr uint32_t B = (uint32_t)sizeof(cplx_t<R>);
    BatchTile t;
    t.tid = (uint32_t)frame_deposit((uint64_t)tid & ((1ull << (nb - 4)) - 1ull), mask) * B;
#pragma unroll
    for (int i = 0; i < 4; i++) t.reg[i] = (uint32_t)frame_uniform(frame_deposit(1ull << (nb - 4 + i), mask)) * B;
    return t;
}

// byte offset of register value j; base: the tile's, uniform.  The thread's
// part is made opaque per use: hoisted out of the tile loop, the sixteen sums
// would hold (or spill) sixteen registers through the interpreter.
__device__ __forceinline__ uint32_t batch_thread(const BatchTile &t)
{
    uint32_t x = t.tid;
    asm volatile("" : "+v"(x));
    return x;
}
__device__ __forceinline__ uint32_t batch_reg(const BatchTile &t, uint32_t base, int j)
{
    uint32_t o = base;
#pragma unroll
    for (int i = 0; i < 4; i++)
        if ((j >> i) & 1) o |= t.reg[i];
    return o;
}
template <typename R>
__device__ __forceinline__ void batch_load(const cplx_t<R> *slot, const BatchTile &t, uint32_t base,
                                           typename FVec<R>::t (&v)[16])
{
    const uint32_t x = batch_thread(t);
#pragma unroll
    for (int j = 0; j < 16; j++)
        v[j] = frame_ld<R, false>((const cplx_t<R> *)((const char *)slot + batch_reg(t, base, j) + x));
}
template <typename R>
__device__ __forceinline__ void batch_store(cplx_t<R> *slot, const BatchTile &t, uint32_t base,
                                            const typename FVec<R>::t (&v)[16])
{
    const uint32_t x = batch_thread(t);
#pragma unroll
    for (int j = 0; j < 16; j++) frame_st<R, false>((cplx_t<R> *)((char *)slot + batch_reg(t, base, j) + x), v[j]);
}

// What a thread accumulates over the tiles of the low nb qubits.  Tile-index
// bits of the thread (0 .. nb-5) enter only through signs, so one total per
// thread serves every qubit among them; the qubits above the tile take the
// tile's sums (block_reduce), one qubit per thread.
struct ObsAcc {
    double tot = 0.0;
    double reg[4] = {};         // P(1) of the register bits
    double rzz[3] = {};         // <ZZ> of neighbouring register bits
    double link = 0.0;          // Z of register bit 0 (ZZ with the highest thread bit)
};

template <typename V>
__device__ __forceinline__ double pr(const V &x)
{
    const double r = (double)x.x, i = (double)x.y;
    return fmar(r, r, i * i);
}

// norm, P(1) and neighbour <ZZ> sums of one tile into the accumulators; s[0]:
// the tile's mass, s[1]: its Z of the top register bit
template <typename V>
__device__ __forceinline__ void observe_z(const V (&v)[16], ObsAcc &a, bool zz, double (&s)[2])
{
    double t = 0.0, r[4] = {}, z3 = 0.0, q[3] = {}, z0 = 0.0;
#pragma unroll
    for (int j = 0; j < 16; j++) {
        const double p = pr(v[j]);
        t += p;
#pragma unroll
        for (int i = 0; i < 4; i++)
            if ((j >> i) & 1) r[i] += p;
        if (zz) {
#pragma unroll
            for (int i = 0; i < 3; i++) q[i] += (((j >> i) ^ (j >> (i + 1))) & 1) ? -p : p;
            z0 += (j & 1) ? -p : p;
            z3 += (j & 8) ? -p : p;
        }
    }
    a.tot += t;
#pragma unroll
    for (int i = 0; i < 4; i++) a.reg[i] += r[i];
    if (zz) {
#pragma unroll
        for (int i = 0; i < 3; i++) a.rzz[i] += q[i];
        a.link += z0;
    }
    s[0] = t;
    s[1] = z3;
}

// 2 Re sum conj(a) b over the pairs across each register bit
template <typename V>
__device__ __forceinline__ void observe_x(const V (&v)[16], double (&x)[4])
{
#pragma unroll
    for (int i = 0; i < 4; i++) {
        double s = 0.0;
#pragma unroll
        for (int j = 0; j < 16; j++) {
            if ((j >> i) & 1) continue;
            const V a = v[j], b = v[j | (1 << i)];
            s += fmar((double)a.x, (double)b.x, (double)a.y * (double)b.y);
        }
        x[i] += s + s;
    }
}

// the thread's values with tile bits b .. b+3 as register bits
template <typename R>
__device__ __forceinline__ void tile_read(const cplx_t<R> *t, typename FVec<R>::t (&v)[16], int tid, int b)
{
    constexpr int B = (int)sizeof(cplx_t<R>);
    const int lo = tid & ((1 << b) - 1), x0 = lo | ((tid >> b) << (b + 4));
    const int s0 = lds_slot<B>(x0);
#pragma unroll
    for (int j = 0; j < 16; j++) {
        const cplx_t<R> x = t[s0 ^ lds_slot<B>(j << b)];
        v[j].x = x.x;
        v[j].y = x.y;
    }
}

template <typename R>
__device__ __forceinline__ void tile_write(cplx_t<R> *t, const typename FVec<R>::t (&v)[16], int tid, int nb)
{
    constexpr int B = (int)sizeof(cplx_t<R>);
    const int s0 = lds_slot<B>(tid);
#pragma unroll
    for (int j = 0; j < 16; j++) t[s0 ^ lds_slot<B>(j << (nb - 4))] = cplx_t<R>{v[j].x, v[j].y};
}

// Pauli strings over one tile of the low tb qubits (tiles in index order, the
// tile's amplitudes in LDS): term k adds sum_l Re[conj(a_(i^x)) a_i i^ny
// (-1)^popcount(i & z)], i = base | l, into out[k].  The partner i ^ x is in
// the tile when x has no bit at or above tb; otherwise it is read from the
// circuit's HBM slot (the final state, which measurement does not modify).
// Terms are reduced eight at a time; every sum runs in a fixed order, and
// out[k] is updated by one thread, tile after tile.
template <typename R>
__device__ __forceinline__ void measure_pauli_tile(Shared &sh, uint32_t lds, int T, uint64_t base, const cplx_t<R> *slot,
                                   const PauliT *terms, int nterms, double *out)
{
    using V = typename FVec<R>::t;
    using SharedV = const __attribute__((address_space(3))) V;
    constexpr int B = (int)sizeof(V);
    const int tid = threadIdx.x;
    const uint64_t lowmask = (uint64_t)T - 1ull;
    // an LDS pointer of its own address space: a choice between it and the
    // slot stays two loads instead of a flat one
    auto in_tile = [&](int l) { return *(SharedV *)(uintptr_t)(lds + (uint32_t)(lds_slot<B>(l) * B)); };
    for (int c0 = 0; c0 < nterms; c0 += 8) {
        const int cnt = nterms - c0 < 8 ? nterms - c0 : 8;
        double v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            v[j] = 0.0;
            if (j >= cnt) continue;   // uniform across the block
            const uint64_t x = terms[c0 + j].x, z = terms[c0 + j].z;
            const int ny = terms[c0 + j].ny & 3;
            const uint64_t xl = x & lowmask, xh = x & ~lowmask;
            double s = 0.0;
            for (int l = tid; l < T; l += NT) {
                const V a = in_tile(l);
                const V b = xh == 0 ? in_tile(l ^ (int)xl)
                                    : frame_ld<R, false>(&slot[(base ^ xh) | ((uint64_t)l ^ xl)]);
                const double br = (double)b.x, bi = (double)b.y, ar = (double)a.x, ai = (double)a.y;
                const double re = fmar(br, ar, bi * ai);     // Re conj(b) a
                const double im = fmar(br, ai, -(bi * ar));  // Im conj(b) a
                const double c = ny == 0 ? re : ny == 1 ? -im : ny == 2 ? -re : im;
                s += (__popcll((base | (uint64_t)l) & z) & 1) ? -c : c;
            }
            v[j] = s;
        }
        block_reduce(sh, v, cnt, sh.res);
        if (tid < cnt) out[c0 + tid] += sh.res[tid];
        __syncthreads();
    }
}

__device__ __forceinline__ int cdf_at(int l) { return l + (l >> 4); }

// Inclusive scan of p over T entries in LDS (as doubles, at cdf_at), index order.
__device__ __forceinline__ void lds_scan(Shared &sh, double *cdf, int T, double offset)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int per = T >= NT ? T / NT : 1;
    const int lo = tid * per;
    double s = 0.0;
    if (lo < T)
        for (int e = 0; e < per; e++) s += cdf[cdf_at(lo + e)];
    double x = s;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const double y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    if (lane == 63) sh.red[wave][0] = x;
    __syncthreads();
    double run = offset;
    for (int w = 0; w < wave; w++) run += sh.red[w][0];
    run += x - s;
    __syncthreads();
    if (lo < T)
        for (int e = 0; e < per; e++) {
            run += cdf[cdf_at(lo + e)];
            cdf[cdf_at(lo + e)] = run;
        }
    __syncthreads();
}

// first l with u < cdf_l, T when there is none
__device__ __forceinline__ int cdf_find(const double *cdf, int T, double u)
{
    int lo = 0, hi = T;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (u < cdf[cdf_at(mid)]) hi = mid;
        else lo = mid + 1;
    }
    return lo;
}

// A tile of |0..0> other than the first is zero, and so it leaves a pass,
// unless the pass's scale is not finite: the last one's of a circuit with a
// parameter that is not (passes before it carry the scale on, so their zeros
// may stay until then).
__device__ __forceinline__ bool zero_stays_zero(FConst<FPass> P)
{
    return P->scale_r - P->scale_r == 0.0 && P->scale_i - P->scale_i == 0.0;
}

// Pass `level` of the circuits list[0..): one workgroup per tile, those of
// circuit i from first_tile[i] on.  Few circuits past a tile's size, one
// workgroup each, leave most of the chip idle: 39 circuits of 10 to 16 qubits
// took 3.1 ms, the time of the longest one's 14 passes over 16 tiles.
template <typename R>
__global__ __launch_bounds__(NT, 2) void k_batch_pass(const BInst *__restrict__ insts, const int32_t *__restrict__ list,
                                                      const int32_t *__restrict__ first_tile, int count, int level,
                                                      const FPass *__restrict__ passes, const FOp *__restrict__ prog,
                                                      double2 *__restrict__ own)
{
    using V = typename FVec<R>::t;
    __shared__ double2 tile[1 << kBatchMaxTileBits];
    const FConst<int32_t> ft0 = (FConst<int32_t>)(uintptr_t)first_tile;
    int lo = 0, hi = count;   // the last circuit that starts at or before this tile
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (ft0[mid] <= (int)blockIdx.x) lo = mid;
        else hi = mid;
    }
    const FConst<BInst> I = (FConst<BInst>)(uintptr_t)(insts + ((FConst<int32_t>)(uintptr_t)list)[lo]);
    const FConst<FPass> P = (FConst<FPass>)(uintptr_t)(passes + I->first_pass + level);
    const int tid = threadIdx.x, nb = I->tile_bits, threads = 1 << (nb - kFrameRegBits);
    const bool active = tid < threads;
    const uint64_t mask = P->mask;
    const uint64_t base = frame_uniform(frame_deposit((uint64_t)((int)blockIdx.x - ft0[lo]), ~mask));
    cplx_t<R> *slot = (cplx_t<R> *)(own + I->slot_offset);
    constexpr uint32_t B = (uint32_t)sizeof(cplx_t<R>);
    const BatchTile bt = batch_tile<R>(mask, nb, tid);
    V v[16];
    if (level > 0) {
        batch_load<R>(slot, bt, (uint32_t)base * B, v);
    } else {
#pragma unroll
        for (int j = 0; j < 16; j++) v[j] = V{R(j == 0 && tid == 0 && base == 0), R(0)};
    }
    if (level > 0 || base == 0 || !zero_stays_zero(P)) {
        const FrameThread ft = frame_thread(P, prog, tid, nb - kFrameRegBits, active);
        frame_tile<R>(MLX_FRAME_LDS(tile), v, P, prog, ft, base, tid, nb);
    }
    if (active) batch_store<R>(slot, bt, (uint32_t)base * B, v);
}

// Pauli strings of the circuits list[0..), eight to a workgroup: those of
// circuit i from workgroup first[i] on, its final state in its own slot.  The
// sums run in measure_pauli_tile's order, so both give the same bits.  Bound
// by the partners' loads from L2 (512 KiB per tile of 12 qubits).  The
// persistent kernel measures a circuit's strings one workgroup per circuit, at
// 3.4 us per string and tile, most of it address and parity arithmetic: 100
// strings of four 15-qubit circuits took 2.5 ms, here 0.27 ms.
template <typename R>
__global__ __launch_bounds__(NT) void k_batch_pauli(const BInst *__restrict__ insts, const int32_t *__restrict__ list,
                                                    const int32_t *__restrict__ first, int count,
                                                    const PauliT *__restrict__ terms, const double2 *__restrict__ own,
                                                    double *__restrict__ obs)
{
    using V = typename FVec<R>::t;
    constexpr int PER = (1 << kBatchMaxTileBits) / NT;
    __shared__ struct {
        double red[NW][kPauliChunk], res[kPauliChunk];
    } sh;
    const FConst<int32_t> f0 = (FConst<int32_t>)(uintptr_t)first;
    int lo = 0, hi = count;   // the last circuit that starts at or before this workgroup
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (f0[mid] <= (int)blockIdx.x) lo = mid;
        else hi = mid;
    }
    const FConst<BInst> I = (FConst<BInst>)(uintptr_t)(insts + ((FConst<int32_t>)(uintptr_t)list)[lo]);
    const int tid = threadIdx.x, n = I->n, nb = I->tile_bits;
    const int c0 = kPauliChunk * ((int)blockIdx.x - f0[lo]);
    const int cnt = I->num_pauli - c0 < kPauliChunk ? I->num_pauli - c0 : kPauliChunk;
    const FConst<PauliT> term = (FConst<PauliT>)(uintptr_t)(terms + I->pauli_offset + c0);
    const cplx_t<R> *slot = (const cplx_t<R> *)(own + I->pauli_slot);
    const int T = n <= nb ? 1 << n : 1 << nb;
    double acc = 0.0;
    for (uint64_t base = 0; base < 1ull << n; base += (uint64_t)T) {
        V a[PER];
#pragma unroll
        for (int e = 0; e < PER; e++) {
            const int l = tid + NT * e;
            a[e] = l < T ? frame_ld<R, false>(&slot[base + (uint64_t)l]) : V{R(0), R(0)};
        }
        double v[kPauliChunk];
#pragma unroll
        for (int j = 0; j < kPauliChunk; j++) {
            v[j] = 0.0;
            if (j >= cnt) continue;   // uniform across the block
            const uint64_t x = term[j].x, z = term[j].z;
            const int ny = term[j].ny & 3;
            const int own_par = (__popcll(z & base) ^ __popcll(z & (uint64_t)tid)) & 1;
            double s = 0.0;
#pragma unroll
            for (int e = 0; e < PER; e++) {
                const int l = tid + NT * e;
                if (l >= T) continue;
                const V b = frame_ld<R, false>(&slot[(base + (uint64_t)l) ^ x]);
                const double br = (double)b.x, bi = (double)b.y, ar = (double)a[e].x, ai = (double)a[e].y;
                const double re = fmar(br, ar, bi * ai);     // Re conj(b) a
                const double im = fmar(br, ai, -(bi * ar));  // Im conj(b) a
                const double c = ny == 0 ? re : ny == 1 ? -im : ny == 2 ? -re : im;
                s += (own_par ^ (__popcll(z & (uint64_t)(NT * e)) & 1)) ? -c : c;
            }
            v[j] = s;
        }
        block_reduce(sh, v, cnt, sh.res);
        if (tid < cnt) acc += sh.res[tid];
        __syncthreads();
    }
    if (tid < cnt) obs[I->obs_offset + obs_size(n) + c0 + tid] = acc;
}

template <typename R>
__device__ __forceinline__ void run_circuit(Shared &sh, uint32_t lds, const BInst &I, const FPass *passes, const FOp *prog, double2 *slot_raw,
                            double2 *own, double *tile_sums, const double *draws, double *obs, uint64_t *outcomes,
                            const PauliT *terms, void *state_out)
{
    using V = typename FVec<R>::t;
    const int tid = threadIdx.x;
    const int n = I.n, nb = I.tile_bits;              // tile bits: 4 at least, above n for tiny circuits
    const bool resident = n <= nb;
    const uint64_t ntiles = resident ? 1 : 1ull << (n - nb);
    const int threads = 1 << (nb - kFrameRegBits);    // that hold amplitudes
    const bool active = tid < threads;
    cplx_t<R> *t = (cplx_t<R> *)sh.tile;
    // gate passes already run by k_batch_pass on the circuit's own slot
    const bool ready = I.slot_offset >= 0;
    cplx_t<R> *slot = (cplx_t<R> *)(ready ? own + I.slot_offset : slot_raw);

    // ---- gate passes ----
    for (int pi = ready ? I.num_passes : 0; pi < I.num_passes; pi++) {
        const FConst<FPass> P = (FConst<FPass>)(uintptr_t)(passes + I.first_pass + pi);
        const uint64_t mask = P->mask;
        const FrameThread ft = frame_thread(P, prog, tid, nb - kFrameRegBits, active);
        const BatchTile bt = batch_tile<R>(mask, nb, tid);
        // threads past the tile's load what thread tid mod threads loads and store nothing
        const bool load = pi > 0 && !resident, store = !resident && active;
        V pre[16];
        uint64_t base = 0;
        constexpr uint32_t B = (uint32_t)sizeof(cplx_t<R>);
        if (load) batch_load<R>(slot, bt, 0u, pre);
        for (uint64_t ti = 0; ti < ntiles; ti++) {
            // the values live from here to the stores only (a resident
            // circuit has one pass): kept across passes they cost the
            // interpreter's fixed registers a second copy, and more spills
            V v[16];
            const uint64_t next = frame_uniform(frame_step(base, frame_uniform((~mask) & (mask + 1)), mask));
            if (load) {
#pragma unroll
                for (int j = 0; j < 16; j++) v[j] = pre[j];
                if (ti + 1 < ntiles) batch_load<R>(slot, bt, (uint32_t)next * B, pre);
            } else {   // the first pass starts from |0..0>
#pragma unroll
                for (int j = 0; j < 16; j++) v[j] = V{R(j == 0 && tid == 0 && base == 0), R(0)};
            }
            if (load || base == 0 || !zero_stays_zero(P)) frame_tile<R>(lds, v, P, prog, ft, base, tid, nb);
            if (store) batch_store<R>(slot, bt, (uint32_t)base * B, v);
            if (resident) {
                __syncthreads();   // a layout change may still be read
                if (active) tile_write<R>(t, v, tid, nb);
            }
            base = next;
        }
        __syncthreads();   // the slot's stores are visible to the workgroup
    }
    if (I.num_passes == 0) {   // empty circuit: |0..0>
        if (resident) {
            V v[16];
#pragma unroll
            for (int j = 0; j < 16; j++) v[j] = V{R(j == 0 && tid == 0), R(0)};
            if (active) tile_write<R>(t, v, tid, nb);
        } else {
            const uint64_t dim = 1ull << n;
            for (uint64_t i = tid; i < dim; i += NT) slot[i] = cplx_t<R>{R(i == 0), R(0)};
        }
        __syncthreads();
    }

    // ---- the final state, when asked for (geometric-tensor overlaps) or
    // measured by k_batch_pauli and not in the circuit's own slot yet ----
    for (int k = 0; k < 2; k++) {
        if (k ? I.pauli_slot < 0 || ready : I.state_offset < 0) continue;
        cplx_t<R> *so = k ? (cplx_t<R> *)(own + I.pauli_slot) : (cplx_t<R> *)state_out + I.state_offset;
        const uint64_t dim = 1ull << n;
        if (resident) {
            for (uint64_t i = tid; i < dim; i += NT) so[i] = t[lds_slot<(int)sizeof(V)>((int)i)];
        } else {
            for (uint64_t i = tid; i < dim; i += NT) so[i] = slot[i];
        }
    }

    // ---- tiles of the low nb qubits, index order: norm, P(1), <ZZ>, <X> of
    // those qubits, Pauli strings, tile sums for the shots ----
    const bool want_shots = I.num_shots > 0, zz = (I.flags & BF_ZZ) != 0, want_x = (I.flags & BF_X) != 0;
    const int nhigh = resident ? 0 : n - nb, tb = nb - kFrameRegBits;
    const int nzz = n > 1 ? n - 1 : 0;
    double *pauli_out = obs + I.obs_offset + obs_size(n);
    const int npauli = I.pauli_slot >= 0 ? 0 : I.num_pauli;
    for (int k = tid; k < npauli; k += NT) pauli_out[k] = 0.0;
    ObsAcc acc;
    double hi = 0.0, hzz = 0.0;   // thread i: P(1) of qubit nb + i; thread 64 + i: <ZZ> of (nb - 1 + i, nb + i)
    double xs[3][4] = {};         // <X> of the register bits, of tile bits 0..3 and of the four below the register bits
    const bool lds_tile = want_x || npauli > 0;
    __syncthreads();
    for (uint64_t ti = 0; ti < ntiles; ti++) {
        V v[16];
        if (resident) tile_read<R>(t, v, tid & (threads - 1), tb);
        else
#pragma unroll
            for (int j = 0; j < 16; j++)
                v[j] = frame_ld<R, false>(&slot[(ti << nb) | (uint64_t)((tid & (threads - 1)) + threads * j)]);
        double s2[2] = {0.0, 0.0};
        if (active) {
            observe_z<V>(v, acc, zz, s2);
            if (want_x) observe_x<V>(v, xs[0]);
        }
        if (!resident) {
            block_reduce(sh, s2, 2, sh.res);
            const int i = tid & 63;
            if (tid < 64 && i < nhigh && ((ti >> i) & 1ull)) hi += sh.res[0];
            if (tid >= 64 && tid < 128 && i < nhigh) {
                // the tile's top register bit is the qubit below the first high one
                const bool flip = (((ti >> i) ^ (i ? ti >> (i - 1) : 0)) & 1ull) != 0;
                const double x = i ? sh.res[0] : sh.res[1];
                hzz += flip ? -x : x;
            }
            if (want_shots && tid == 0) tile_sums[ti] = sh.res[0];
        }
        if (lds_tile) {
            if (!resident) {
                if (active) tile_write<R>(t, v, tid, nb);
                __syncthreads();
            }
            if (want_x && active) {
                // the thread bits' qubits, four at a time; a last set that
                // overlaps counts its new bits only
#pragma unroll
                for (int s = 0; s < 2; s++) {
                    const int b = 4 * s < tb - 4 ? 4 * s : tb - 4;
                    if (4 * s >= tb || b < 0) continue;
                    V w[16];
                    tile_read<R>(t, w, tid, b);
                    observe_x<V>(w, xs[1 + s]);
                }
                if (tb > 0 && tb < 4) {   // fewer than four thread bits: pairs straight from LDS
#pragma unroll
                    for (int q = 0; q < 3; q++) {
                        if (q >= tb) break;
                        double s = 0.0;
                        for (int j = 0; j < 16; j++) {
                            const int l = tid + threads * j;
                            if ((l >> q) & 1) continue;
                            const cplx_t<R> a = t[lds_slot<(int)sizeof(V)>(l)], b = t[lds_slot<(int)sizeof(V)>(l | (1 << q))];
                            s += fmar((double)a.x, (double)b.x, (double)a.y * (double)b.y);
                        }
                        xs[1][q] += s + s;
                    }
                }
            }
            if (npauli > 0)
                measure_pauli_tile<R>(sh, lds, resident ? 1 << n : 1 << nb, ti << nb, slot, terms + I.pauli_offset,
                                      npauli, pauli_out);
            __syncthreads();   // before the next tile is written
        }
    }
    // values of the circuit as per-thread terms, reduced over the block
    {
        const int xb = 1 + n + nzz, nv = xb + n;
        const int lane = tid & 63, wave = tid >> 6;
        auto put = [&](int k, double x) {
            const double s = wsum(x);
            if (lane == 0) sh.red[wave][k] = s;
        };
        put(0, acc.tot);
        for (int q = 0; q < n && q < nb; q++) {
            if (!(I.flags & BF_Z)) break;
            double x = 0.0;
            if (q < tb) x = ((tid >> q) & 1) ? acc.tot : 0.0;
            else
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (q - tb == i) x = acc.reg[i];
            put(1 + q, x);
        }
        if (zz)
            for (int q = 0; q + 1 < n && q + 1 < nb; q++) {
                double x = 0.0;
                if (q + 1 < tb) x = (((tid >> q) ^ (tid >> (q + 1))) & 1) ? -acc.tot : acc.tot;
                else if (q + 1 == tb) x = ((tid >> q) & 1) ? -acc.link : acc.link;
                else
#pragma unroll
                    for (int i = 0; i < 3; i++)
                        if (q - tb == i) x = acc.rzz[i];
                put(1 + n + q, x);
            }
        // already block sums, one per thread: three of the four rows hold 0
        if (tid < nhigh)
            for (int w = 0; w < NW; w++) sh.red[w][1 + nb + tid] = w ? 0.0 : hi;
        if (tid >= 64 && tid < 64 + nhigh)
            for (int w = 0; w < NW; w++) sh.red[w][1 + n + nb - 1 + (tid - 64)] = w ? 0.0 : hzz;
        if (want_x) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (tb + i < n) put(xb + tb + i, xs[0][i]);
            const int b1 = tb > 4 ? tb - 4 : 0;   // first bit of the second set
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if (i < tb && i < n) put(xb + i, xs[1][i]);
                if (tb > 4 && b1 + i >= 4 && b1 + i < n) put(xb + b1 + i, xs[2][i]);
            }
        }
        __syncthreads();
        // slots that no flag asked for hold 0
        const int nvis = nhigh && want_x ? xb + nb : nv;   // <X> above the tile follows
        for (int k = tid; k < nvis; k += NT) {
            const bool on = k == 0 || (k < 1 + n ? (I.flags & BF_Z) != 0 : k < xb ? zz : want_x);
            double s = 0.0;
            if (on)
                for (int w = 0; w < NW; w++) s += sh.red[w][k];
            obs[I.obs_offset + k] = s;
        }
        __syncthreads();
    }
    // ---- <X> of the qubits above the low tile: tiles that keep the lowest
    // four qubits (runs of 64 bytes or more) and take nb - 4 of the others ----
    if (want_x && nhigh) {
        const int xb = 1 + n + nzz, step = nb - 4;
        for (int q0 = nb; q0 < n; q0 += step) {
            const int top = q0 + step <= n ? q0 : n - step;   // the set's first qubit after the lowest four
            BatchTile bt;
            constexpr uint32_t B = (uint32_t)sizeof(cplx_t<R>);
            bt.tid = ((uint32_t)(tid & 15) | ((uint32_t)((tid & (threads - 1)) >> 4) << top)) * B;
#pragma unroll
            for (int i = 0; i < 4; i++) bt.reg[i] = B << (top + nb - 8 + i);
            double x0[4] = {}, x1[4] = {};
            for (uint64_t ti = 0; ti < ntiles; ti++) {
                const uint64_t base = ((ti & ((1ull << (top - 4)) - 1)) << 4) | ((ti >> (top - 4)) << (top + step));
                V v[16];
                batch_load<R>(slot, bt, (uint32_t)base * B, v);
                if (active) observe_x<V>(v, x0);       // tile bits nb-4 .. nb-1
                if (nb >= 9) {                         // tile bits nb-8 .. nb-5 (those above the lowest four count)
                    if (active) tile_write<R>(t, v, tid, nb);
                    __syncthreads();
                    if (active) {
                        V w[16];
                        tile_read<R>(t, w, tid, nb - 8);
                        observe_x<V>(w, x1);
                    }
                    __syncthreads();
                }
            }
            double x8[8];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                x8[i] = x0[i];
                x8[4 + i] = x1[i];
            }
            block_reduce(sh, x8, 8, sh.res);
            if (tid < 8) {
                const int b = tid < 4 ? nb - 4 + tid : nb - 8 + (tid - 4);   // tile bit
                const int qq = top + b - 4;                                    // its qubit
                if (b >= 4 && qq >= q0 && (tid < 4 || nb >= 9)) obs[I.obs_offset + xb + qq] = sh.res[tid];
            }
            __syncthreads();
        }
    }

    // ---- shots: first index with u < cdf_i, else the last nonzero ----
    if (!want_shots) return;
    double *cdf = (double *)sh.tile;
    const int T = resident ? 1 << n : 1 << nb;
    if (resident) {
        double pv[16];
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const int l = tid + threads * j;
            pv[j] = active && l < T ? p2<R>(t[lds_slot<(int)sizeof(V)>(l)]) : 0.0;
        }
        if (tid == 0) sh.last_nz = -1;
        __syncthreads();   // the amplitudes are read before the CDF takes their place
        int mylast = -1;
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const int l = tid + threads * j;
            if (!active || l >= T) continue;
            cdf[cdf_at(l)] = pv[j];
            if (pv[j] > 0.0) mylast = l;
        }
        if (mylast >= 0) atomicMax(&sh.last_nz, mylast);
        __syncthreads();
        lds_scan(sh, cdf, T, 0.0);
        const int fallback = sh.last_nz < 0 ? 0 : sh.last_nz;
        for (int s = tid; s < I.num_shots; s += NT) {
            const int l = cdf_find(cdf, T, draws[I.draw_offset + s]);
            outcomes[I.out_offset + s] = (uint64_t)(l < T ? l : fallback);
        }
        __syncthreads();
        return;
    }
    // global state: tile prefix in place over tile_sums[ntiles .. 2 ntiles)
    double *incl = tile_sums + ntiles;
    if (tid == 0) {
        double run = 0.0;
        for (uint64_t i = 0; i < ntiles; i++) {
            run += tile_sums[i];
            incl[i] = run;
        }
    }
    __syncthreads();
    // Each shot's slot holds, until it is resolved, a mark and the tile it is
    // looked for in: first the one the prefix names, the next one when
    // rounding leaves its draw past that tile's own sums.
    constexpr uint64_t kMark = 1ull << 63;
    uint64_t *oc = outcomes + I.out_offset;
    for (int s = tid; s < I.num_shots; s += NT) {
        const double u = draws[I.draw_offset + s];
        uint64_t lo = 0, hi = ntiles;
        while (lo < hi) {
            const uint64_t mid = (lo + hi) >> 1;
            if (u < incl[mid]) hi = mid;
            else lo = mid + 1;
        }
        oc[s] = kMark | lo;
    }
    for (uint64_t ti = 0; ti < ntiles; ti++) {
        int mine = 0;
        for (int s = tid; s < I.num_shots; s += NT) mine |= oc[s] == (kMark | ti);
        // any thread's (a flag of the kernel's own: the library's reduction
        // over the workgroup keeps its LDS address in a register across the
        // whole measurement, one more for this kernel to spill, and in one
        // build it was set where no lane was active)
        if (tid == 0) sh.next = 0;
        __syncthreads();
        if (mine) sh.next = 1;
        __syncthreads();
        const int any = sh.next;
        __syncthreads();
        if (!any) continue;
        for (int l = tid; l < T; l += NT) cdf[cdf_at(l)] = p2<R>(slot[(ti << nb) | (uint64_t)l]);
        __syncthreads();
        lds_scan(sh, cdf, T, ti ? incl[ti - 1] : 0.0);
        for (int s = tid; s < I.num_shots; s += NT) {
            if (oc[s] != (kMark | ti)) continue;
            const int l = cdf_find(cdf, T, draws[I.draw_offset + s]);
            oc[s] = l < T ? (ti << nb) | (uint64_t)l : kMark | (ti + 1);
        }
        __syncthreads();
    }
    for (int s = tid; s < I.num_shots; s += NT) {
        if (!(oc[s] & kMark)) continue;
        // u >= total mass: the last index with nonzero probability
        uint64_t last = 0;
        for (uint64_t ti = ntiles; ti-- > 0;) {
            if (tile_sums[ti] > 0.0) {
                for (int l = T - 1; l >= 0; l--)
                    if (p2<R>(slot[(ti << nb) | (uint64_t)l]) > 0.0) {
                        last = (ti << nb) | (uint64_t)l;
                        break;
                    }
                break;
            }
        }
        oc[s] = last;
    }
    __syncthreads();
}

// One precision per launch: a kernel with both interpreters (42 KiB each)
// would put the ends of the queue loop further apart than a branch reaches.
template <typename R>
__global__ __launch_bounds__(NT, 2) void k_batch(const BInst *__restrict__ insts, const int32_t *__restrict__ order,
                                                 int ninst, int *__restrict__ counter,
                                                 const FPass *__restrict__ passes, const FOp *__restrict__ prog,
                                                 double2 *__restrict__ scratch, uint64_t slot_amps,
                                                 double2 *__restrict__ own, double *__restrict__ tile_scratch, uint64_t tile_slot,
                                                 const double *__restrict__ draws, double *__restrict__ obs,
                                                 uint64_t *__restrict__ outcomes, const PauliT *__restrict__ terms,
                                                 void *__restrict__ state_out)
{
    __shared__ Shared sh;
    double2 *slot = scratch + (uint64_t)blockIdx.x * slot_amps;
    double *ts = tile_scratch + (uint64_t)blockIdx.x * tile_slot;
    for (;;) {
        if (threadIdx.x == 0) sh.next = atomicAdd(counter, 1);
        __syncthreads();
        // every lane read the same queue slot: make that explicit, so the
        // instance and its passes are fetched with scalar (wave-uniform) loads
        const int k = __builtin_amdgcn_readfirstlane(sh.next);
        __syncthreads();
        if (k >= ninst) break;
        BInst I;
        const FConst<uint32_t> src = (FConst<uint32_t>)(uintptr_t)(insts + *(FConst<int32_t>)(uintptr_t)(order + k));
#pragma unroll
        for (int w = 0; w < (int)(sizeof I / sizeof(uint32_t)); w++) ((uint32_t *)&I)[w] = src[w];
        run_circuit<R>(sh, MLX_FRAME_LDS(sh.tile), I, passes, prog, slot, own, ts, draws, obs, outcomes, terms, state_out);
        __syncthreads();
    }
}

__global__ void k_reset_counter(int *c) { c[threadIdx.x] = 0; }

// One cache-blocked pass over a large state: each workgroup streams tiles of
// 2^P.nbits amplitudes through LDS and applies the pass's ops there.  The
// next tile's loads are issued before the current tile's ops run, and the
// barriers order LDS only, so loads, LDS work and the previous tile's stores
// overlap.  NT: streaming accesses (runs are >= 16 amplitudes, whole lines).
template <typename R, bool NT, int THREADS, int TB>
__global__ __launch_bounds__(THREADS) void k_tile_pass(cplx_t<R> *__restrict__ a, BPass P,
                                                       const BOp *__restrict__ ops, uint64_t ntiles)
{
    constexpr int PER = (1 << TB) / THREADS;
    static_assert(PER >= 1 && (1 << TB) / 64 <= 64, "tile shape");
    __shared__ cplx_t<R> t[1 << TB];
    __shared__ uint64_t dlo[64], dhi[64];
    const int tid = threadIdx.x;
    const int T = 1 << P.nbits;   // P.nbits <= TB (checked by the launcher)
    if (tid < 128) {
        const int j = tid & 63, hi = tid >> 6;
        uint64_t o = 0;
        for (int b = 0; b < 6; b++) {
            const int qi = hi * 6 + b;
            if (qi < P.nbits && ((j >> b) & 1)) o |= 1ull << P.qubits[qi];
        }
        if (hi) dhi[j] = o;
        else dlo[j] = o;
    }
    __syncthreads();
    // thread tid moves tile amplitudes l = tid + THREADS i (l % 64 = tid % 64)
    const uint64_t lo = dlo[tid & 63];
    const int hi0 = tid >> 6;
    constexpr int HSTEP = THREADS / 64;
    cplx_t<R> pre[PER];
    uint64_t ti = blockIdx.x;
    if (ti < ntiles) {
        const uint64_t base = tile_base(ti, P) | lo;
#pragma unroll
        for (int i = 0; i < PER; i++)
            if (tid + THREADS * i < T) pre[i] = ld<NT>(&a[base | dhi[hi0 + HSTEP * i]]);
    }
    for (; ti < ntiles; ti += gridDim.x) {
#pragma unroll
        for (int i = 0; i < PER; i++)
            if (tid + THREADS * i < T) t[tid + THREADS * i] = pre[i];
        lds_barrier();
        const uint64_t nti = ti + gridDim.x;
        if (nti < ntiles) {
            const uint64_t nbase = tile_base(nti, P) | lo;
#pragma unroll
            for (int i = 0; i < PER; i++)
                if (tid + THREADS * i < T) pre[i] = ld<NT>(&a[nbase | dhi[hi0 + HSTEP * i]]);
        }
        const uint64_t base = tile_base(ti, P);
        run_pass_ops<R, THREADS, kSegRegsPass, true>(t, T, ops + P.first_op, P.num_ops, base);
#pragma unroll
        for (int i = 0; i < PER; i++)
            if (tid + THREADS * i < T) st<NT>(&a[(base | lo) | dhi[hi0 + HSTEP * i]], t[tid + THREADS * i]);
        lds_barrier();   // every thread has read its write-back values before the next tile lands
    }
}

// Persistent grid of one resident wave of workgroups for this instantiation.
template <typename R, bool NT, int THREADS, int TB>
hipError_t run_tile_pass(void *amps, const BPass &P, const BOp *d_ops, uint64_t ntiles, int cus, hipStream_t st)
{
    static std::atomic<int> per_cu_cached{0};
    int per_cu = per_cu_cached.load(std::memory_order_relaxed);
    if (!per_cu) {
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_tile_pass<R, NT, THREADS, TB>, THREADS, 0) !=
                hipSuccess ||
            per_cu < 1)
            per_cu = 1;
        per_cu_cached.store(per_cu, std::memory_order_relaxed);
    }
    const uint64_t want = (uint64_t)cus * (uint64_t)per_cu;
    const unsigned grid = (unsigned)(ntiles < want ? ntiles : want);
    k_tile_pass<R, NT, THREADS, TB><<<grid, THREADS, 0, st>>>((cplx_t<R> *)amps, P, d_ops, ntiles);
    return hipGetLastError();
}

template <typename R, bool NT>
hipError_t tile_pass_shape(void *amps, const BPass &P, const BOp *d_ops, uint64_t ntiles, int cus, int threads,
                           int tb, hipStream_t st)
{
    if (tb <= 11) {
        if (threads <= 256) return run_tile_pass<R, NT, 256, 11>(amps, P, d_ops, ntiles, cus, st);
        return run_tile_pass<R, NT, 512, 11>(amps, P, d_ops, ntiles, cus, st);
    }
    if (threads <= 256) return run_tile_pass<R, NT, 256, 12>(amps, P, d_ops, ntiles, cus, st);
    return run_tile_pass<R, NT, 512, 12>(amps, P, d_ops, ntiles, cus, st);
}

}  // namespace

// One pass of the single-state blocked path; tile_bits (11 or 12) is the
// LDS tile the kernel is built for (>= P.nbits), threads its workgroup size.
hipError_t launch_tile_pass(void *amps, int prec, int n, const BPass &P, const BOp *d_ops, int cus, int threads,
                            int tile_bits, hipStream_t st)
{
    if (P.nbits > tile_bits || tile_bits > kBatchMaxTileBits) return hipErrorInvalidValue;
    const uint64_t ntiles = 1ull << (n - P.nbits);
    const bool nt = ((1ull << n) * (prec == 1 ? 8ull : 16ull)) >= gate_tuning().nt_min_bytes;
    if (prec == 1)
        return nt ? tile_pass_shape<float, true>(amps, P, d_ops, ntiles, cus, threads, tile_bits, st)
                  : tile_pass_shape<float, false>(amps, P, d_ops, ntiles, cus, threads, tile_bits, st);
    return nt ? tile_pass_shape<double, true>(amps, P, d_ops, ntiles, cus, threads, tile_bits, st)
              : tile_pass_shape<double, false>(amps, P, d_ops, ntiles, cus, threads, tile_bits, st);
}

hipError_t launch_batch_pass(int prec, const BInst *insts, const int32_t *list, const int32_t *first_tile, int count,
                             int level, int tiles, const FPass *passes, const FOp *prog, double2 *own, hipStream_t st)
{
    auto go = [&](auto kernel) {
        kernel<<<tiles, NT, 0, st>>>(insts, list, first_tile, count, level, passes, prog, own);
    };
    go(prec == MOONLAB_HIP_C64 ? k_batch_pass<float> : k_batch_pass<double>);
    return hipGetLastError();
}

hipError_t launch_batch_pauli(int prec, const BInst *insts, const int32_t *list, const int32_t *first, int count,
                              int groups, const PauliT *terms, const double2 *own, double *obs, hipStream_t st)
{
    auto go = [&](auto kernel) { kernel<<<groups, NT, 0, st>>>(insts, list, first, count, terms, own, obs); };
    go(prec == MOONLAB_HIP_C64 ? k_batch_pauli<float> : k_batch_pauli<double>);
    return hipGetLastError();
}

hipError_t launch_reset_counters(int *counters, hipStream_t st)
{
    k_reset_counter<<<1, 2, 0, st>>>(counters);
    return hipGetLastError();
}

// order: `count` circuits of one precision; counter: their queue head; grid:
// workgroups at most, with a slot and tile sums each.
hipError_t launch_batch(int prec, const BInst *insts, const int32_t *order, int count, int *counter, const FPass *passes,
                        const FOp *prog, double2 *scratch, uint64_t slot_amps, double2 *own, double *tile_scratch,
                        uint64_t tile_slot, const double *draws, double *obs, uint64_t *outcomes,
                        const PauliT *terms, void *state_out, int grid, hipStream_t st)
{
    auto go = [&](auto kernel) {
        kernel<<<count < grid ? count : grid, NT, 0, st>>>(insts, order, count, counter, passes, prog, scratch, slot_amps,
                                                           own, tile_scratch, tile_slot, draws, obs, outcomes, terms,
                                                           state_out);
    };
    go(prec == MOONLAB_HIP_C64 ? k_batch<float> : k_batch<double>);
    return hipGetLastError();
}

}  // namespace mlx
