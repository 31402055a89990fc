// sv_frame.hip -- passes of the Pauli-rotation engine over one state
// (moonlab_hip_apply_gates_blocked; program format and lowering:
// frame_program.h, frame_plan.cpp).
//
// Reference counterpart: the per-gate loops of src/quantum/gates.c:123-1048;
// here a pass reads and writes the state once for many gates.
#include <hip/hip_runtime.h>

#include "frame_device.h"
#include "sv_internal.h"

namespace mlx {
namespace {

// One pass: a workgroup of 2^(TB-4) threads streams tiles of 2^TB amplitudes.
// Tiles enter and leave in the IO layout (lanes over the low tile bits: runs
// of contiguous amplitudes); the next tile's loads are issued before the
// current tile's rotations.  Bound by latency: two waves per SIMD (complex128;
// registers and LDS hold no more) between loads, layout changes and rotations.
// A 30-qubit complex128 pass of 27 rotations takes 8.3 ms, 4.1 TB/s, with the
// vector ALUs at 36 % and LDS at 28 %; the register-phase engine's took 15.5.
// Its parts alone: an empty pass 5.5-6.5 ms, a rotation 0.076 ms (72 % of the
// FP64 rate), a change of layout 0.27-0.4 ms.
template <typename R, bool NT, int TB, int WPE>
__global__ __launch_bounds__(1 << (TB - 4), WPE) void k_frame_pass(cplx_t<R> *__restrict__ a, const FPass *__restrict__ pass,
                                                                   const FOp *__restrict__ prog, uint64_t ntiles)
{
    constexpr int THREADS = 1 << (TB - 4), HSTEP = THREADS / 64, NHI = 1 << (TB - 6);
    __shared__ cplx_t<R> t[1 << TB];
    __shared__ uint64_t dlo[64], dhi[NHI];
    const int tid = threadIdx.x;
    const FConst<FPass> P = (FConst<FPass>)(uintptr_t)pass;
    const uint64_t mask = P->mask;
    for (int e = tid; e < 64 + NHI; e += THREADS) {
        if (e < 64) dlo[e] = frame_deposit((uint64_t)e, mask);
        else dhi[e - 64] = frame_deposit((uint64_t)(e - 64) << 6, mask);
    }
    __syncthreads();
    const uint64_t lo = dlo[tid & 63];
    const int hi0 = tid >> 6;
    const FrameThread ft = frame_thread(P, prog, tid, TB - 4, true);
    typename FVec<R>::t v[16], pre[16];
    const TileWalk walk = tile_walk(ntiles);
    uint64_t ti = walk.t;
    uint64_t base = frame_uniform(frame_deposit(ti, ~mask));
    const uint64_t step = frame_uniform(frame_deposit(walk.step, ~mask));
    if (ti < walk.end) {
#pragma unroll
        for (int j = 0; j < 16; j++) pre[j] = frame_ld<R, NT>(&a[(base | lo) | dhi[hi0 + HSTEP * j]]);
    }
    for (; ti < walk.end; ti += walk.step) {
#pragma unroll
        for (int j = 0; j < 16; j++) v[j] = pre[j];
        const uint64_t next = frame_step(base, step, mask);
        if (ti + walk.step < walk.end) {
#pragma unroll
            for (int j = 0; j < 16; j++) pre[j] = frame_ld<R, NT>(&a[(next | lo) | dhi[hi0 + HSTEP * j]]);
        }
        frame_tile<R>(MLX_FRAME_LDS(t), v, P, prog, ft, base, tid, TB);
#pragma unroll
        for (int j = 0; j < 16; j++) frame_st<R, NT>(&a[(base | lo) | dhi[hi0 + HSTEP * j]], v[j]);
        base = next;
    }
}

// A whole state of 4..11 qubits as one tile of one workgroup: a chain of
// rotations, 106 of them on 10 qubits in 60 us where a kernel for each of the
// circuit's 202 gates took 0.8 ms.
template <typename R>
__global__ __launch_bounds__(128) void k_frame_small(cplx_t<R> *__restrict__ a,
                                                     const FPass *__restrict__ pass,
                                                     const FOp *__restrict__ prog)
{
    const FConst<FPass> P = (FConst<FPass>)(uintptr_t)pass;
    __shared__ cplx_t<R> t[1 << 11];
    const int tid = threadIdx.x, threads = 1 << (P->nbits - kFrameRegBits);
    const bool active = tid < threads;
    const FrameThread ft = frame_thread(P, prog, tid, P->nbits - kFrameRegBits, active);
    typename FVec<R>::t v[16];
#pragma unroll
    for (int j = 0; j < 16; j++) v[j] = active ? frame_ld<R, false>(&a[tid + threads * j]) : typename FVec<R>::t{R(0), R(0)};
    frame_tile<R>(MLX_FRAME_LDS(t), v, P, prog, ft, 0, tid, P->nbits);
#pragma unroll
    for (int j = 0; j < 16; j++)
        if (active) frame_st<R, false>(&a[tid + threads * j], v[j]);
}

// Tiles per workgroup: at most 8 (short-lived workgroups that the dispatcher
// keeps refilling stream HBM faster than a resident wave of persistent ones;
// 2, 4, 8, 16 and 32 are within 2 % at 30 qubits), fewer when that leaves
// under 1024 workgroups: 256 CUs hold two each, and with 8 tiles a 20-qubit
// state (256 tiles) ran on 32 of them (12 passes 1.50 ms; 2 tiles 0.68 ms).
constexpr uint64_t kTilesPerGroup = 8, kMinGroups = 1024;

template <typename R, bool NT, int TB>
hipError_t run_frame_pass(void *amps, const FPass *d_pass, const FOp *d_prog, uint64_t ntiles, hipStream_t st)
{
    // complex64: two 512-thread workgroups fit a CU's LDS, 4 waves per SIMD
    // (at most 128 registers); complex128 has 2 waves per SIMD by its LDS
    constexpr int WPE = sizeof(R) == 4 ? 4 : 2;
    uint64_t per = kTilesPerGroup;
    while (per > 1 && ntiles / per < kMinGroups) per >>= 1;
    const unsigned grid = (unsigned)(ntiles / per);
    k_frame_pass<R, NT, TB, WPE><<<grid, 1 << (TB - 4), 0, st>>>((cplx_t<R> *)amps, d_pass, d_prog, ntiles);
    return hipGetLastError();
}

}  // namespace

// One pass over a state of n >= P.nbits qubits (P.nbits 12 or 13, or n itself
// when n is 4..11).  d_pass: the pass on the device; d_prog: the program with
// one spare unit after it.
hipError_t launch_frame_pass(void *amps, int prec, int n, const FPass &P, const FPass *d_pass, const FOp *d_prog,
                             hipStream_t st)
{
    if (n < 12) {
        if (P.nbits != n || n < kFrameRegBits) return hipErrorInvalidValue;
        if (prec == MOONLAB_HIP_C64) k_frame_small<float><<<1, 128, 0, st>>>((float2 *)amps, d_pass, d_prog);
        else k_frame_small<double><<<1, 128, 0, st>>>((double2 *)amps, d_pass, d_prog);
        return hipGetLastError();
    }
    if ((P.nbits != 12 && P.nbits != 13) || n < P.nbits) return hipErrorInvalidValue;
    const uint64_t ntiles = 1ull << (n - P.nbits);
    const bool nt = ((1ull << n) * (prec == MOONLAB_HIP_C64 ? 8ull : 16ull)) >= gate_tuning().nt_min_bytes;
    auto go = [&](auto r) {
        using R = decltype(r);
        if (P.nbits == 13)
            return nt ? run_frame_pass<R, true, 13>(amps, d_pass, d_prog, ntiles, st)
                      : run_frame_pass<R, false, 13>(amps, d_pass, d_prog, ntiles, st);
        return nt ? run_frame_pass<R, true, 12>(amps, d_pass, d_prog, ntiles, st)
                  : run_frame_pass<R, false, 12>(amps, d_pass, d_prog, ntiles, st);
    };
    return prec == MOONLAB_HIP_C64 ? go(float()) : go(double());
}

}  // namespace mlx
