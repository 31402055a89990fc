// frame_device.h -- device side of the Pauli-rotation engine
// (frame_program.h): 16 tile amplitudes per thread in registers, rotations
// on them, LDS only to change the layout.
#pragma once

#include <hip/hip_runtime.h>

#include "frame_program.h"
#include "sv_device.h"

namespace mlx {

// the fields of one rotation, fetched by one scalar load
struct FHead {
    int32_t  arm;
    uint32_t zt;
    uint64_t zg;
    double   t;
    float    tf;
};

__device__ __forceinline__ FHead frame_head(const FOp *o)
{
    return FHead{o->arm, o->zt, o->zg, o->t, o->tf};
}

// p, with an address that depends on `arm` (never negative): a fetch from it
// issues only once `arm` has arrived, so the wait before a rotation does not
// include the fetch of the one after it
__device__ __forceinline__ const FOp *after(const FOp *p, int32_t arm) { return p + (arm >> 31); }

__device__ __forceinline__ double frame_t(const FHead &h, uint32_t flip, double)
{
    return __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, h.t) ^ ((uint64_t)flip << 32));
}
__device__ __forceinline__ float frame_t(const FHead &h, uint32_t flip, float)
{
    return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, h.tf) ^ flip);
}

__device__ __forceinline__ float fmad(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fmad(double a, double b, double c) { return __builtin_fma(a, b, c); }

// sign functional index 0..7 of an arm with direction d -> 4-bit mask
constexpr int frame_zr(int d, int rest, int own)
{
    return (rest & ((1 << d) - 1)) | ((rest >> d) << (d + 1)) | (own << d);
}
constexpr bool frame_par(int x) { return ((x ^ (x >> 1) ^ (x >> 2) ^ (x >> 3)) & 1) != 0; }

// y = a - i t s b on the pairs across register bit D (rotation about a string
// with an even number of Ys)
template <typename R, int D, int ZR>
__device__ __forceinline__ void farm_x(const cplx_t<R> (&in)[16], cplx_t<R> (&out)[16], R t)
{
#pragma unroll
    for (int j = 0; j < 16; j++) {
        const R s = frame_par(ZR & j) ? -t : t;
        const cplx_t<R> a = in[j], b = in[j ^ (1 << D)];
        out[j].x = fmad(s, b.y, a.x);
        out[j].y = fmad(-s, b.x, a.y);
    }
}

// y = a + t s b, s opposite on the two values of a pair (odd number of Ys)
template <typename R, int D, int ZR>
__device__ __forceinline__ void farm_y(const cplx_t<R> (&in)[16], cplx_t<R> (&out)[16], R t)
{
#pragma unroll
    for (int j = 0; j < 16; j++) {
        const R s = frame_par(ZR & j) ? -t : t;
        const cplx_t<R> a = in[j], b = in[j ^ (1 << D)];
        out[j].x = fmad(s, b.x, a.x);
        out[j].y = fmad(s, b.y, a.y);
    }
}

// y = a (1 - i t s) (diagonal string)
template <typename R, int ZR>
__device__ __forceinline__ void farm_z(const cplx_t<R> (&in)[16], cplx_t<R> (&out)[16], R t)
{
#pragma unroll
    for (int j = 0; j < 16; j++) {
        const R s = frame_par(ZR & j) ? -t : t;
        const cplx_t<R> a = in[j];
        out[j].x = fmad(s, a.y, a.x);
        out[j].y = fmad(-s, a.x, a.y);
    }
}

// One rotation from one register set into another.  Every value is written by
// its arm (two FMAs), so the loop that alternates the sets needs no copies.
template <typename R>
__device__ __forceinline__ void frame_op(const cplx_t<R> (&in)[16], cplx_t<R> (&out)[16], const FHead &h, uint32_t tid,
                                         uint64_t base)
{
    const uint32_t flip = ((uint32_t)__popc(h.zt & tid) ^ (uint32_t)__popcll(h.zg & base)) << 31;
    const R t = frame_t(h, flip, R(0));
#define MLX_FARM_X(D, K) case FARM_X + 8 * D + K: farm_x<R, D, frame_zr(D, K, 0)>(in, out, t); break;
#define MLX_FARM_Y(D, K) case FARM_Y + 8 * D + K: farm_y<R, D, frame_zr(D, K, 1)>(in, out, t); break;
#define MLX_FARM_8(M, D) M(D, 0) M(D, 1) M(D, 2) M(D, 3) M(D, 4) M(D, 5) M(D, 6) M(D, 7)
#define MLX_FARM_Z(K) case FARM_Z + K: farm_z<R, K>(in, out, t); break;
    switch (h.arm) {
        MLX_FARM_8(MLX_FARM_X, 0)
        MLX_FARM_8(MLX_FARM_X, 1)
        MLX_FARM_8(MLX_FARM_X, 2)
        MLX_FARM_8(MLX_FARM_X, 3)
        MLX_FARM_8(MLX_FARM_Y, 0)
        MLX_FARM_8(MLX_FARM_Y, 1)
        MLX_FARM_8(MLX_FARM_Y, 2)
        MLX_FARM_8(MLX_FARM_Y, 3)
        MLX_FARM_Z(0) MLX_FARM_Z(1) MLX_FARM_Z(2) MLX_FARM_Z(3) MLX_FARM_Z(4) MLX_FARM_Z(5) MLX_FARM_Z(6) MLX_FARM_Z(7)
        MLX_FARM_Z(8) MLX_FARM_Z(9) MLX_FARM_Z(10) MLX_FARM_Z(11) MLX_FARM_Z(12) MLX_FARM_Z(13) MLX_FARM_Z(14)
        MLX_FARM_Z(15)
    default:   // FARM_SCALE
#pragma unroll
        for (int j = 0; j < 16; j++) {
            out[j].x = t * in[j].x;
            out[j].y = t * in[j].y;
        }
        break;
    }
#undef MLX_FARM_X
#undef MLX_FARM_Y
#undef MLX_FARM_8
#undef MLX_FARM_Z
}

// thread bits spread over the index bits that are no pivots
__device__ __forceinline__ int frame_thread_index(uint32_t pivots, int tid)
{
    int x = tid;
#pragma unroll
    for (int i = 0; i < kFrameRegBits; i++) {
        const int p = (int)((pivots >> (5 * i)) & 31u);
        x = ((x >> p) << (p + 1)) | (x & ((1 << p) - 1));
    }
    return x;
}

// What a thread keeps over the tiles of a pass: the output layout's LDS
// address and its word of the sign table.
struct FrameThread {
    uint32_t out_slot;
    uint32_t sign;
};

__device__ __forceinline__ FrameThread frame_thread(const FPass &P, const FOp *prog, int tid, int tbits, bool active)
{
    FrameThread f{0, 0};
    if (P.flags & FP_OUT) {
        const FOut *o = (const FOut *)(prog + P.out);
        for (int b = 0; b < tbits; b++) f.out_slot ^= ((tid >> b) & 1) ? o->col[b] : 0u;
    }
    if (P.table >= 0 && active) f.sign = ((const uint16_t *)(prog + P.table))[tid];
    return f;
}

// The phases of a pass on one tile, then the signs, the scale and the output
// layout: v enters and leaves in the IO layout (register bits = top four tile
// bits).  Every thread of the workgroup calls it (barriers); threads that
// hold no amplitudes (tid >= 2^(nbits-4)) have active = false.
template <typename R, bool ALL>
__device__ __forceinline__ void frame_tile(cplx_t<R> *lds, cplx_t<R> (&v)[16], const FPass &P, const FOp *prog,
                                           const FrameThread &ft, uint64_t base, int tid, int nbits, bool active)
{
    constexpr int B = (int)sizeof(cplx_t<R>);
    char *lb = (char *)lds;
    uint32_t slot = (uint32_t)lds_slot<B>(tid) * B;   // of the thread's value 0 in the current layout
    uint32_t off[16];
#pragma unroll
    for (int j = 0; j < 16; j++) off[j] = (uint32_t)lds_slot<B>(j << (nbits - kFrameRegBits)) * B;
    const FOp *p = prog + P.first;
    cplx_t<R> w[16];
    for (int ph = 0; ph < P.nphases; ph++) {
        const FPhase *h = (const FPhase *)p;
        const int cnt = h->nops;
        p += 3;
        FHead h0 = frame_head(p);
        if (h->relayout) {
            uint32_t to[16];
#pragma unroll
            for (int j = 0; j < 16; j++) to[j] = h->off[j];
            if (ALL || active) {
#pragma unroll
                for (int j = 0; j < 16; j++) *(cplx_t<R> *)(lb + (slot ^ off[j])) = v[j];
            }
            lds_barrier();
            slot = (uint32_t)lds_slot<B>(frame_thread_index(h->pivots, tid)) * B;
            if (ALL || active) {
#pragma unroll
                for (int j = 0; j < 16; j++) v[j] = *(const cplx_t<R> *)(lb + (slot ^ to[j]));
            }
#pragma unroll
            for (int j = 0; j < 16; j++) off[j] = to[j];
        }
        // the unit after a phase's last rotation is the next phase's header
        // or a later unit of the program (one spare unit ends it): fetched, not run
        for (int q = 1; q <= cnt; q += 2) {
            const FHead h1 = frame_head(after(p + 1, h0.arm));
            frame_op<R>(v, w, h0, (uint32_t)tid, base);
            if (q < cnt) {
                h0 = frame_head(after(p + 2, h1.arm));
                frame_op<R>(w, v, h1, (uint32_t)tid, base);
            } else {
#pragma unroll
                for (int j = 0; j < 16; j++) v[j] = w[j];
            }
            p += 2;
        }
        if (cnt & 1) p -= 1;
    }
    if (P.flags & (FP_SIGN | FP_SCALE | FP_CSCALE)) {
        uint32_t s = ft.sign;
        for (int c = 0; c < P.ncross; c++) {
            const FCross *x = (const FCross *)(prog + P.cross) + c;
            const uint32_t a = (uint32_t)__popcll(x->ga & base) & 1u, b = (uint32_t)__popcll(x->gb & base) & 1u;
            const uint32_t fa = x->wa ^ (0u - ((uint32_t)__popc(x->ta & tid) & 1u));
            const uint32_t fb = x->wb ^ (0u - ((uint32_t)__popc(x->tb & tid) & 1u));
            s ^= (a ? fb : 0u) ^ (b ? fa : 0u) ^ (a & b ? 0xFFFFu : 0u);
        }
        const R sr = (R)P.scale_r, si = (R)P.scale_i;
        const bool cplx = (P.flags & FP_CSCALE) != 0;
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const bool neg = (s >> j) & 1u;
            const R r = neg ? -sr : sr;
            if (cplx) {
                v[j] = cmul(v[j], r, neg ? -si : si);
            } else {
                v[j].x *= r;
                v[j].y *= r;
            }
        }
    }
    if (P.flags & FP_OUT) {
        const FOut *o = (const FOut *)(prog + P.out);
        uint32_t to[16];
#pragma unroll
        for (int j = 0; j < 16; j++) to[j] = o->off[j];
        if (ALL || active) {
#pragma unroll
            for (int j = 0; j < 16; j++) *(cplx_t<R> *)(lb + (slot ^ off[j])) = v[j];
        }
        uint32_t os = ft.out_slot;
        for (int c = 0; c < P.nshift; c++) {
            const FShift *x = (const FShift *)(prog + P.shift) + c;
            os ^= (__popcll(x->gmask & base) & 1) ? x->off : 0u;
        }
        lds_barrier();
        if (ALL || active) {
#pragma unroll
            for (int j = 0; j < 16; j++) v[j] = *(const cplx_t<R> *)(lb + (os ^ to[j]));
        }
        // Between two changes a thread writes only slots that it alone has
        // read; the output's permutation breaks that, so nothing is written
        // (by the next tile) before every thread has read.
        lds_barrier();
    }
}

}  // namespace mlx
