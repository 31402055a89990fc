// frame_program.h -- programs of the Pauli-rotation engine, shared by the
// host planner (frame_plan.cpp) and the kernels (frame_device.h).
//
// A circuit is lowered to Pauli rotations exp(-i theta/2 P) and to CNOT, CZ,
// SWAP, X and Z gates.  The latter never touch an amplitude: inside a pass
// they only change the frame F (a permutation x -> A x + b of the tile
// indices with a sign (-1)^Q(x), Q quadratic) through which the stored
// amplitudes are read, psi = F psi', and a rotation about P acts on the
// stored amplitudes as one about F^-1 P F.  A pass ends by undoing F: the
// signs on the register values, the permutation as the last change of layout.
//
// A rotation with |theta| <= pi/2 (larger angles leave a Pauli to the frame)
// runs unnormalized, 1 - i tan(theta/2) P: two FMAs per amplitude, no
// multiplication by the cosine; the cosines' product is applied once at the
// end of a pass.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "batch_device.h"

namespace mlx {

constexpr int kFrameRegBits = 4;    // register bits of a layout: 16 amplitudes per thread
constexpr int kFrameMaxTileBits = 13;

// Arms of the rotation interpreter.  d = register bit the rotation pairs
// values across, zr = register bits of its sign functional: value j takes the
// sign (-1)^parity(zr & j).
enum FrameArm : int32_t {
    FARM_X = 0,     // + 8 d + (zr without bit d, zr_d = 0): y = a - i t s b
    FARM_Y = 32,    // + 8 d + (zr without bit d, zr_d = 1): y = a + t s b
    FARM_Z = 64,    // + zr: y = a (1 - i t s)
    FARM_SCALE = 80,// y = t a
    FARM_COUNT = 81,
};

// One unit (32 bytes) of a program: a rotation, or part of a phase header or
// of a sign table.
struct FOp {
    int32_t  arm;
    uint32_t zt;        // sign bit: parity(zt & thread) ...
    uint64_t zg;        // ... ^ parity(zg & tile base)
    double   t;
    float    tf;        // (float)t, for complex64
    uint32_t pad;
};
static_assert(sizeof(FOp) == 32, "program unit");

// A phase: a layout of the tile over (register value j, thread t), stored
// index x = R j + T t, and the rotations that run in it.  R's four columns
// are the directions the rotations pair values across; T inserts zeros at the
// four pivot positions p, ascending: x + (x & nm), nm = -(1 << p), per pivot.
// Followed by `nops` >= 1 rotations.  Only a pass's first phase may stay in
// the layout it is entered in (the IO layout).
struct FPhase {
    int32_t  nops;
    int32_t  relayout;
    uint32_t nm[4];
    uint32_t pad[2];
    uint32_t from[16];      // LDS byte offset of register value j before: slot(R_before j)
    uint32_t off[16];       // and in this layout: slot(R j)
};
constexpr int kFPhaseUnits = 5;
static_assert(sizeof(FPhase) == kFPhaseUnits * sizeof(FOp), "phase header units");

// Output layout (after the last phase) when FP_OUT is set.
struct FOut {
    uint32_t from[16];      // LDS byte offset of register value j in the last layout
    uint32_t off[16];       // of output register value j (constant shift included)
    uint32_t col[12];       // of thread bit b
    uint32_t pad[4];
};
constexpr int kFOutUnits = 6;
static_assert(sizeof(FOut) == kFOutUnits * sizeof(FOp), "output layout units");

// parity(gmask & base) shifts the stored index: XOR `off` into the LDS byte
// offset an output value is read from.
struct FShift {
    uint64_t gmask;
    uint32_t off;
    uint32_t pad[5];
};
static_assert(sizeof(FShift) == sizeof(FOp), "shift unit");

// Sign term (fa + a)(fb + b), fa and fb the tile-local parts, a = parity(ga &
// base), b = parity(gb & base): adds a fb + b fa + a b.  fa on value j of
// thread t: bit j of wa, flipped by parity(ta & t).
struct FCross {
    uint64_t ga, gb;
    uint16_t ta, tb;
    uint16_t wa, wb;
    uint32_t pad[2];
};
static_assert(sizeof(FCross) == sizeof(FOp), "cross unit");

enum : int32_t {
    FP_OUT = 1,       // the output layout differs from the last phase's
    FP_SIGN = 2,      // a sign table: 2^(nbits-4) uint16, bit j = sign of value j
    FP_SCALE = 4,     // multiply by scale_r
    FP_CSCALE = 8,    // multiply by scale_r + i scale_i
};

// One pass over the state.  Units: phases first, then FOut, FCross, FShift
// entries and the sign table at the given unit indices (absolute).
struct FPass {
    int32_t  first;
    int32_t  nphases;
    int32_t  nbits;           // tile bits
    int32_t  flags;
    int32_t  out, cross, shift, table;
    int32_t  ncross, nshift;
    double   scale_r, scale_i;
    uint64_t mask;            // the tile's qubits: tile-index bit b is its b-th lowest bit
};

}  // namespace mlx
