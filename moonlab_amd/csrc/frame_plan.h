// frame_plan.h -- host planner of the Pauli-rotation engine.
#pragma once

#include <stdint.h>

#include <complex>
#include <vector>

#include "../../include/moonlab_hip_statevec.h"
#include "frame_program.h"

namespace mlx {

enum FGateKind : int8_t { FG_ROT, FG_CX, FG_CZ, FG_SWAP, FG_X, FG_Z };

// A lowered gate: a rotation scale (1 - i t P), P = i^|x&z| X^x Z^z, or a
// frame gate (CX: control a, target b; CZ, SWAP: a, b; X, Z: a).
struct FGate {
    FGateKind kind;
    int8_t    a, b;
    uint64_t  x, z;
    double    t, scale;
};

// What a gate's parameters make of a state: PARAMS_FINITE, or, where one that
// the gate reads is not finite, NaN in every amplitude or in those of one
// value of a qubit only (phases, controlled rotations, a U3 with its theta
// finite).
enum GateParams : int8_t { PARAMS_FINITE, PARAMS_SPOIL_ALL, PARAMS_SPOIL_PART };
GateParams gate_params(const moonlab_hip_gate_t &g);

// Gate list -> rotations and frame gates, and the global phase they leave
// out.  False on an invalid gate or qubit, or, unless any_angle, a parameter
// that is not finite (whose rotation would reach every amplitude).
bool frame_lower(const moonlab_hip_gate_t *g, int ng, int n, std::vector<FGate> &out, std::complex<double> &phase,
                 bool any_angle = false);

// Seeds per tile set and register basis of the batch engine's plans.
constexpr int kBatchLookahead = 0;

// Plan passes over tile sets of tb qubits (n <= tb: one pass over max(n, 4)
// qubits) that keep the lowest anchor_bits qubits.  amp_bytes: 16 or 8.
// lookahead: seeds per tile set and register basis (0: greedy).  Passes and
// units are appended.
void frame_plan(const std::vector<FGate> &gates, std::complex<double> phase, int n, int tb, int anchor_bits,
                int amp_bytes, int lookahead, std::vector<FPass> &passes, std::vector<FOp> &prog);

}  // namespace mlx
