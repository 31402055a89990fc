// engine.h -- internal interface of the circuit engine shared by the job API,
// the circuit API and the MI355X backend entry points.
#pragma once

#include <stdint.h>
#include <stdlib.h>

#include <utility>
#include <vector>

#include "../../include/moonlab_hip_statevec.h"
#include "../../include/moonlab_scheduler.h"

namespace mlx {

// One recorded gate of the job / circuit APIs (scheduler.c:40-46,
// moonlab_qgtl_backend.c:29-35): the tag, its qubits and theta.
struct GateRec {
    int    type;
    int    target;
    int    control;
    double theta;
    int    has_param;
    // gates added through moonlab_mi355x_circuit_add_gate_ex (codes 14..24 of
    // the state-vector gate table): second control or target, phi and lambda
    int    extra = -1;
    double phi = 0.0, lam = 0.0;
    int    ext = 0;
};

bool gate_takes_param(int type);   // RX, RY, RZ
bool gate_is_two_qubit(int type);  // CNOT, CY, CZ, SWAP

// Checks the circuit API applies at add time (moonlab_qgtl_backend.c:93-99).
bool gate_rec_valid(const GateRec &g, int num_qubits);

// splitmix64 seed mixer and xorshift64 draw of the job path
// (scheduler.c:143-148, moonlab_qgtl_backend.c:159-167, 238-239).
uint64_t splitmix64(uint64_t x);
double   xorshift_u(uint64_t *s);

// Per-worker shot slicing (scheduler.c:201-236): the uniform draws for all
// shots in slice order.  seed == 0 takes the reference's clock-based seed.
int fill_job_draws(uint64_t seed, int total_shots, int num_workers, std::vector<double> &u);

struct RunRequest {
    int                 num_qubits;
    int                 precision;
    const GateRec      *gates;
    int                 num_gates;
    const double       *draws;          // num_draws uniform values, or nullptr
    int                 num_draws;
    bool                want_amps;
    bool                want_probs;
    bool                want_z;
    int                 fusion_max;     // 0 = unfused
    bool                blocked;        // cache-blocked tile passes
    bool                per_gate = false;   // one kernel per gate, whatever the circuit
    void               *stream = nullptr;   // run on this HIP stream instead of the state's own
};

// Doubles the device writes and the C results hand over (free() releases
// them).  Not cleared, and on 2 MiB pages from 4 MiB up: clearing a vector of
// the 20-qubit amplitudes first took 3 ms, twice what their download takes.
class HostBuf {
  public:
    HostBuf() = default;
    HostBuf(HostBuf &&o) noexcept : p_(o.p_), n_(o.n_) { o.p_ = nullptr, o.n_ = 0; }
    HostBuf &operator=(HostBuf &&o) noexcept
    {
        std::swap(p_, o.p_);
        std::swap(n_, o.n_);
        return *this;
    }
    ~HostBuf() { free(p_); }
    bool    alloc(size_t n);   // false: out of memory
    double *data() const { return p_; }
    size_t  size() const { return n_; }
    double *release()
    {
        double *p = p_;
        p_ = nullptr;
        n_ = 0;
        return p;
    }

  private:
    double *p_ = nullptr;
    size_t  n_ = 0;
};

struct RunResult {
    std::vector<uint64_t> outcomes;
    HostBuf               amps;         // 2 * 2^n (widened for complex64)
    HostBuf               probs;
    std::vector<double>   z;
    double                norm = 0.0;
    double                device_seconds = 0.0;
};

// Run a gate list from |0..0> on a pooled device state.  Returns a
// moonlab_hip_status_t value; the text is in moonlab_hip_last_error().
int run_circuit(const RunRequest &rq, RunResult &rr);
// The same with gates of the full code table (rq.gates is ignored).
int run_circuit_gates(const RunRequest &rq, const moonlab_hip_gate_t *gates, int num_gates, RunResult &rr);

// The gates and seed of a job of this library's own scheduler.  Absent in
// the plugin, whose jobs belong to the host process: there the address is null.
struct JobView {
    uint64_t                    seed;
    const std::vector<GateRec> *gates;
};
__attribute__((weak, visibility("hidden"))) JobView own_job(const moonlab_job_t *job);

}  // namespace mlx
