/* job_stub.c -- test infrastructure: a host scheduler whose jobs are opaque
 * (the pointer is not even an address), for the plugin to read through the
 * public job API (tests/test_plugin_read_cpu.py). */
#include <stdio.h>
#include <string.h>

int dumps = 0;

int moonlab_job_num_qubits(const void *job) { return job == (void *)8 ? 2 : -1; }
int moonlab_job_num_gates(const void *job) { return job == (void *)8 ? 2 : -1; }
int moonlab_job_num_shots(const void *job) { return job == (void *)8 ? 4 : -1; }
int moonlab_job_num_workers(const void *job) { return job == (void *)8 ? 1 : -1; }
int moonlab_register_backend(const void *be) { return be ? 0 : -1; }

int moonlab_job_to_json(const void *job, char *out, size_t size)
{
    static const char js[] = "{ \"rng_seed\": \"0x0000000000000007\", \"gates\": [ { \"type\": 4, \"target\": 0, \"control\": -1 }, "
                             "{ \"type\": 7, \"target\": 1, \"control\": -1, \"theta\": 0.5 } ] }";
    if (job != (void *)8) return -1;
    dumps++;
    if (out && size >= sizeof js) memcpy(out, js, sizeof js);
    return (int)sizeof js - 1;
}
