// frame_deep.cpp -- test infrastructure: programs of thousands of rotations in
// one pass through the emulator of frame_emulator.cpp.  Stored values grow by
// 1 / cos a rotation, so such a pass is rescaled on its way and the squared
// norm it takes back at its end lies far outside a double's range.
#define main frame_emulator_main
#include "frame_emulator.cpp"
#undef main

// Rounding of g gates, on either side at most four ulps of the norm a gate,
// as the largest error over the largest amplitude (at least the norm over
// 2^(n/2)); run() counts in units of 1e-12 (complex64: that and its tangents).
static double allowed(int n, size_t gates) { return 1.0 + (double)gates * 0x1p-50 * pow(2.0, 0.5 * n) / 1e-12; }

int main() {
    std::mt19937_64 rng(23);
    auto U = [&]() { return (double)(rng() % 100000) / 100000.0 * 6.2; };
    int checked = 0;
    auto check = [&](const char *what, int n, const std::vector<moonlab_hip_gate_t> &g, int tb) {
        for (int B : {16, 8}) {
            const double e = run(n, g, tb, B, 0, true);
            checked++;
            if (!(e < allowed(n, g.size()))) { printf("MISMATCH %s n=%d tb=%d bytes=%d gates=%zu err=%g of %g\n", what, n, tb, B, g.size(), e, allowed(n, g.size())); exit(1); }
        }
    };
    auto brick = [&](int n, int depth, bool angles) {
        std::vector<moonlab_hip_gate_t> g;
        for (int d = 0; d < depth; d++) {
            for (int q = 0; q < n; q++) g.push_back(angles ? moonlab_hip_gate_t{7 + (int)(rng() % 3), q, -1, -1, U(), 0, 0} : moonlab_hip_gate_t{4, q, -1, -1, 0, 0, 0});
            for (int o : {0, 1}) for (int q = o; q + 1 < n; q += 2) g.push_back({10, q + 1, q, -1, 0, 0, 0});
        }
        return g;
    };
    // Hadamard and CNOT layers: the norm doubles with every rotation
    for (int d : {250, 500, 751, 2000}) check("layers", 4, brick(4, d, false), 12);
    for (int d : {100, 200, 301, 800}) check("layers", 10, brick(10, d, false), 12);
    for (int d : {84, 251, 400}) check("layers", 12, brick(12, d, false), 12);
    check("angles", 10, brick(10, 1000, true), 12);
    // a pass before the last one
    std::vector<moonlab_hip_gate_t> g = brick(10, 320, false);
    for (int q = 10; q < 14; q++) { g.push_back({4, q, -1, -1, 0, 0, 0}); g.push_back({10, q, q - 10, -1, 0, 0, 0}); g.push_back({8, q - 10, -1, -1, 0.3, 0, 0}); }
    check("tiles", 14, g, 12);
    check("tiles", 14, g, 13);
    printf("ok: %d plans of up to %ld rotations\n", checked, g_rots);
}
