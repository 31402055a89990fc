// frame_long.cpp -- test infrastructure: what planning a gate costs in a short
// and in a long circuit, as rotation passes (one tile and several).
#include <chrono>
#include <cstdio>
#include <random>
#include <vector>
#include "frame_plan.h"
using namespace mlx;

static double cost(int n, int gates) {
    std::mt19937_64 rng(3);
    std::vector<moonlab_hip_gate_t> g;
    while ((int)g.size() < gates) {
        for (int q = 0; q < n; q++) g.push_back({7 + (int)(rng() % 3), q, -1, -1, (double)(rng() % 6000) / 1e3, 0, 0});
        for (int o : {0, 1}) for (int q = o; q + 1 < n; q += 2) g.push_back({10, q + 1, q, -1, 0, 0, 0});
    }
    const auto t = std::chrono::steady_clock::now();
    std::vector<FGate> f; std::complex<double> ph;
    frame_lower(g.data(), (int)g.size(), n, f, ph);
    std::vector<FPass> p; std::vector<FOp> o;
    frame_plan(f, ph, n, 12, 3, 16, 2, p, o);
    return std::chrono::duration<double>(std::chrono::steady_clock::now() - t).count() / (double)g.size();
}

int main() {
    for (int n : {10, 14}) {
        double s = 1e9;
        for (int k = 0; k < 5; k++) s = std::min(s, cost(n, 10000));
        printf("%d %g %g\n", n, s * 1e6, cost(n, 600000) * 1e6);
    }
}
