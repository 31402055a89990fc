// frame_emulator.cpp -- test infrastructure: runs the Pauli-rotation engine's
// programs (frame_lower + frame_plan) on a host state thread by thread, with
// the kernels' layouts, LDS slots, signs and output permutation, and compares
// the result with the oracle's gate-by-gate run, global phase included.
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>
#include "frame_plan.h"
extern "C" {
#include "sv_oracle.h"
}
using cd = std::complex<double>;
using namespace mlx;
static int par(uint64_t x) { return __builtin_popcountll(x) & 1; }
static uint64_t ins0(uint64_t x, int q) { return ((x >> q) << (q + 1)) | (x & ((1ull << q) - 1)); }
static long g_phases, g_relayouts, g_rots, g_passes, g_cross, g_shift, g_tables;
[[noreturn]] static void die(const char *s) { printf("%s\n", s); exit(1); }

static void run_tile(std::vector<cd> &tile, const FPass &P, const std::vector<FOp> &prog, uint64_t base, int B) {
    const int nb = P.nbits, TH = 1 << (nb - 4);
    auto slot = [&](int x) { return (uint32_t)(B == 8 ? lds_slot<8>(x) : lds_slot<16>(x)) * B; };
    std::vector<cd> lds(1 << nb);
    std::vector<std::vector<cd>> v(TH, std::vector<cd>(16));
    std::vector<uint32_t> sl(TH);
    uint32_t off[16];
    for (int j = 0; j < 16; j++) off[j] = slot(j << (nb - 4));
    for (int t = 0; t < TH; t++) { sl[t] = slot(t); for (int j = 0; j < 16; j++) v[t][j] = tile[t + TH * j]; }
    auto change = [&](const std::vector<uint32_t> &ns, const uint32_t *to) {
        std::vector<int> wr(1 << nb), rd(1 << nb);
        for (int t = 0; t < TH; t++) for (int j = 0; j < 16; j++) { uint32_t b = sl[t] ^ off[j]; if (b % B || b / B >= (1u << nb)) die("slot out of range"); wr[b / B]++; lds[b / B] = v[t][j]; }
        for (int t = 0; t < TH; t++) for (int j = 0; j < 16; j++) { uint32_t b = ns[t] ^ to[j]; if (b % B || b / B >= (1u << nb)) die("slot out of range"); rd[b / B]++; v[t][j] = lds[b / B]; }
        for (int i = 0; i < (1 << nb); i++) if (wr[i] != 1 || rd[i] != 1) die("layout change is no bijection");
    };
    size_t p = (size_t)P.first;
    for (int ph = 0; ph < P.nphases; ph++) {
        FPhase h; memcpy(&h, &prog[p], sizeof h); p += kFPhaseUnits;
        if (!h.relayout && ph) die("a later phase without a layout change");
        if (memcmp(h.from, off, sizeof off)) die("header does not start from the layout before");
        g_phases++;
        if (h.nops < 1) die("empty phase");
        if (h.relayout) {
            g_relayouts++;
            std::vector<uint32_t> ns(TH);
            for (int t = 0; t < TH; t++) { int x = t; for (int i = 0; i < 4; i++) x += x & (int)h.nm[i]; ns[t] = slot(x); }
            change(ns, h.off); memcpy(off, h.off, sizeof off); sl = ns;
        }
        for (int q = 0; q < h.nops; q++, p++) {
            const FOp &o = prog[p];
            if (o.arm < 0 || o.arm >= FARM_COUNT) die("bad arm");
            g_rots++;
            for (int t = 0; t < TH; t++) {
                const double ot = B == 8 ? (double)o.tf : o.t;
                const double s0 = (par(o.zt & (uint32_t)t) ^ par(o.zg & base)) ? -ot : ot;
                std::vector<cd> in = v[t];
                for (int j = 0; j < 16; j++) {
                    if (o.arm == FARM_SCALE) { v[t][j] = s0 * in[j]; continue; }
                    if (o.arm >= FARM_Z) { v[t][j] = in[j] * cd(1, par((o.arm - FARM_Z) & j) ? s0 : -s0); continue; }
                    const int own = o.arm >= FARM_Y, a = o.arm & 31, d = a >> 3, r = a & 7;
                    const int zr = (r & ((1 << d) - 1)) | ((r >> d) << (d + 1)) | (own << d);
                    const double s = par(zr & j) ? -s0 : s0;
                    v[t][j] = own ? in[j] + s * in[j ^ (1 << d)] : in[j] - cd(0, s) * in[j ^ (1 << d)];
                }
            }
        }
    }
    if (P.flags & (FP_SIGN | FP_SCALE | FP_CSCALE))
        for (int t = 0; t < TH; t++) {
            uint32_t s = 0;
            if (P.table >= 0) { uint16_t w; memcpy(&w, (const char *)&prog[(size_t)P.table] + 2 * t, 2); s = w; if (!t) g_tables++; }
            for (int c = 0; c < P.ncross; c++) {
                FCross x; memcpy(&x, &prog[(size_t)(P.cross + c)], sizeof x);
                if (!t) g_cross++;
                const int a = par(x.ga & base), b = par(x.gb & base);
                const uint32_t fa = x.wa ^ (par(x.ta & t) ? 0xFFFFu : 0), fb = x.wb ^ (par(x.tb & t) ? 0xFFFFu : 0);
                s ^= (a ? fb : 0) ^ (b ? fa : 0) ^ (a & b ? 0xFFFFu : 0);
            }
            for (int j = 0; j < 16; j++) v[t][j] *= ((s >> j) & 1 ? -1.0 : 1.0) * cd(P.scale_r, P.flags & FP_CSCALE ? P.scale_i : 0.0);
        }
    if (P.flags & FP_OUT) {
        FOut o; memcpy(&o, &prog[(size_t)P.out], sizeof o);
        if (memcmp(o.from, off, sizeof off)) die("output does not start from the last layout");
        uint32_t sh = 0;
        for (int c = 0; c < P.nshift; c++) { FShift x; memcpy(&x, &prog[(size_t)(P.shift + c)], sizeof x); g_shift++; if (par(x.gmask & base)) sh ^= x.off; }
        std::vector<uint32_t> ns(TH);
        for (int t = 0; t < TH; t++) { ns[t] = sh; for (int b = 0; b < nb - 4; b++) if ((t >> b) & 1) ns[t] ^= o.col[b]; }
        change(ns, o.off);
    }
    for (int t = 0; t < TH; t++) for (int j = 0; j < 16; j++) tile[t + TH * j] = v[t][j];
}

// relative error, as a multiple of what is allowed: 1e-12; complex64 programs
// (B = 8) also round each tangent to a float, half an ulp (2^-25) per rotation
static double run(int n, const std::vector<moonlab_hip_gate_t> &g, int tb, int B, int look, bool nonzero_start) {
    std::vector<FGate> fg; cd phase;
    if (!frame_lower(g.data(), (int)g.size(), n, fg, phase)) die("frame_lower refused a valid list");
    std::vector<FPass> passes; std::vector<FOp> prog;
    frame_plan(fg, phase, n, tb, 3, B, look, passes, prog);
    prog.push_back(FOp{});
    const int m = n < 4 ? 4 : n;
    std::vector<double> want(2ull << n, 0.0);
    std::vector<cd> st(1ull << m, cd(0));
    want[0] = 1.0;
    if (nonzero_start) { std::mt19937_64 r(5); for (auto &x : want) x = (double)(r() % 2001) / 1000.0 - 1.0; }
    for (uint64_t i = 0; i < (1ull << n); i++) st[i] = cd(want[2 * i], want[2 * i + 1]);
    svo_apply_gates(n, want.data(), (const svo_gate_t *)g.data(), (int)g.size());
    for (const FPass &P : passes) {
        g_passes++;
        if (P.nbits != (n <= tb ? m : tb)) die("tile bits");
        if (__builtin_popcountll(P.mask) != P.nbits || (P.mask >> m)) die("tile set");
        int qs[64], k = 0; for (int q = 0; q < m; q++) if ((P.mask >> q) & 1) qs[k++] = q;
        for (uint64_t ti = 0; ti < (1ull << (m - P.nbits)); ti++) {
            uint64_t base = ti; for (int b = 0; b < P.nbits; b++) base = ins0(base, qs[b]);
            std::vector<cd> t(1 << P.nbits);
            auto addr = [&](int l) { uint64_t a = base; for (int b = 0; b < P.nbits; b++) if (l & (1 << b)) a |= 1ull << qs[b]; return a; };
            for (int l = 0; l < (1 << P.nbits); l++) t[l] = st[addr(l)];
            run_tile(t, P, prog, base, B);
            for (int l = 0; l < (1 << P.nbits); l++) st[addr(l)] = t[l];
        }
    }
    double err = 0, nrm = 0;
    for (uint64_t i = 0; i < (1ull << m); i++) { cd w = i < (1ull << n) ? cd(want[2 * i], want[2 * i + 1]) : cd(0); err = std::max(err, std::abs(st[i] - w)); nrm = std::max(nrm, std::abs(w)); }
    double rots = 0;
    for (const FGate &f : fg) rots += f.kind == FG_ROT;
    return err / nrm / (1e-12 + (B == 8 ? rots * 0x1p-25 : 0.0));
}

int main() {
    std::mt19937_64 rng(11);
    auto U = [&](double s) { return (double)(rng() % 100000) / 100000.0 * s; };
    int checked = 0; double worst = 0;
    auto note = [&](double e, const char *what, int n, int tb) { checked++; if (e > worst) worst = e; if (!(e < 1.0)) { printf("MISMATCH %s n=%d tb=%d err=%g\n", what, n, tb, e); exit(1); } };
    for (int t = 0; t <= 24; t++) {   // every gate alone, on and off the tile
        for (int n : {3, 6}) for (int tb : {4, 5, 13}) for (int rep = 0; rep < 4; rep++) {
            int q[3]; for (int i = 0; i < 3; i++) do q[i] = rng() % n; while ((i > 0 && q[i] == q[0]) || (i > 1 && q[i] == q[1]));
            note(run(n, {{t, q[0], q[1], q[2], U(20) - 10, U(20) - 10, U(20) - 10}}, tb, 16, rep & 1 ? 8 : 0, true), "gate", n, tb);
        }
    }
    for (double th : {0.0, M_PI / 2, M_PI, -M_PI, 3 * M_PI / 2, 2 * M_PI, 4 * M_PI, 1e-9, 1e5}) for (int t : {7, 8, 9, 16, 17, 18, 19, 20, 21})
        note(run(3, {{t, 1, 0, 2, th, th, -th}, {17, 2, -1, -1, th, 0, 0}, {t, 0, 2, 1, -th, th, 0}}, 13, 16, 8, true), "angle", 3, 13);
    for (int trial = 0; trial < 60; trial++) {
        int n = 1 + rng() % 14;
        std::vector<moonlab_hip_gate_t> g;
        for (int k = 0; k < 140; k++) {
            int t = rng() % 25; int q[3];
            if (n < 2 && ((t >= 10 && t <= 13) || t >= 18)) t = 17;
            if (n < 3 && t >= 23) t = 4;
            for (int i = 0; i < 3; i++) { int guard = 0; do q[i] = rng() % n; while (((i > 0 && q[i] == q[0]) || (i > 1 && q[i] == q[1])) && ++guard < 99); }
            g.push_back({t, q[0], q[1], q[2], U(14) - 7, U(14) - 7, U(14) - 7});
        }
        for (int tb : {4, 6, 8, 12, 13}) note(run(n, g, tb, trial & 1 ? 8 : 16, trial % 3 ? 8 : 0, true), "table", n, tb);
    }
    for (int trial = 0; trial < 6; trial++) {   // layered circuits: CNOT, CZ brickwork, ladders
        const int n = 13 + trial % 4;
        std::vector<moonlab_hip_gate_t> g;
        for (int q = 0; q < n; q++) g.push_back({4, q, -1, -1, 0, 0, 0});
        for (int d = 0; d < 12; d++) {
            for (int q = 0; q < n; q++) g.push_back({trial % 3 == 1 ? 17 : 7 + (int)(rng() % 3), q, -1, -1, U(6), U(6), U(6)});
            const int e = trial % 3 == 0 ? 10 : 12;
            if (trial % 3 == 2) { for (int q = 0; q + 1 < n; q++) g.push_back({e, q + 1, q, -1, 0, 0, 0}); }
            else for (int o : {0, 1}) for (int q = o; q + 1 < n; q += 2) g.push_back({e, q + 1, q, -1, 0, 0, 0});
        }
        for (int tb : {12, 13}) note(run(n, g, tb, trial & 1 ? 8 : 16, 8, true), "layers", n, tb);
    }
    const moonlab_hip_gate_t bad = {7, 0, -1, -1, NAN, 0, 0};   // stays with the general path
    std::vector<FGate> fg; cd ph;
    if (frame_lower(&bad, 1, 2, fg, ph)) die("a parameter that is not finite was accepted");
    if (!g_cross || !g_shift || !g_tables) die("signs or shifts from outside the tile never occurred");
    printf("ok: %d plans, worst %.1e of what is allowed; %ld passes, %ld tile phases, %ld layout changes, %ld rotations, %ld cross, %ld shift\n",
           checked, worst, g_passes, g_phases, g_relayouts, g_rots, g_cross, g_shift);
}
