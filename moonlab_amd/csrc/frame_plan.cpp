// frame_plan.cpp -- lowering and pass planning of the Pauli-rotation engine
// (program format: frame_program.h).
//
// Reference counterpart: the gate loops of src/quantum/gates.c:123-1048 and
// the 1q run fusion of src/optimization/fusion/fusion.c:247-292; tableau
// updates under CNOT / CZ / SWAP / X / Z follow the stabilizer formalism
// (Aaronson and Gottesman 2004).
#include "frame_plan.h"

#include <math.h>
#include <stddef.h>
#include <string.h>

#include <algorithm>

#include "fusion.h"

namespace mlx {
namespace {

using cd = std::complex<double>;

int par(uint64_t x) { return __builtin_popcountll(x) & 1; }

// c (1 - i (s/c) P) for exp(-i theta/2 P), c = cos, s = sin of theta/2.  For
// |s| > |c| the Pauli factor is split off: -i s P (1 + i (c/s) P).
struct Rot {
    double t, scale;
    bool   pauli;     // times -i P
};

Rot make_rot(double c, double s)
{
    if (fabs(c) >= fabs(s)) return Rot{s / c, c, false};
    return Rot{-c / s, s, true};
}

// One step of a run of single-qubit gates: a rotation about X, Y or Z.
struct Step {
    int    axis;      // 0 X, 1 Y, 2 Z
    double c, s;      // of theta/2
};

// The gates waiting on one qubit: up to three steps, applied in order and
// times phase, or, for longer runs, their product u (three Euler rotations
// are shorter then).
struct Pending {
    Step st[3];
    int  nst = 0;
    bool folded = false;
    cd   phase = 1.0;
    cd   u[4];
};

class Lowering {
  public:
    Lowering(int n, std::vector<FGate> &out, cd &phase) : out_(out), phase_(phase), pend_((size_t)n) {}

    // exp(-i theta/2 P) on the masks (x, z)
    void rot(uint64_t x, uint64_t z, double c, double s)
    {
        const Rot r = make_rot(c, s);
        if (r.pauli) {   // -i P = -i i^|x&z| X^x Z^z
            phase_ *= ipow(3 + __builtin_popcountll(x & z));
            for (uint64_t m = z; m; m &= m - 1) frame(FG_Z, __builtin_ctzll(m), -1);
            for (uint64_t m = x; m; m &= m - 1) frame(FG_X, __builtin_ctzll(m), -1);
        }
        if (r.t == 0.0) {
            phase_ *= r.scale;
            return;
        }
        out_.push_back(FGate{FG_ROT, -1, -1, x, z, r.t, r.scale});
    }
    void rot_angle(uint64_t x, uint64_t z, double theta) { rot(x, z, cos(theta / 2.0), sin(theta / 2.0)); }
    void frame(FGateKind k, int a, int b) { out_.push_back(FGate{k, (int8_t)a, (int8_t)b, 0, 0, 0.0, 1.0}); }
    static cd ipow(int k)
    {
        static const cd p[4] = {cd(1, 0), cd(0, 1), cd(-1, 0), cd(0, -1)};
        return p[k & 3];
    }

    // a single-qubit gate: phase times a step
    void step(int q, int axis, double c, double sn, cd phase = 1.0)
    {
        Pending &p = pend_[(size_t)q];
        p.phase *= phase;
        const Step st{axis, c, sn};
        if (p.folded) {
            fold(p, st);
        } else if (p.nst && p.st[p.nst - 1].axis == axis) {   // same axis: angles add
            Step &l = p.st[p.nst - 1];
            l = Step{axis, l.c * c - l.s * sn, l.s * c + l.c * sn};
        } else if (p.nst < 3) {
            p.st[p.nst++] = st;
        } else {
            step_matrix(p.st[0], p.u);
            for (int i = 1; i < 3; i++) fold(p, p.st[i]);
            fold(p, st);
            p.folded = true;
        }
    }

    // Emit qubit q's pending gates; a last rotation about axis `keep` (2 Z, 0
    // X, -1 none) stays pending: it commutes with the gate that follows and
    // may merge with the rotation after it.
    void flush(int q, int keep)
    {
        Pending &p = pend_[(size_t)q];
        if (!p.nst) {
            phase_ *= p.phase;
            p.phase = 1.0;
            return;
        }
        if (p.folded) euler(p);
        phase_ *= p.phase;
        p.phase = 1.0;
        const uint64_t b = 1ull << q;
        int m = p.nst;
        const bool hold = p.st[m - 1].axis == keep;
        if (hold) m--;
        for (int i = 0; i < m; i++)
            rot(p.st[i].axis == 2 ? 0 : b, p.st[i].axis == 0 ? 0 : b, p.st[i].c, p.st[i].s);
        if (hold) p.st[0] = p.st[m];
        p.nst = hold ? 1 : 0;
    }

    static void step_matrix(const Step &l, cd u[4])
    {
        if (l.axis == 2) { u[0] = cd(l.c, -l.s); u[1] = u[2] = 0.0; u[3] = cd(l.c, l.s); }
        else if (l.axis == 0) { u[0] = u[3] = l.c; u[1] = u[2] = cd(0.0, -l.s); }
        else { u[0] = u[3] = l.c; u[1] = -l.s; u[2] = l.s; }
    }

  private:
    static void fold(Pending &p, const Step &l)
    {
        cd m[4];
        step_matrix(l, m);
        const cd a = p.u[0], b = p.u[1], c = p.u[2], d = p.u[3];
        p.u[0] = m[0] * a + m[1] * c;
        p.u[1] = m[0] * b + m[1] * d;
        p.u[2] = m[2] * a + m[3] * c;
        p.u[3] = m[2] * b + m[3] * d;
    }

    // u = RZ(beta) RY(gamma) RZ(delta) times a phase (into p.phase).  A sum or difference that an
    // entry of modulus 0 leaves open is taken as 0; each is known up to 2 pi,
    // and the one of the smaller entry takes the branch that agrees with the
    // phase the larger entry gives.
    static void euler(Pending &p)
    {
        const double c = abs(p.u[0]), s = abs(p.u[2]);
        const double h = hypot(c, s);
        double sum = c > 0.0 ? arg(p.u[3] * conj(p.u[0])) : 0.0;      // beta + delta
        double dif = s > 0.0 ? arg(-p.u[2] * conj(p.u[1])) : 0.0;     // beta - delta
        cd ph;
        if (c >= s) {
            ph = p.u[0] / c * std::polar(1.0, 0.5 * sum);
            if (s > 0.0 && real(p.u[2] * conj(ph * std::polar(1.0, 0.5 * dif))) < 0.0) dif += 2.0 * M_PI;
        } else {
            ph = p.u[2] / s * std::polar(1.0, -0.5 * dif);
            if (c > 0.0 && real(p.u[0] * conj(ph * std::polar(1.0, -0.5 * sum))) < 0.0) sum += 2.0 * M_PI;
        }
        const double beta = 0.5 * (sum + dif), delta = 0.5 * (sum - dif);
        p.phase *= ph;
        p.st[0] = Step{2, cos(0.5 * delta), sin(0.5 * delta)};
        p.st[1] = Step{1, c / h, s / h};
        p.st[2] = Step{2, cos(0.5 * beta), sin(0.5 * beta)};
        p.nst = 3;
        p.folded = false;
    }

    std::vector<FGate>  &out_;
    cd                  &phase_;
    std::vector<Pending> pend_;
};

}  // namespace

GateParams gate_params(const moonlab_hip_gate_t &g)
{
    const bool theta = std::isfinite(g.theta);
    switch (g.type) {
    case MOONLAB_HIP_GATE_RX:
    case MOONLAB_HIP_GATE_RY:
    case MOONLAB_HIP_GATE_RZ: return theta ? PARAMS_FINITE : PARAMS_SPOIL_ALL;
    case MOONLAB_HIP_GATE_U3:
        if (!theta) return PARAMS_SPOIL_ALL;
        return std::isfinite(g.phi) && std::isfinite(g.lam) ? PARAMS_FINITE : PARAMS_SPOIL_PART;
    case MOONLAB_HIP_GATE_PHASE:
    case MOONLAB_HIP_GATE_CPHASE:
    case MOONLAB_HIP_GATE_CRX:
    case MOONLAB_HIP_GATE_CRY:
    case MOONLAB_HIP_GATE_CRZ: return theta ? PARAMS_FINITE : PARAMS_SPOIL_PART;
    default: return PARAMS_FINITE;   // reads none
    }
}

bool frame_lower(const moonlab_hip_gate_t *g, int ng, int n, std::vector<FGate> &out, cd &phase, bool any_angle)
{
    phase = 1.0;
    Lowering L(n, out, phase);
    const double r8 = 0.70710678118654752440;            // cos(pi/4)
    const double c8 = cos(M_PI / 8.0), s8 = sin(M_PI / 8.0);
    const cd I(0.0, 1.0);
    static_assert(MOONLAB_HIP_GATE_RY == MOONLAB_HIP_GATE_RX + 1 && MOONLAB_HIP_GATE_RZ == MOONLAB_HIP_GATE_RX + 2,
                  "axis = type - RX");
    for (int i = 0; i < ng; i++) {
        const moonlab_hip_gate_t &x = g[i];
        if (!gate_valid(x, n)) return false;
        if (!any_angle && gate_params(x) != PARAMS_FINITE) return false;
        const int t = x.target, c = x.control, e = x.extra;
        const uint64_t T = t >= 0 ? 1ull << t : 0, C = c >= 0 ? 1ull << c : 0;
        double si, co;
        switch (x.type) {
        case MOONLAB_HIP_GATE_I: continue;
        case MOONLAB_HIP_GATE_X: L.step(t, 0, 0.0, 1.0, I); continue;
        case MOONLAB_HIP_GATE_Y: L.step(t, 1, 0.0, 1.0, I); continue;
        case MOONLAB_HIP_GATE_Z: L.step(t, 2, 0.0, 1.0, I); continue;
        case MOONLAB_HIP_GATE_H:   // X RY(pi/2)
            L.step(t, 1, r8, r8);
            L.step(t, 0, 0.0, 1.0, I);
            continue;
        case MOONLAB_HIP_GATE_S: L.step(t, 2, r8, r8, cd(r8, r8)); continue;
        case MOONLAB_HIP_GATE_SDG: L.step(t, 2, r8, -r8, cd(r8, -r8)); continue;
        case MOONLAB_HIP_GATE_T: L.step(t, 2, c8, s8, cd(c8, s8)); continue;
        case MOONLAB_HIP_GATE_TDG: L.step(t, 2, c8, -s8, cd(c8, -s8)); continue;
        case MOONLAB_HIP_GATE_PHASE:
            sincos(x.theta / 2.0, &si, &co);
            L.step(t, 2, co, si, cd(co, si));
            continue;
        case MOONLAB_HIP_GATE_RX:
        case MOONLAB_HIP_GATE_RY:
        case MOONLAB_HIP_GATE_RZ:
            sincos(x.theta / 2.0, &si, &co);
            L.step(t, x.type - MOONLAB_HIP_GATE_RX, co, si);
            continue;
        case MOONLAB_HIP_GATE_U3: {   // e^(i (phi + lam) / 2) RZ(phi) RY(theta) RZ(lam)
            double sp, cp, sl, cl;
            sincos(x.theta / 2.0, &si, &co);
            sincos(x.phi / 2.0, &sp, &cp);
            sincos(x.lam / 2.0, &sl, &cl);
            L.step(t, 2, cl, sl, cd(cl, sl));
            L.step(t, 1, co, si);
            L.step(t, 2, cp, sp, cd(cp, sp));
            continue;
        }
        default: break;
        }
        switch (x.type) {
        case MOONLAB_HIP_GATE_CNOT:
            L.flush(c, 2);
            L.flush(t, 0);
            L.frame(FG_CX, c, t);
            break;
        case MOONLAB_HIP_GATE_CY:        // S, CNOT, S^dag on the target; CY_TRUE: S^dag, CNOT, S
        case MOONLAB_HIP_GATE_CY_TRUE: {
            const double s = x.type == MOONLAB_HIP_GATE_CY ? r8 : -r8;
            L.flush(c, 2);
            L.flush(t, -1);
            L.rot(0, T, r8, s);
            L.frame(FG_CX, c, t);
            L.rot(0, T, r8, -s);
            break;
        }
        case MOONLAB_HIP_GATE_CZ:
            L.flush(c, 2);
            L.flush(t, 2);
            L.frame(FG_CZ, c, t);
            break;
        case MOONLAB_HIP_GATE_SWAP:
            L.flush(c, -1);
            L.flush(t, -1);
            L.frame(FG_SWAP, c, t);
            break;
        case MOONLAB_HIP_GATE_CPHASE:    // e^(i l/4) exp(-i l/4 Zc) exp(-i l/4 Zt) exp(i l/4 Zc Zt)
            L.flush(c, 2);
            L.flush(t, 2);
            phase *= std::polar(1.0, x.theta / 4.0);
            L.rot_angle(0, C, x.theta / 2.0);
            L.rot_angle(0, T, x.theta / 2.0);
            L.rot_angle(0, C | T, -x.theta / 2.0);
            break;
        case MOONLAB_HIP_GATE_CRX:       // exp(-i th/4 P) exp(i th/4 Zc P)
        case MOONLAB_HIP_GATE_CRY:
        case MOONLAB_HIP_GATE_CRZ: {
            const uint64_t px = x.type == MOONLAB_HIP_GATE_CRZ ? 0 : T, pz = x.type == MOONLAB_HIP_GATE_CRX ? 0 : T;
            L.flush(c, 2);
            L.flush(t, -1);
            L.rot_angle(px, pz, x.theta / 2.0);
            L.rot_angle(px, pz | C, -x.theta / 2.0);
            break;
        }
        case MOONLAB_HIP_GATE_TOFFOLI:
        case MOONLAB_HIP_GATE_FREDKIN: {
            // H CCZ H on one qubit; Fredkin = CX(e, t), Toffoli(c, t -> e), CX(e, t).
            // CCZ = e^(i pi/8) times rotations by +-pi/4 about the Z strings of its qubits.
            const bool fred = x.type == MOONLAB_HIP_GATE_FREDKIN;
            for (int q : {c, t, e}) L.flush(q, -1);
            const int tgt = fred ? e : t, other = fred ? t : e;
            const uint64_t X = 1ull << tgt, O = 1ull << other;
            if (fred) L.frame(FG_CX, e, t);
            L.rot(X, X, r8, r8);
            L.frame(FG_X, tgt, -1);
            phase *= cd(c8, s8);
            for (uint64_t m : {C, O, X, C | O | X}) L.rot(0, m, c8, s8);
            for (uint64_t m : {C | O, C | X, O | X}) L.rot(0, m, c8, -s8);
            L.rot(X, X, r8, r8);
            L.frame(FG_X, tgt, -1);
            if (fred) L.frame(FG_CX, e, t);
            break;
        }
        default: return false;
        }
    }
    for (int q = 0; q < n; q++) L.flush(q, -1);
    return true;
}

namespace {

// How a gate acts on each qubit: diagonally (z), as a function of X (x) or
// otherwise (o).  Two gates commute when, on every shared qubit, both act
// diagonally or both as functions of X.
struct Kinds {
    uint64_t z, x, o;
};

Kinds kinds_of(const FGate &g)
{
    const uint64_t a = g.a >= 0 ? 1ull << g.a : 0, b = g.b >= 0 ? 1ull << g.b : 0;
    switch (g.kind) {
    case FG_ROT: return Kinds{g.z & ~g.x, g.x & ~g.z, g.x & g.z};
    case FG_CX: return Kinds{a, b, 0};
    case FG_CZ: return Kinds{a | b, 0, 0};
    case FG_SWAP: return Kinds{0, 0, a | b};
    case FG_X: return Kinds{0, a, 0};
    default: return Kinds{a, 0, 0};
    }
}

// Stored-frame image of a Pauli: (-1)^s i^|x&z| X^x Z^z Z_global^g.
struct Row {
    uint32_t x = 0, z = 0;
    uint64_t g = 0;
    int      s = 0;
};

// product a b of commuting images
Row mul(const Row &a, const Row &b)
{
    Row r;
    r.x = a.x ^ b.x;
    r.z = a.z ^ b.z;
    r.g = a.g ^ b.g;
    const int e = __builtin_popcount(a.x & a.z) + __builtin_popcount(b.x & b.z) + 2 * __builtin_popcount(a.z & b.x) -
                  __builtin_popcount(r.x & r.z);
    r.s = a.s ^ b.s ^ ((e >> 1) & 1);
    return r;
}

// A sign term (fa + a)(fb + b): the value functionals of two Z images.
struct Quad {
    uint32_t za, zb;
    uint64_t ga, gb;
    int      sa, sb;
};

struct LRot {
    Row    p;
    double t;
};

// A layout: stored index of register value j and thread t.
struct Layout {
    uint32_t r[kFrameRegBits];     // columns of R
    int      piv[kFrameRegBits];   // pivot positions, ascending
    int      nb;
};

// Pivots of four independent columns, the highest possible positions (thread
// bits then are the low index bits); false when they are dependent.
bool set_pivots(Layout &L)
{
    uint32_t rows[kFrameRegBits];
    for (int i = 0; i < kFrameRegBits; i++) rows[i] = L.r[i];
    int k = 0;
    for (int b = L.nb - 1; b >= 0 && k < kFrameRegBits; b--) {
        int f = -1;
        for (int i = k; i < kFrameRegBits; i++)
            if ((rows[i] >> b) & 1) {
                f = i;
                break;
            }
        if (f < 0) continue;
        std::swap(rows[f], rows[k]);
        for (int i = 0; i < kFrameRegBits; i++)
            if (i != k && ((rows[i] >> b) & 1)) rows[i] ^= rows[k];
        L.piv[k++] = b;
    }
    if (k < kFrameRegBits) return false;
    std::sort(L.piv, L.piv + kFrameRegBits);
    return true;
}

Layout io_layout(int nb)
{
    Layout L;
    L.nb = nb;
    for (int i = 0; i < kFrameRegBits; i++) {
        L.r[i] = 1u << (nb - kFrameRegBits + i);
        L.piv[i] = nb - kFrameRegBits + i;
    }
    return L;
}

bool same(const Layout &a, const Layout &b)
{
    return memcmp(a.r, b.r, sizeof a.r) == 0;   // pivots follow from the columns
}

uint32_t reg_index(const Layout &L, int j)
{
    uint32_t x = 0;
    for (int i = 0; i < kFrameRegBits; i++)
        if ((j >> i) & 1) x ^= L.r[i];
    return x;
}

// thread-bit mask of a functional z: thread bit b is the b-th index bit that
// is no pivot
uint32_t thread_mask(const Layout &L, uint32_t z)
{
    uint32_t m = 0;
    int b = 0;
    for (int q = 0; q < L.nb; q++) {
        bool piv = false;
        for (int i = 0; i < kFrameRegBits; i++) piv = piv || L.piv[i] == q;
        if (piv) continue;
        if ((z >> q) & 1) m |= 1u << b;
        b++;
    }
    return m;
}

uint32_t reg_mask(const Layout &L, uint32_t z)
{
    uint32_t m = 0;
    for (int i = 0; i < kFrameRegBits; i++)
        if (par(z & L.r[i])) m |= 1u << i;
    return m;
}

// pattern of a functional over the 16 register values
uint32_t walsh16(uint32_t zr)
{
    uint32_t w = 0;
    static const uint32_t p[4] = {0xAAAAu, 0xCCCCu, 0xF0F0u, 0xFF00u};
    for (int i = 0; i < 4; i++)
        if ((zr >> i) & 1) w ^= p[i];
    return w;
}

uint32_t slot_bytes(uint32_t x, int amp_bytes)
{
    return (uint32_t)((amp_bytes == 8 ? lds_slot<8>((int)x) : lds_slot<16>((int)x)) * amp_bytes);
}

// independent of the first k columns?
bool independent(const uint32_t *cols, int k, uint32_t v)
{
    uint32_t rows[kFrameRegBits + 1];
    for (int i = 0; i < k; i++) rows[i] = cols[i];
    for (int i = 0; i < k; i++) {
        if (!rows[i]) continue;
        const uint32_t top = 1u << (31 - __builtin_clz(rows[i]));
        for (int l = i + 1; l < k; l++)
            if (rows[l] & top) rows[l] ^= rows[i];
        if (v & top) v ^= rows[i];
    }
    return v != 0;
}

constexpr size_t kLookaheadOps = 4096;   // candidates are compared on (or seeded by) these pending gates

class PassBuilder {
  public:
    PassBuilder(int amp_bytes, int lookahead, std::vector<FPass> &passes, std::vector<FOp> &prog)
        : bytes_(amp_bytes), look_(lookahead), passes_(passes), prog_(prog)
    {
    }
    cd scale = 1.0;   // not yet applied

    void build(const std::vector<const FGate *> &gates, uint64_t set, int nb, bool last)
    {
        FPass P{};
        P.nbits = nb;
        int local[64];
        for (int q = 0; q < 64; q++) local[q] = -1;
        int k = 0;
        for (int q = 0; q < 64 && k < nb; q++)
            if (set & (1ull << q)) {
                local[q] = k++;
                P.mask |= 1ull << q;
            }
        image(gates, local, nb);
        P.first = (int32_t)prog_.size();
        Layout cur = io_layout(nb);
        phases(P, cur);
        finish(P, cur, last);
        passes_.push_back(P);
    }

  private:
    // Walk the pass's gates through the tableau: rotations become images,
    // the rest the frame.
    void image(const std::vector<const FGate *> &gates, const int *local, int nb)
    {
        X_.assign((size_t)nb, Row());
        Z_.assign((size_t)nb, Row());
        for (int i = 0; i < nb; i++) X_[(size_t)i].x = Z_[(size_t)i].z = 1u << i;
        rots_.clear();
        quads_.clear();
        auto zrow = [&](int q) {
            if (local[q] >= 0) return Z_[(size_t)local[q]];
            Row r;
            r.g = 1ull << q;
            return r;
        };
        for (const FGate *g : gates) {
            switch (g->kind) {
            case FG_ROT: {
                // i^|x&z| prod X prod Z, images multiplied as i^k X^x Z^z
                int k = __builtin_popcountll(g->x & g->z);
                Row p;
                auto times = [&](const Row &b) {
                    k += 2 * b.s + __builtin_popcount(b.x & b.z) + 2 * __builtin_popcount(p.z & b.x);
                    p.x ^= b.x;
                    p.z ^= b.z;
                    p.g ^= b.g;
                };
                for (uint64_t m = g->x; m; m &= m - 1) times(X_[(size_t)local[__builtin_ctzll(m)]]);
                for (uint64_t m = g->z; m; m &= m - 1) times(zrow(__builtin_ctzll(m)));
                p.s = ((k - __builtin_popcount(p.x & p.z)) >> 1) & 1;
                rots_.push_back(LRot{p, g->t});
                // the norm that the rounded tangent leaves, not the cosine
                const long double t = bytes_ == 8 ? (long double)(float)g->t : (long double)g->t;
                grow_ *= 1.0L + t * t;
                if (grow_ > 0x1p1000L) {   // 2^1000 of it move to the exponent
                    grow_ *= 0x1p-1000L;
                    exp_ -= 500;
                }
                if (g->scale < 0.0) scale = -scale;
                break;
            }
            case FG_CX: {
                const int t = local[g->b];
                if (local[g->a] >= 0) X_[(size_t)local[g->a]] = mul(X_[(size_t)local[g->a]], X_[(size_t)t]);
                Z_[(size_t)t] = mul(Z_[(size_t)t], zrow(g->a));
                break;
            }
            case FG_CZ: {
                const Row za = zrow(g->a), zb = zrow(g->b);
                if (local[g->a] >= 0) X_[(size_t)local[g->a]] = mul(X_[(size_t)local[g->a]], zb);
                if (local[g->b] >= 0) X_[(size_t)local[g->b]] = mul(X_[(size_t)local[g->b]], za);
                quads_.push_back(Quad{za.z, zb.z, za.g, zb.g, za.s, zb.s});
                break;
            }
            case FG_SWAP:
                std::swap(X_[(size_t)local[g->a]], X_[(size_t)local[g->b]]);
                std::swap(Z_[(size_t)local[g->a]], Z_[(size_t)local[g->b]]);
                break;
            case FG_X: Z_[(size_t)local[g->a]].s ^= 1; break;
            case FG_Z: {
                const Row z = zrow(g->a);
                if (local[g->a] >= 0) X_[(size_t)local[g->a]].s ^= 1;
                quads_.push_back(Quad{z.z, 0, z.g, 0, z.s, 1});
                break;
            }
            }
        }
    }

    // The pass's factor 2^exp_ / sqrt(grow_) into the scale.  Only here, where
    // the growth and the rescalings that took it back on the way (phases) have
    // met: either alone is 2^-500 for a thousand rotations.
    void settle()
    {
        const long double f = ldexpl(1.0L / sqrtl(grow_), (int)exp_);
        scale = cd((double)(f * scale.real()), (double)(f * scale.imag()));
        grow_ = 1.0L;
        exp_ = 0;
    }

    // x and z of an image in one word; two commute when parity(a & swap(b)) is 0
    static uint32_t packed(const Row &p) { return p.x | (p.z << 16); }
    static uint32_t swapped(uint32_t v) { return (v >> 16) | (v << 16); }

    // Rotations of rest_ from head_ on that a phase takes, in order: those whose
    // direction is one of its (up to four) basis vectors and that commute with
    // every rotation put off.  fixed: the basis is given whole.  "Commutes with
    // every one" is checked against a basis of their span (at most 2 x tile
    // bits words); once that is full nothing more can be taken: the scan ends
    // at stop_, so that a long circuit's planning stays linear.
    int scan(uint32_t *basis, int &nbasis, bool fixed)
    {
        take_.clear();
        def_.clear();
        uint32_t span[2 * kFrameMaxTileBits];   // swapped words, echelon form by leading bit
        int rank = 0;
        const size_t m = rest_.size();
        size_t i = head_;
        for (; i < m && rank < 2 * nb_; i++) {
            const int id = rest_[i];
            const uint32_t w = pack_[(size_t)id], x = w & 0xFFFFu;
            bool ok = true;
            for (int d = 0; d < rank && ok; d++) ok = !(__builtin_popcount(w & span[d]) & 1);
            if (ok && x) {
                bool in = false;
                for (int b = 0; b < nbasis; b++) in = in || basis[b] == x;
                if (!in) {
                    if (!fixed && nbasis < kFrameRegBits && independent(basis, nbasis, x)) basis[nbasis++] = x;
                    else ok = false;
                }
            }
            if (ok) {
                take_.push_back(id);
                continue;
            }
            def_.push_back(id);
            uint32_t v = swapped(w);
            for (int d = 0; d < rank; d++) v = std::min(v, v ^ span[d]);   // clears span[d]'s leading bit
            if (v) span[rank++] = v;
        }
        stop_ = i;
        return (int)take_.size();
    }

    void phases(FPass &P, Layout &cur)
    {
        nb_ = P.nbits;
        rest_.resize(rots_.size());
        pack_.resize(rots_.size());
        for (size_t i = 0; i < rest_.size(); i++) {
            rest_[i] = (int)i;
            pack_[i] = packed(rots_[i].p);
        }
        double grown = 0.0;
        size_t hpos = 0, best_stop = 0;   // header of the latest phase
        head_ = 0;
        while (head_ < rest_.size()) {
            // candidates: for the first phase the layout the tile enters in
            // (no exchange through LDS; later phases have used up theirs), a
            // basis grown greedily, and bases seeded by the next pending directions
            uint32_t best[kFrameRegBits], b[kFrameRegBits];
            int nbest = kFrameRegBits, nb = kFrameRegBits, got = 0;
            memcpy(best, cur.r, sizeof best);
            if (P.nphases == 0) {
                got = scan(best, nbest, true);
                if (got > 0) got++;   // a layout change costs about eight rotations' arithmetic, mostly hidden
                best_take_.swap(take_);
                best_def_.swap(def_);
                best_stop = stop_;
            }
            auto candidate = [&](uint32_t seed) {
                nb = 0;
                if (seed) b[nb++] = seed;
                const int c = scan(b, nb, false);
                if (c > got) {
                    got = c;
                    memcpy(best, b, sizeof best);
                    nbest = nb;
                    best_take_.swap(take_);
                    best_def_.swap(def_);
                    best_stop = stop_;
                }
            };
            candidate(0);
            if (look_ > 0) {
                uint32_t seen[64];
                int ns = 0;
                const size_t end = std::min(rest_.size(), head_ + kLookaheadOps);
                for (size_t i = head_; i < end && ns < look_ && ns < 64; i++) {
                    const uint32_t x = rots_[(size_t)rest_[i]].p.x;
                    if (!x || std::find(seen, seen + ns, x) != seen + ns) continue;
                    seen[ns++] = x;
                    if (ns > 1) candidate(x);   // the first is the greedy basis
                }
            }
            // complete the basis with the highest unit vectors that keep it independent
            for (int q = P.nbits - 1; q >= 0 && nbest < kFrameRegBits; q--)
                if (independent(best, nbest, 1u << q)) best[nbest++] = 1u << q;
            Layout L;
            L.nb = P.nbits;
            memcpy(L.r, best, sizeof best);
            std::sort(L.r, L.r + kFrameRegBits);
            set_pivots(L);
            FPhase h{};
            h.relayout = !same(L, cur);
            for (int j = 0; j < 16; j++) h.from[j] = slot_bytes(reg_index(cur, j), bytes_);
            if (h.relayout) cur = L;
            for (int i = 0; i < kFrameRegBits; i++) h.nm[i] = 0u - (1u << cur.piv[i]);
            for (int j = 0; j < 16; j++) h.off[j] = slot_bytes(reg_index(cur, j), bytes_);
            // in the layout of the phase before: its rotations go on
            const bool join = !h.relayout && P.nphases > 0;
            if (!join) {
                hpos = prog_.size();
                prog_.resize(hpos + kFPhaseUnits);
                memcpy((void *)&prog_[hpos], &h, sizeof h);
                P.nphases++;
            }
            for (int i : best_take_) {
                const LRot &o = rots_[(size_t)i];
                prog_.push_back(encode(o, cur));
                // stored values grow by 1 / cos: rescale before single precision could overflow
                grown += 0.5 * log2(1.0 + o.t * o.t);
                if (grown > 32.0) {
                    const double k = floor(grown), f = exp2(-k);
                    prog_.push_back(FOp{FARM_SCALE, 0, 0, f, (float)f, 0});
                    exp_ += (int64_t)k;
                    grown -= k;
                }
            }
            const int32_t nops = (int32_t)(prog_.size() - hpos) - kFPhaseUnits;
            memcpy((char *)&prog_[hpos] + offsetof(FPhase, nops), &nops, sizeof nops);
            // those put off stay ahead of the ones not looked at
            head_ = best_stop - best_def_.size();
            std::copy(best_def_.begin(), best_def_.end(), rest_.begin() + (long)head_);
        }
    }

    FOp encode(const LRot &o, const Layout &L) const
    {
        const uint32_t zr = reg_mask(L, o.p.z);
        const int k = __builtin_popcount(o.p.x & o.p.z) & 3;
        double t = o.p.s ? -o.t : o.t;
        FOp f{};
        if (o.p.x) {
            int d = 0;
            while (L.r[d] != o.p.x) d++;
            const uint32_t rest = (zr & ((1u << d) - 1)) | (zr >> (d + 1) << d);
            if (k & 1) {          // i^(k+1) real
                f.arm = FARM_Y + 8 * d + (int)rest;
                if (k == 1) t = -t;
            } else {              // -i i^k
                f.arm = FARM_X + 8 * d + (int)rest;
                if (k == 2) t = -t;
            }
        } else {
            f.arm = FARM_Z + (int)zr;
        }
        f.zt = thread_mask(L, o.p.z);
        f.zg = o.p.g;
        f.t = t;
        f.tf = (float)t;
        return f;
    }

    // Signs and scale in the last layout, then the output layout.
    void finish(FPass &P, const Layout &cur, bool last)
    {
        const int nb = P.nbits, tbits = nb - kFrameRegBits;
        // local part of the signs as a quadratic form over (value bits 0..3,
        // thread bits above): m[i] bit l = coefficient of bits i and l
        uint32_t m[kFrameMaxTileBits] = {}, lin = 0;
        int cst = 0;
        bool any = false;
        std::vector<FCross> cross;
        for (const Quad &q : quads_) {
            const uint32_t fa = reg_mask(cur, q.za) | (thread_mask(cur, q.za) << 4);
            const uint32_t fb = reg_mask(cur, q.zb) | (thread_mask(cur, q.zb) << 4);
            for (int i = 0; i < nb; i++)
                if ((fa >> i) & 1) m[i] ^= fb;
            if (q.sa) lin ^= fb;
            if (q.sb) lin ^= fa;
            cst ^= q.sa & q.sb;
            if (q.ga | q.gb) {
                FCross c{};
                c.ga = q.ga;
                c.gb = q.gb;
                c.ta = (uint16_t)(fa >> 4);
                c.tb = (uint16_t)(fb >> 4);
                c.wa = (uint16_t)(walsh16(fa & 15) ^ (q.sa ? 0xFFFFu : 0u));
                c.wb = (uint16_t)(walsh16(fb & 15) ^ (q.sb ? 0xFFFFu : 0u));
                cross.push_back(c);
            }
        }
        uint32_t sym[kFrameMaxTileBits];   // strictly lower part: coefficient of bit i with each lower bit
        for (int i = 0; i < nb; i++) {
            if ((m[i] >> i) & 1) lin ^= 1u << i;
            sym[i] = 0;
            for (int l = 0; l < i; l++)
                if (((m[i] >> l) ^ (m[l] >> i)) & 1) sym[i] |= 1u << l;
            any = any || sym[i];
        }
        any = any || lin || cst;
        if (any) {
            // q(x | 2^i) = q(x) + parity(sym[i] & x) + lin_i, doubled bit by bit
            const int units = tbits > 4 ? 1 << (tbits - 4) : 1;
            P.table = (int32_t)prog_.size();
            prog_.resize(prog_.size() + (size_t)units);
            table_.assign((size_t)1 << tbits, 0);
            uint32_t w = 0;   // value bits, thread 0
            for (int j = 0; j < 16; j++) {
                int v = cst;
                for (int i = 0; i < 4; i++)
                    if ((j >> i) & 1) v ^= ((lin >> i) & 1) ^ par(sym[i] & (uint32_t)j & ((1u << i) - 1));
                w |= (uint32_t)v << j;
            }
            table_[0] = (uint16_t)w;
            for (int i = 4; i < nb; i++) {
                const uint32_t base = walsh16(sym[i] & 15) ^ (((lin >> i) & 1) ? 0xFFFFu : 0u);
                const uint32_t st = sym[i] >> 4;
                for (uint32_t t = 0; t < (1u << (i - 4)); t++)
                    table_[t | (1u << (i - 4))] = (uint16_t)(table_[t] ^ base ^ (par(st & t) ? 0xFFFFu : 0u));
            }
            memcpy((void *)&prog_[(size_t)P.table], table_.data(), table_.size() * sizeof(uint16_t));
        }
        if (any || !cross.empty()) P.flags |= FP_SIGN;
        if (!any) P.table = -1;
        P.cross = (int32_t)prog_.size();
        P.ncross = (int32_t)cross.size();
        for (const FCross &c : cross) push(c);
        // the scale, when this pass is the last or it has run far from 1
        settle();
        const double mag = log2(abs(scale));
        if (scale != cd(1.0) && (last || fabs(mag) > 20.0)) {
            // the phase waits for the last pass
            const cd apply = last ? scale : cd(abs(scale));
            P.scale_r = apply.real();
            P.scale_i = apply.imag();
            P.flags |= apply.imag() != 0.0 ? FP_CSCALE : FP_SCALE;
            scale = last ? cd(1.0) : scale / abs(scale);
        } else {
            P.scale_r = 1.0;
        }
        // output: index y = A x + b, rows of A the Z images; read from A^-1 (y + b)
        std::vector<uint32_t> a((size_t)nb), inv((size_t)nb);   // rows of A | rows of the inverse
        uint32_t b0 = 0;
        bool ident = same(cur, io_layout(nb));
        std::vector<uint64_t> gm((size_t)nb);
        for (int i = 0; i < nb; i++) {
            a[(size_t)i] = Z_[(size_t)i].z;
            inv[(size_t)i] = 1u << i;
            gm[(size_t)i] = Z_[(size_t)i].g;
            if (Z_[(size_t)i].s) b0 |= 1u << i;
            ident = ident && a[(size_t)i] == (1u << i) && !Z_[(size_t)i].s && !gm[(size_t)i];
        }
        P.shift = P.out = (int32_t)prog_.size();
        if (ident) return;
        P.flags |= FP_OUT;
        for (int c = 0; c < nb; c++) {   // Gauss-Jordan; A is invertible
            int r = c;
            while (!((a[(size_t)r] >> c) & 1)) r++;
            std::swap(a[(size_t)r], a[(size_t)c]);
            std::swap(inv[(size_t)r], inv[(size_t)c]);
            for (int i = 0; i < nb; i++)
                if (i != c && ((a[(size_t)i] >> c) & 1)) {
                    a[(size_t)i] ^= a[(size_t)c];
                    inv[(size_t)i] ^= inv[(size_t)c];
                }
        }
        auto col = [&](uint32_t y) {   // A^-1 y
            uint32_t x = 0;
            for (int i = 0; i < nb; i++)
                if (par(inv[(size_t)i] & y)) x |= 1u << i;
            return x;
        };
        FOut o{};
        const uint32_t xb = slot_bytes(col(b0), bytes_);
        for (int j = 0; j < 16; j++) o.from[j] = slot_bytes(reg_index(cur, j), bytes_);
        for (int j = 0; j < 16; j++) o.off[j] = xb ^ slot_bytes(col((uint32_t)j << tbits), bytes_);
        for (int t = 0; t < tbits; t++) o.col[t] = slot_bytes(col(1u << t), bytes_);
        const size_t at = prog_.size();
        prog_.resize(at + kFOutUnits);
        memcpy((void *)&prog_[at], &o, sizeof o);
        P.shift = (int32_t)prog_.size();
        for (int i = 0; i < nb; i++)
            if (gm[(size_t)i]) {
                FShift s{};
                s.gmask = gm[(size_t)i];
                s.off = slot_bytes(col(1u << i), bytes_);
                push(s);
                P.nshift++;
            }
    }

    template <typename T> void push(const T &v)
    {
        static_assert(sizeof(T) == sizeof(FOp), "one unit");
        FOp f;
        memcpy((void *)&f, &v, sizeof f);
        prog_.push_back(f);
    }

    int                    bytes_, look_, nb_ = 0;
    std::vector<FPass>    &passes_;
    std::vector<FOp>      &prog_;
    std::vector<uint32_t>  pack_;
    long double            grow_ = 1.0L;   // the pass's squared growth of the norm ...
    int64_t                exp_ = 0;       // ... and what is to be multiplied back, as a power of two
    std::vector<Row>       X_, Z_;
    std::vector<LRot>      rots_;
    std::vector<Quad>      quads_;
    std::vector<int>       rest_, take_, def_, best_take_, best_def_;
    size_t                 head_ = 0, stop_ = 0;   // rest_ before head_ is done; where a scan ended
    std::vector<uint16_t>  table_;
};

}  // namespace

void frame_plan(const std::vector<FGate> &gates, cd phase, int n, int tb, int anchor_bits, int amp_bytes,
                int lookahead, std::vector<FPass> &passes, std::vector<FOp> &prog)
{
    PassBuilder B(amp_bytes, lookahead, passes, prog);
    B.scale = phase / abs(phase);   // every gate is unitary: its factors' roundings go
    std::vector<const FGate *> rest, cur, later;
    rest.reserve(gates.size());
    for (const FGate &g : gates) rest.push_back(&g);
    const bool resident = n <= tb;
    const int nb = resident ? std::max(n, kFrameRegBits) : tb;
    if (resident) {
        if (!rest.empty() || phase != cd(1.0)) B.build(rest, (1ull << nb) - 1, nb, true);
        return;
    }
    // Tile sets as in plan_passes (batch.cpp): a pass takes, in circuit
    // order, every gate whose X part fits the tile set and that commutes with
    // every gate put off; with lookahead, windows of neighbouring qubits
    // seeded by the first pending X parts outside the anchor compete with the
    // set grown from the anchor, and the one that takes the most gates wins.
    // At most tb - 2 anchor qubits, so that any gate fits an empty pass.
    const int anchor = tb - 2 < anchor_bits ? tb - 2 : anchor_bits;
    const uint64_t anchor_mask = (1ull << anchor) - 1;
    std::vector<Kinds> kinds(gates.size());
    std::vector<uint64_t> need(gates.size());
    for (size_t i = 0; i < gates.size(); i++) {
        kinds[i] = kinds_of(gates[i]);
        need[i] = kinds[i].x | kinds[i].o;
    }
    uint64_t az = 0, ax = 0, ao = 0;   // how any gate acts on the qubits
    for (const Kinds &k : kinds) {
        az |= k.z;
        ax |= k.x;
        ao |= k.o;
    }
    const FGate *g0 = gates.data();
    uint64_t S = 0;
    // the pending gates rest[head, lim) that a pass takes; it ends (at stop)
    // once no gate could commute with all that are put off
    size_t head = 0, stop = 0;
    auto scan = [&](uint64_t S0, size_t lim, std::vector<const FGate *> *take, std::vector<const FGate *> *defer) {
        uint64_t Sx = S0, bz = 0, bx = 0, bo = 0;
        size_t taken = 0, i = head;
        for (; i < lim && ((az & ~(bx | bo)) | (ax & ~(bz | bo)) | (ao & ~(bz | bx | bo))); i++) {
            const size_t id = (size_t)(rest[i] - g0);
            const Kinds &k = kinds[id];
            const bool clash = (k.z & (bx | bo)) | (k.x & (bz | bo)) | (k.o & (bz | bx | bo));
            if (!clash && __builtin_popcountll(Sx | need[id]) <= tb) {
                Sx |= need[id];
                taken++;
                if (take) take->push_back(rest[i]);
            } else {
                bz |= k.z;
                bx |= k.x;
                bo |= k.o;
                if (defer) defer->push_back(rest[i]);
            }
        }
        if (take) S = Sx;
        stop = i;
        return taken;
    };
    std::vector<uint64_t> tried;
    const int free_bits = tb - anchor;
    while (head < rest.size()) {
        const size_t lim = std::min(rest.size(), head + kLookaheadOps);
        uint64_t bestS0 = anchor_mask;
        size_t best = lookahead > 0 ? scan(anchor_mask, lim, nullptr, nullptr) : 0;
        tried.clear();
        int seeds = 0;
        for (size_t i = head; i < rest.size() && seeds < lookahead; i++) {
            const uint64_t nd = need[(size_t)(rest[i] - g0)] & ~anchor_mask;
            if (!nd) continue;
            seeds++;
            const int q = __builtin_ctzll(nd);
            for (const int lo0 : {q, q - free_bits / 2, q - free_bits + 1}) {
                uint64_t S0 = anchor_mask | nd;
                const int lo = lo0 < 0 ? 0 : lo0;
                for (int k = lo; k < n && __builtin_popcountll(S0) < tb; k++) S0 |= 1ull << k;
                for (int k = lo - 1; k >= 0 && __builtin_popcountll(S0) < tb; k--) S0 |= 1ull << k;
                if (std::find(tried.begin(), tried.end(), S0) != tried.end()) continue;
                tried.push_back(S0);
                const size_t c = scan(S0, lim, nullptr, nullptr);
                if (c > best) {
                    best = c;
                    bestS0 = S0;
                }
            }
        }
        cur.clear();
        later.clear();
        scan(bestS0, rest.size(), &cur, &later);
        for (int q = 0; q < n && __builtin_popcountll(S) < nb; q++) S |= 1ull << q;
        B.build(cur, S, nb, later.empty() && stop == rest.size());
        head = stop - later.size();
        std::copy(later.begin(), later.end(), rest.begin() + (long)head);
    }
    if (gates.empty() && phase != cd(1.0)) B.build(cur, (1ull << nb) - 1, nb, true);
}

}  // namespace mlx
