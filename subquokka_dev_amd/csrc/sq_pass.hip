// sq_pass.hip -- the plain sweep (MEM_Runner::run(vector<Gate*>&),
// MEM_Runner.cpp:101-134) as a schedule of register passes.
//
// The planner (plan_register_passes) cuts the gate list into steps: a merged
// step is a run of one-qubit dense and diagonal gates whose dense targets lie
// in the resident qubits -- lane bits 0-2 plus up to pass_qbits + 3 chosen
// qubits, pass_qbits of them in registers and three in the top lane
// positions -- and costs one read and one write of the state
// (kernels/pass.hpp).  The encoder writes each step's ops in the pass's
// virtual positions and folds a controlled phase into the dense gate that
// follows it on either qubit (complex<double>).  Every other gate
// (two-qubit dense, permutations) runs alone with its own kernel, and so does
// a merged step that would cost no more than one pass done gate by gate.
// Per-qubit gate order is kept, so the schedule computes the same map as the
// gates in input order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "subquokka_hip.h"
#include "engine_internal.hpp"
#include "host/planner.hpp"
#include "kernels/pass.hpp"

using sq::LoweredGate;
using sq::OpClass;
using namespace sqk;

namespace {

static_assert(kPassMaxKH <= 5, "PlainLaunch holds five register qubits");
static_assert(kPassLaneHi == 3, "PlainLaunch holds three lane positions");

// The op records of a program, in a byte workspace that outlives the call.
template <typename T> class OpBuffer {
    std::vector<unsigned char> &mem;
    size_t n = 0;

public:
    explicit OpBuffer(std::vector<unsigned char> &m) : mem(m) {}
    PassOp<T> *extend(size_t k) {   // k more records (contents undefined)
        const size_t need = (n + k) * sizeof(PassOp<T>) + alignof(PassOp<T>);
        if (need > mem.size()) {
            // keep the records where alignment puts them in the larger block
            std::vector<unsigned char> next(std::max(need, 2 * mem.size()));
            std::swap(mem, next);
            if (n) std::memcpy(static_cast<void *>(data()), align(next), n * sizeof(PassOp<T>));
        }
        n += k;
        return data() + (n - k);
    }
    void push_back(const PassOp<T> &o) { *extend(1) = o; }
    PassOp<T> *data() { return static_cast<PassOp<T> *>(align(mem)); }
    PassOp<T> &operator[](size_t i) { return data()[i]; }
    PassOp<T> &back() { return data()[n - 1]; }
    size_t size() const { return n; }
    bool empty() const { return n == 0; }

private:
    static void *align(std::vector<unsigned char> &m) {
        const uintptr_t a = alignof(PassOp<T>);
        return reinterpret_cast<void *>((reinterpret_cast<uintptr_t>(m.data()) + a - 1) / a * a);
    }
};

// A gate of a register pass: dense on one qubit, diagonal on one or two (t
// ascending) or a CNOT (t: target, control), in the pass's virtual positions.
struct PassGate {
    OpClass cls;
    int k;
    bool cnot = false;
    int t[2];
    std::complex<double> m[4];
    uint32_t diag_active;
    // the lowered gate with its targets mapped through vpos (sq::relabel)
    PassGate(const LoweredGate &g, const std::vector<int> &vpos)
        : cls(g.cls), k(g.k), t{vpos[g.t[0]], g.k > 1 ? vpos[g.t[1]] : 0}, m{g.m[0], g.m[1], g.m[2], g.m[3]},
          diag_active(g.diag_active) {
        if (cls == OpClass::Dense && k == 2) {
            cnot = true;
            if (sq::cnot_target(g) != g.t[0]) std::swap(t[0], t[1]);
            return;
        }
        if (k == 2 && t[0] > t[1]) {
            std::swap(t[0], t[1]);
            std::swap(m[1], m[2]);
            diag_active = (diag_active & 9u) | ((diag_active & 2u) << 1) | ((diag_active & 4u) >> 1);
        }
    }
};

template <typename T>
void encode_pass_op(const PassGate &g, const std::vector<int> &regs, OpBuffer<T> &ops) {
    constexpr int VB = Traits<T>::VB;
    constexpr int S = VB + 6;
    auto slot = [&](int t) {
        const auto it = std::find(regs.begin(), regs.end(), t);
        return it == regs.end() ? -1 : (int)(it - regs.begin());
    };
    PassOp<T> o{};
    int nc = 0;
    auto push = [&](std::complex<double> z) { o.coef[nc++] = {(T)z.real(), (T)z.imag()}; };
    o.b = -1;
    if (g.cls == OpClass::Dense) {
        for (int i = 0; i < 4; i++) push(g.m[i]);
        const int t = g.t[0];
        // imaginary parts that are exactly zero as stored (in T)
        bool all_real = true;
        for (int i = 0; i < 4; i++) all_real = all_real && o.coef[i].im == (T)0;
        if (t < VB) {
            o.kind = PO_DENSE_VEC;
            o.c = all_real ? 15 : 0;
        } else if (t < S) {
            o.kind = PO_DENSE_LANE;
            o.a = t - VB;
            o.c = all_real ? 15 : 0;
        } else {
            o.kind = PO_DENSE_REG;
            o.a = slot(t);
            o.c = all_real ? 15 : (o.coef[0].im == (T)0 ? 1 : 0);
        }
        ops.push_back(o);
        return;
    }
    // diagonal: entry l = bit(t0) | bit(t1) << 1, t0 < t1.  The op's entries are
    // the gate's entries in the order the kernel reads them; bit k of active
    // is set when entry k is not 1.
    auto entries = [&](int s0, int s1, int s2, int s3) {
        const int src[4] = {s0, s1, s2, s3};
        o.active = 0;
        for (int k = 0; k < 4; k++) {
            push(g.m[src[k]]);
            o.active |= ((g.diag_active >> src[k]) & 1u) << k;
        }
    };
    if (g.k == 1) {
        const int t = g.t[0], j = slot(t);
        if (j >= 0) {            // e[(register bit << 1) | other bit], no other bit
            o.kind = PO_DIAG_REG1;
            o.a = j;
            o.c = 1;             // no lane-dependent bit: factors per register half
            entries(0, 0, 1, 1);
        } else {
            o.kind = PO_DIAG_FREE;
            o.a = t;
            o.c = t >= S;        // a tile bit: the same for the whole wave
            entries(0, 1, 0, 1);
        }
        ops.push_back(o);
        return;
    }
    const int t0 = g.t[0], t1 = g.t[1], j0 = slot(t0), j1 = slot(t1);
    if (j0 >= 0 && j1 >= 0) {
        o.kind = PO_DIAG_REG2;
        o.a = j0;
        o.b = j1;
        entries(0, 1, 2, 3);
    } else if (j0 >= 0) {        // register bit is entry bit 0: e[(r << 1) | y] = d[r | y << 1]
        o.kind = PO_DIAG_REG1;
        o.a = j0;
        o.b = t1;
        o.c = t1 >= S;           // y a tile bit: one factor per register half for the wave
        entries(0, 2, 1, 3);
    } else if (j1 >= 0) {        // register bit is entry bit 1: e = d
        o.kind = PO_DIAG_REG1;
        o.a = j1;
        o.b = t0;
        o.c = t0 >= S;
        entries(0, 1, 2, 3);
    } else {
        o.kind = PO_DIAG_FREE;
        o.a = t0;
        o.b = t1;
        o.c = t0 >= S && t1 >= S;
        entries(0, 1, 2, 3);
    }
    ops.push_back(o);
}

// FP operations the kernel executes per amplitude for one op (an FMA counts
// two): dense pairs take 14 per amplitude in general, 12 with m0 real and 6
// with all four coefficients real; a diagonal factor costs 6 per amplitude it
// multiplies, and register halves, register entries and tile-uniform entries
// whose factor is 1 are skipped.  A controlled phase folded into a dense op
// adds nothing.
template <typename T> double executed_flops(const PassOp<T> &o) {
    const double quarter = __builtin_popcount(o.active & 15u) / 4.0;
    switch (o.kind) {
    case PO_DENSE_REG:
    case PO_DENSE_REG_C: return o.c == 15 ? 6.0 : (o.c == 1 ? 12.0 : 14.0);
    case PO_DENSE_LANE:
    case PO_DENSE_LANE_C:
    case PO_DENSE_VEC: return o.c == 15 ? 6.0 : 14.0;
    case PO_DIAG_FREE: return o.c ? 6.0 * quarter : 6.0;
    case PO_DIAG_REG1: return o.c ? 6.0 * quarter : 3.0 * (((o.active & 3u) != 0) + ((o.active & 12u) != 0));
    case PO_DIAG_REG2: return 6.0 * quarter;
    // the lane factor (or the scalar alone) and the register table: 6 each;
    // forming L x t per amplitude when both are present: 6 more
    case PO_PHASES: return o.b ? (o.a ? 12.0 : 6.0) : 6.0;
    // three shears: 6 FMAs per pair; a scaled lane rotation: one FMA per part
    case PO_ROT_REG: return 6.0;
    case PO_ROT_LANE: return o.a >= 4 ? 6.0 : 4.0;
    default: return 0.0;
    }
}

// A one-qubit dense gate as phase, real rotation, phase:
//   U = g diag(1, zl) R diag(1, zr),   R = [[c, -s], [s, c]],  c, s >= 0,
// i.e. U = g [[c, -s zr], [s zl, c zl zr]].  The pass applies R as three
// shears (6 FMAs per pair) or, on lane bits 0-3, scaled to one FMA per part,
// instead of 14-16 operations per pair for U; the phases of all qubits of a
// pass that fall due together go into one PO_PHASES op.  ok = false when
// the coefficients are already real, or when the product of the factors
// differs from U by more than 1e-15 (a matrix that is not unitary).
struct PhaseSplit {
    bool ok = false;
    std::complex<double> g{1.0, 0.0}, zl{1.0, 0.0}, zr{1.0, 0.0};
    double c = 1.0, s = 0.0;
};
PhaseSplit phase_split(const PassGate &u) {
    PhaseSplit p;
    if (u.cls != OpClass::Dense || u.k != 1) return p;
    bool real = true;
    for (int i = 0; i < 4; i++) real = real && u.m[i].imag() == 0.0;
    if (real) return p;
    const std::complex<double> u00 = u.m[0], u01 = u.m[1], u10 = u.m[2], u11 = u.m[3];
    const double c = std::abs(u00), s = std::abs(u10);
    std::complex<double> g, zl(1.0, 0.0), zr(1.0, 0.0);
    if (c > 0) g = u00 / c;
    else if (s > 0) g = u10 / s;   // zl = 1
    else return p;
    if (s > 0) {
        if (c > 0) zl = u10 * std::conj(g) / s;
        zr = -u01 * std::conj(g) / s;
    } else {
        zr = u11 * std::conj(g) / c;
    }
    const std::complex<double> w[4] = {g * c, -g * s * zr, g * s * zl, g * c * zl * zr};
    for (int i = 0; i < 4; i++)
        if (std::abs(w[i] - u.m[i]) > 1e-15) return p;
    p.ok = true;
    p.g = g; p.zl = zl; p.zr = zr; p.c = c; p.s = s;
    return p;
}

// The rotation [[c, -s], [s, c]] (c, s >= 0, c^2 + s^2 = 1 to rounding: the
// shears reproduce it only then) on virtual position q as an op:
// three shears on a register slot, inside the complex64 vector and on lane
// bits 4-5 (after the swap with register bit 0); on lane bits 0-3 the
// rotation divided by c (or by s when c is small against s), which *scale is
// set to (the caller applies it with the pass's scalar).
template <typename T>
PassOp<T> rotation_op(double c, double s, int q, const std::vector<int> &regs, double &scale) {
    constexpr int VB = Traits<T>::VB;
    constexpr int S = VB + 6;
    PassOp<T> o{};
    o.b = -1;
    scale = 1.0;
    const double k = -s / (1.0 + c);
    o.coef[0] = {(T)k, (T)s};
    if (q < VB) {
        o.kind = PO_ROT_REG;
        o.c = 1;
    } else if (q < S) {
        o.kind = PO_ROT_LANE;
        o.a = q - VB;
        if (o.a < 4) {
            // R / c (one FMA per part; its error stays eps (c|x| + s|p|)) while
            // s / c <= 8 (complex<float>: s / c <= 1), else R / s with the
            // partner's sign flipped on half the lanes; the scale per gate stays
            // above 1/8 (1/sqrt(2)), far from the range limits of the pass
            o.c = (sizeof(T) == 8 ? 8.0 : 1.0) * c >= s ? 0 : 1;
            scale = o.c == 0 ? c : s;
            o.coef[0] = {(T)(o.c == 0 ? s / c : c / s), (T)0};
        }
    } else {
        o.kind = PO_ROT_REG;
        o.a = (int)(std::find(regs.begin(), regs.end(), q) - regs.begin());
    }
    return o;
}

// CP(pi) / CZ as lowered: a two-qubit diagonal whose only entry other than 1
// is -1 (within one ulp: e^{i pi} evaluates to -1 + 1.2e-16 i; leaving out
// that term changes each amplitude by less than one ulp of its magnitude).
bool is_sign_cp(const PassGate &d) {
    return d.cls == OpClass::Diag && d.k == 2 && d.diag_active == 8u && d.m[3].real() == -1.0 &&
           std::abs(d.m[3].imag()) <= 0x1p-52;
}
template <typename T> PassOp<T> sign_op(const PassGate &d, const std::vector<int> &regs, int S) {
    PassOp<T> o{};
    o.kind = PO_SIGN;
    o.pad[0] = o.pad[1] = -1;
    int nt = 0;
    for (int x = 0; x < 2; x++) {
        const int t = d.t[x];
        const auto it = std::find(regs.begin(), regs.end(), t);
        if (t < S) o.a |= 1 << t;
        else if (it != regs.end()) o.b |= 1 << (int)(it - regs.begin());
        else o.pad[nt++] = t;
    }
    return o;
}

template <typename T> PassOp<T> cnot_op(const PassGate &g, const std::vector<int> &regs) {
    constexpr int VB = Traits<T>::VB, S = VB + 6;
    auto slot = [&](int p) {
        const auto it = std::find(regs.begin(), regs.end(), p);
        return it == regs.end() ? -1 : (int)(it - regs.begin());
    };
    PassOp<T> o{};
    o.kind = PO_CNOT;
    const int t = g.t[0], c = g.t[1];
    o.b = t < VB ? 2 : (t < S ? 1 : 0);
    o.a = o.b == 0 ? slot(t) : t - VB;
    o.active = c < S ? 1u : (slot(c) >= 0 ? 0u : 2u);
    o.c = o.active == 0 ? slot(c) : c;
    return o;
}

// Appends a PO_PHASES op (and its coefficient records): fac[p] is the factor
// diag(1, fac[p]) of virtual position p, for p < S and the register slots;
// gs a scalar.  A single register factor goes into a PO_DIAG_REG1 op of its
// own (half the registers), two or more into the 2^KH table.  Returns the FP
// operations per amplitude.
template <typename T>
double emit_phases(const std::complex<double> *fac, const std::vector<int> &regs, int S,
                   std::complex<double> gs, OpBuffer<T> &ops) {
    static_assert(sizeof(PassOp<T>) == 8 * sizeof(cx<T>), "a coefficient record holds 8 coefficients");
    const std::complex<double> one(1.0, 0.0);
    int lane_mask = 0;
    for (int p = 0; p < S; p++)
        if (fac[p] != one) lane_mask |= 1 << p;
    std::vector<int> js;
    for (int j = 0; j < (int)regs.size(); j++)
        if (fac[regs[j]] != one) js.push_back(j);
    double flops = 0;
    if (js.size() == 1) {   // e[(register bit << 1)]: 1 for bit 0, the factor for bit 1
        PassOp<T> o{};
        o.kind = PO_DIAG_REG1;
        o.a = js[0];
        o.b = -1;
        o.c = 1;
        const std::complex<double> z = fac[regs[js[0]]];
        o.coef[0] = o.coef[1] = {(T)1, (T)0};
        o.coef[2] = o.coef[3] = {(T)z.real(), (T)z.imag()};
        o.active = 12u;
        ops.push_back(o);
        flops += executed_flops(o);
    }
    const bool table = js.size() >= 2;
    if (!lane_mask && !table && gs == one) return flops;
    auto rec = [](const std::complex<double> *z, int n) {
        PassOp<T> r{};
        cx<T> w[8];
        for (int i = 0; i < 8; i++) w[i] = {(T)(i < n ? z[i].real() : 1.0), (T)(i < n ? z[i].imag() : 0.0)};
        std::memcpy(static_cast<void *>(&r), w, sizeof w);
        return r;
    };
    PassOp<T> o{};
    o.kind = PO_PHASES;
    o.a = lane_mask;
    o.b = table;
    const int R = 1 << regs.size();
    o.c = (lane_mask ? 1 : 0) + (table ? (R + 7) / 8 : 0);
    const std::complex<double> l0 = lane_mask || !table ? gs : one;   // else the scalar goes into the table
    o.coef[0] = {(T)l0.real(), (T)l0.imag()};
    ops.push_back(o);
    flops += executed_flops(o);
    if (lane_mask) {
        std::complex<double> z[8];
        for (int p = 0; p < 8; p++) z[p] = p < S ? fac[p] : one;
        ops.push_back(rec(z, 8));
    }
    if (table) {
        std::vector<std::complex<double>> t(R, lane_mask ? one : gs);
        for (int r = 0; r < R; r++)
            for (int j : js)
                if ((r >> j) & 1) t[r] *= fac[regs[j]];
        for (int k = 0; k < (R + 7) / 8; k++) ops.push_back(rec(t.data() + 8 * k, std::min(8, R - 8 * k)));
    }
    return flops;
}

// Runs of diagonal gates (PO_DIAG_TAB).  A diagonal gate with entries of
// modulus 1 is a scalar, a phase per qubit and a controlled phase:
//   diag(d0, d1, d2, d3) = d0 diag(1, z0)(t0) diag(1, z1)(t1) diag(1, 1, 1, c)(t0 t1).
// The factors of a run are collected in long double: gates of a layer often
// share their angle, and the rounding of a quotient would then add up over
// them instead of averaging out (21-qubit MaxCut layers, error against 64
// bits: 7e-14 with double factors, 5e-15 as here and as with one op per gate).
struct Ext {
    long double re = 1.0L, im = 0.0L;
    Ext() = default;
    Ext(const std::complex<double> &z) : re(z.real()), im(z.imag()) {}
    Ext(long double r, long double i) : re(r), im(i) {}
    bool one() const { return re == 1.0L && im == 0.0L; }
    Ext operator*(const Ext &o) const { return {re * o.re - im * o.im, re * o.im + im * o.re}; }
    // 1 / z for |z|^2 = 1 + e, |e| <= 1e-9: conj(z) (1 - e + e^2)
    Ext inv() const {
        const long double e = (re * re - 1.0L) + im * im, s = 1.0L - e + e * e;
        return {re * s, -im * s};
    }
    std::complex<double> hi() const { return {(double)re, (double)im}; }
    std::complex<double> lo() const { return {(double)(re - (double)re), (double)(im - (double)im)}; }
};
bool unit_diagonal(const PassGate &d) {
    for (int i = 0; i < (1 << d.k); i++)
        if (!(std::abs(d.m[i].real() * d.m[i].real() + d.m[i].imag() * d.m[i].imag() - 1.0) <= 1e-9)) return false;
    return true;
}

// Where a pass's virtual positions lie.
struct PassMap {
    enum { Lane = 0, Slot = 1, Tile = 2 };
    int S = 0, n = 0, n_regs = 0, n_tile = 0;
    PassMap() = default;
    char kind[64];
    char idx[64];        // lane position / register slot / tile-number bit
    int slot_pos[8];
    PassMap(int S_, int n_, const std::vector<int> &regs) : S(S_), n(n_), n_regs((int)regs.size()) {
        for (int p = 0; p < n; p++) { kind[p] = p < S ? Lane : Tile; idx[p] = (char)p; }
        for (int j = 0; j < n_regs; j++) { kind[regs[j]] = Slot; idx[regs[j]] = (char)j; slot_pos[j] = regs[j]; }
        for (int p = S; p < n; p++) if (kind[p] == Tile) idx[p] = (char)n_tile++;
    }
};

// Diagonal gates of a pass that wait for the next dense gate on one of their
// qubits (they commute with each other and with everything on other qubits),
// in virtual positions.
template <typename T> struct DiagRun {
    static constexpr int VB = Traits<T>::VB, S = VB + 6, NL = 64 << VB;
    using C = std::complex<double>;
    PassMap map;
    std::vector<const PassGate *> gates;
    uint64_t touched = 0;    // positions of the gates
    // which factors the run has: by slot its lane and tile partners, by lane
    // position its higher lane partners, by tile bit its lane and higher tile
    // partners; pairs of slots (bit 8 j + k, j < k); positions with a phase
    uint32_t slot_lane[8] = {}, slot_tile[8] = {}, lane_lane[8] = {}, tile_lane[32] = {}, tile_tile[32] = {};
    uint64_t slot_slot = 0, single = 0;
    bool scalar = false;
    double old_cost = 0;     // one op per gate (unit: all registers times one factor per lane)
    explicit DiagRun(int n) : z(n), pair((size_t)n * n) {}
    void start(const std::vector<int> &regs) { map = PassMap(S, (int)z.size(), regs); }
    void clear() {
        gates.clear();
        touched = slot_slot = single = 0;
        for (uint32_t *a : {slot_lane, slot_tile, lane_lane}) std::fill(a, a + 8, 0u);
        std::fill(tile_lane, tile_lane + 32, 0u);
        std::fill(tile_tile, tile_tile + 32, 0u);
        scalar = false;
        old_cost = 0;
    }

    void add(const PassGate &d) {
        gates.push_back(&d);
        const C one(1.0, 0.0);
        scalar = scalar || d.m[0] != one;
        const int a = d.t[0], ka = map.kind[a], ia = map.idx[a];
        const uint32_t act = d.diag_active;
        touched |= 1ULL << a;
        if (d.m[1] != d.m[0]) single |= 1ULL << a;
        if (d.k == 1) {
            old_cost += 0.15 + (ka == PassMap::Lane ? 1.0 : 0.5 * __builtin_popcount(act & 3u));
            return;
        }
        const int b = d.t[1], kb = map.kind[b], ib = map.idx[b];
        touched |= 1ULL << b;
        if (d.m[2] != d.m[0]) single |= 1ULL << b;
        const double quarter = 0.15 + __builtin_popcount(act & 15u) / 4.0;
        if (ka == PassMap::Slot && kb == PassMap::Slot) {
            slot_slot |= 1ULL << (8 * std::min(ia, ib) + std::max(ia, ib));
            old_cost += quarter;
        } else if (ka == PassMap::Slot || kb == PassMap::Slot) {
            const int j = ka == PassMap::Slot ? ia : ib, ko = ka == PassMap::Slot ? kb : ka, io = ka == PassMap::Slot ? ib : ia;
            (ko == PassMap::Lane ? slot_lane : slot_tile)[j] |= 1u << io;
            const uint32_t half0 = ka == PassMap::Slot ? 5u : 3u;   // entries whose slot bit is 0
            old_cost += ko == PassMap::Tile ? quarter : 0.15 + 0.5 * (((act & half0) != 0) + ((act & ~half0 & 15u) != 0));
        } else if (ka == PassMap::Tile && kb == PassMap::Tile) {
            tile_tile[std::min(ia, ib)] |= 1u << std::max(ia, ib);
            old_cost += quarter;
        } else {
            if (ka == PassMap::Lane && kb == PassMap::Lane) lane_lane[std::min(ia, ib)] |= 1u << std::max(ia, ib);
            else tile_lane[ka == PassMap::Tile ? ia : ib] |= 1u << (ka == PassMap::Tile ? ib : ia);
            old_cost += 1.15;
        }
    }
    bool slot_table(int j) const { return slot_lane[j] || slot_tile[j]; }
    bool tile_singles() const { return (single & ~slot_positions()) >> S; }
    uint64_t slot_positions() const {
        uint64_t m = 0;
        for (int j = 0; j < map.n_regs; j++) m |= 1ULL << map.slot_pos[j];
        return m;
    }
    bool has_tiles() const {
        for (int k = 0; k < map.n_tile; k++) if (tile_tile[k]) return true;
        return tile_singles();
    }
    bool has_all() const {
        if (scalar || (single & ((1ULL << S) - 1)) || has_tiles()) return true;
        for (int p = 0; p < S; p++) if (lane_lane[p]) return true;
        for (int k = 0; k < map.n_tile; k++) if (tile_lane[k]) return true;
        return false;
    }
    // The run as tables, in the unit of old_cost: 0.05 / 0.03 per tile bit's
    // row of lane entries / one entry (half of them are applied), 0.5 + 0.08
    // per row for the products over tile bits.  With fewer than three waves
    // per SIMD nothing hides a table's fetch (about 500 cycles, one
    // multiplication of 32 registers): `late` adds it.
    double cost() const {
        const double late = map.n_tile < 12 ? 1.0 : 0.0;
        double c = 0;
        if (has_all()) {
            c += 1.2 + late;
            for (int k = 0; k < map.n_tile; k++) c += (tile_lane[k] ? 0.05 : 0.0) + (tile_tile[k] ? 0.08 : 0.0);
            if (has_tiles()) c += 0.5 + late;
        }
        for (int j = 0; j < map.n_regs; j++) {
            if (slot_table(j)) c += 0.7 + late + 0.03 * __builtin_popcount(slot_tile[j]);
            else if ((single >> map.slot_pos[j]) & 1) c += 0.65;
        }
        return c + 0.4 * __builtin_popcountll(slot_slot);
    }

    // Appends the run as ops; due[p]: further phases of position p (below S or
    // a slot), may be null.  Returns the FP operations per amplitude.
    double emit(OpBuffer<T> &ops, const C *due) {
        const double flops = emit_tables(ops, due);
        std::fill(z.begin(), z.end(), Ext());
        for (const PassGate *d : gates)
            if (d->k == 2) pair[std::min(d->t[0], d->t[1]) * map.n + std::max(d->t[0], d->t[1])] = Ext();
        return flops;
    }

private:
    std::vector<Ext> z, pair;   // by position; by two positions (the lower one first); 1 outside emit()

    double emit_tables(OpBuffer<T> &ops, const C *due) {
        const int P = map.n;
        Ext g;
        const PassGate *last = nullptr;   // gates of a layer often share their entries
        Ext z0, z1, c;
        for (const PassGate *d : gates) {
            const bool same = last && last->k == d->k && std::equal(d->m, d->m + (1 << d->k), last->m);
            if (!same) {
                const Ext i0 = Ext(d->m[0]).inv();
                z0 = z1 = c = Ext();
                if (d->m[1] != d->m[0]) z0 = Ext(d->m[1]) * i0;
                if (d->k == 2) {
                    if (d->m[2] != d->m[0]) z1 = Ext(d->m[2]) * i0;
                    if (d->m[3] != d->m[0]) c = Ext(d->m[3]) * i0;
                    if (!z0.one() || !z1.one()) c = c * (z0 * z1).inv();
                }
                last = d;
            }
            g = g * Ext(d->m[0]);
            const int a = d->t[0], b = d->t[1];
            if (!z0.one()) z[a] = z[a] * z0;
            if (d->k == 1) continue;
            if (!z1.one()) z[b] = z[b] * z1;
            if (!c.one()) {
                Ext &e = pair[std::min(a, b) * P + std::max(a, b)];
                e = e.one() ? c : e * c;
            }
        }
        if (due)
            for (int p = 0; p < P; p++)
                if (due[p] != C(1.0, 0.0)) {
                    z[p] = z[p] * Ext(due[p]);
                    single |= 1ULL << p;
                }
        int tile_at[32] = {};
        uint64_t slots = slot_positions();
        for (int p = S, k = 0; k < map.n_tile; p++) if (!((slots >> p) & 1)) tile_at[k++] = p;
        auto of_pair = [&](int p, int q) -> const Ext & { return pair[std::min(p, q) * P + std::max(p, q)]; };
        double flops = 0;
        Row row;
        Ext carry;
        for (int j = 0; j < map.n_regs; j++) {
            const int pj = map.slot_pos[j];
            if (!slot_table(j)) {
                if (z[pj].one()) continue;
                PassOp<T> o{};
                o.kind = PO_DIAG_REG1;
                o.a = j;
                o.b = -1;
                o.c = 1;
                o.coef[0] = o.coef[1] = {(T)1, (T)0};
                o.coef[2] = o.coef[3] = {(T)z[pj].re, (T)z[pj].im};
                o.active = 12u;
                ops.push_back(o);
                flops += executed_flops(o);
                continue;
            }
            cx<double> *w = table(ops, j, slot_tile[j], 0, 0, NL + __builtin_popcount(slot_tile[j]));
            lane_row(z[pj], slot_lane[j], [&](int p) -> const Ext & { return of_pair(p, pj); }, row);
            put_row(row, w);
            for (uint32_t m = slot_tile[j]; m; m &= m - 1) put_carry(of_pair(tile_at[__builtin_ctz(m)], pj), w, carry);
            flops += 3.0;
        }
        for (uint64_t m = slot_slot; m; m &= m - 1) {
            const int j = __builtin_ctzll(m) / 8, k = __builtin_ctzll(m) % 8;
            const Ext &e = of_pair(map.slot_pos[j], map.slot_pos[k]);
            PassOp<T> o{};
            o.kind = PO_DIAG_REG2;
            o.a = j;
            o.b = k;
            o.active = 8u;
            o.coef[0] = o.coef[1] = o.coef[2] = {(T)1, (T)0};
            o.coef[3] = {(T)e.re, (T)e.im};
            ops.push_back(o);
            flops += executed_flops(o);
        }
        if (!has_all()) return flops;
        uint32_t rows = 0, tt = 0;
        for (int k = 0; k < map.n_tile; k++) {
            rows |= (uint32_t)(tile_lane[k] != 0) << k;
            tt |= (uint32_t)(tile_tile[k] != 0) << k;
        }
        const bool tiles = has_tiles();
        cx<double> *w = table(ops, -1, rows, tiles, tt,
                              NL * (1 + __builtin_popcount(rows)) + (tiles ? 32 * (1 + __builtin_popcount(tt)) : 0));
        lane_row(g, (uint32_t)(single & ((1ULL << S) - 1)), [&](int p) -> const Ext & { return z[p]; }, row);
        for (int p = 0; p < S; p++)
            for (uint32_t m = lane_lane[p]; m; m &= m - 1) {
                const int q = __builtin_ctz(m), lo = 1 << p, hi = 1 << q;   // p < q
                for (int x = hi; x < NL; x += 2 * hi)
                    for (int y = x + lo; y < x + hi; y += 2 * lo) times(row.re + y, row.im + y, row.re + y, row.im + y, lo, of_pair(p, q));
            }
        put_row(row, w);
        for (uint32_t m = rows; m; m &= m - 1) {
            const int k = __builtin_ctz(m);
            lane_row(Ext(), tile_lane[k], [&](int p) -> const Ext & { return of_pair(p, tile_at[k]); }, row);
            put_row(row, w);
        }
        if (tiles) {
            for (int k = 0; k < 32; k++) put(k < map.n_tile ? z[tile_at[k]] : Ext(), w);
            for (uint32_t m = tt; m; m &= m - 1) {
                const int k = __builtin_ctz(m);
                for (int q = 0; q < 32; q++) {
                    if ((tile_tile[k] >> q) & 1) put_carry(of_pair(tile_at[k], tile_at[q]), w, carry);
                    else put(Ext(), w);
                }
            }
        }
        return flops + 6.0;
    }

    // (r + i m) f for `cnt` values, f in two parts: one rounding of the
    // product, none of f's own
    static void times(const double *r, const double *m, double *ro, double *mo, int cnt, const Ext &f) {
        const double hr = f.hi().real(), hm = f.hi().imag(), lr = f.lo().real(), lm = f.lo().imag();
        for (int x = 0; x < cnt; x++) {
            const double a = r[x], b = m[x];
            ro[x] = (a * hr - b * hm) + (a * lr - b * lm);
            mo[x] = (a * hm + b * hr) + (a * lm + b * lr);
        }
    }
    // by lane index x: the scalar times the factors f(p) of its set bits p of mask
    struct Row {
        double re[NL], im[NL];
    };
    template <typename F> static void lane_row(const Ext &scalar, uint32_t mask, F f, Row &w) {
        w.re[0] = (double)scalar.re;
        w.im[0] = (double)scalar.im;
        for (int p = 0; p < S; p++) {
            const int half = 1 << p;
            if ((mask >> p) & 1) {
                times(w.re, w.im, w.re + half, w.im + half, half, f(p));
            } else {
                std::copy(w.re, w.re + half, w.re + half);
                std::copy(w.im, w.im + half, w.im + half);
            }
        }
    }
    static void put_row(const Row &r, cx<double> *&w) {
        for (int x = 0; x < NL; x++) w[x] = {r.re[x], r.im[x]};
        w += NL;
    }
    static void put(const Ext &f, cx<double> *&w) { *w++ = {(double)f.re, (double)f.im}; }
    // The same for factors that are often equal and whose product over a subset
    // is taken: each entry takes along what the entries before it lost to
    // rounding, so equal factors do not all err the same way.
    static void put_carry(const Ext &f, cx<double> *&w, Ext &carry) {
        const Ext v = f * carry;
        const std::complex<double> r = v.hi();
        carry = v * Ext(r).inv();
        *w++ = {r.real(), r.imag()};
    }
    // Appends the op and room for its `entries`.
    static cx<double> *table(OpBuffer<T> &ops, int slot, uint32_t rows, bool tiles, uint32_t tt, int entries) {
        static_assert(sizeof(PassOp<T>) % sizeof(cx<double>) == 0, "records hold whole table entries");
        PassOp<T> o{};
        o.kind = PO_DIAG_TAB;
        o.a = slot;
        o.b = tiles;
        o.c = (int32_t)((entries * sizeof(cx<double>) + sizeof(PassOp<T>) - 1) / sizeof(PassOp<T>));
        o.active = rows;
        o.pad[0] = (int32_t)tt;
        ops.push_back(o);
        return reinterpret_cast<cx<double> *>(ops.extend(o.c));
    }
};

template <typename T, int KH>
int launch_pass(sq_engine *e, const PassArgs<T> &a) {
    const uint64_t tiles = a.n_tiles * (a.s2 ? 2 : 1);
    const unsigned grid = e->grid_flat(tiles, kBlock / 64);
    if ((uint64_t)grid * (kBlock / 64) < tiles)   // one tile per wave, no grid-stride loop
        return e->fail(SQ_ERR_ARG, "register pass: " + std::to_string(tiles) + " wave tiles exceed one launch");
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_pass<T, KH>), grid, kBlock, 0, e->stream,
                       reinterpret_cast<cx<T> *>(e->d_state), a);
    return e->check_launch("k_pass");
}

// tables: runs of diagonal gates may become PO_DIAG_TAB ops
template <typename T>
int build_plain_t(sq_engine *e, const sq_gate *gates, const std::vector<LoweredGate> &low,
                  PlainProgram &prog, void *dst, size_t dst_cap, bool tables = true) {
    constexpr int VB = Traits<T>::VB;
    constexpr int S = VB + 6;
    const int n = e->n;
    const int kh = e->pass_qbits;
    prog = PlainProgram{};
    prog.n = n;
    prog.kh = kh;
    if (e->sweep_mode == 1 || n < S + kh) {
        prog.per_gate = true;
        return SQ_OK;
    }
    const size_t ng = low.size();
    std::vector<char> mergeable(ng, 0);
    std::vector<uint64_t> need(ng, 0);   // by input qubit
    for (size_t i = 0; i < ng; i++) {
        const LoweredGate &g = low[i];
        if (g.cls == OpClass::Diag && g.k <= 2) {
            mergeable[i] = 1;
        } else if (g.cls == OpClass::Dense) {
            const int t = g.k == 1 ? g.t[0] : sq::cnot_target(g);
            mergeable[i] = t >= 0;
            if (t >= 0) need[i] = 1ULL << t;
        }
    }
    // the top three lane positions may hold any qubit up to bit 27 of the
    // 16-byte slot index (a lane's offset stays a 32-bit one)
    const int moves = std::max(0, std::min(e->lane_moves, kPassLaneHi));
    // The schedule depends on the gates' qubits and classes only: a list
    // with the structure of a recent one (the same circuit again, or with new
    // angles) reuses its schedule; the op records are encoded every call.
    std::vector<int32_t> &key = e->ws_key;
    key.assign({n, S, kh, moves, std::min(n - 1, 27 + VB), e->plan_beam, (int32_t)ng});
    key.reserve(7 + 5 * ng);
    for (size_t i = 0; i < ng; i++) {
        key.push_back(mergeable[i] | (gates[i].nq << 2) | (need[i] ? (__builtin_ctzll(need[i]) + 1) << 8 : 0));
        for (int j = 0; j < gates[i].nq && j < 4; j++) key.push_back(gates[i].q[j]);
    }
    const std::vector<sq::SweepStep> *steps_ptr = nullptr;
    for (size_t c = 0; c < e->plan_cache.size(); c++) {
        if (e->plan_cache[c].key != key) continue;
        if (c) std::rotate(e->plan_cache.begin(), e->plan_cache.begin() + c, e->plan_cache.begin() + c + 1);
        steps_ptr = &e->plan_cache[0].steps;
        break;
    }
    if (!steps_ptr) {
        sq_engine::PlanCacheEntry ent;
        ent.steps = sq::plan_register_passes(std::vector<sq_gate>(gates, gates + ng), mergeable, need, n, S, kh, moves, std::min(n - 1, 27 + VB),
                                             e->plan_beam);
        ent.key = key;
        e->plan_cache.insert(e->plan_cache.begin(), std::move(ent));
        if (e->plan_cache.size() > 4) e->plan_cache.pop_back();
        steps_ptr = &e->plan_cache[0].steps;
    }
    const std::vector<sq::SweepStep> &steps = *steps_ptr;

    OpBuffer<T> ops(e->ws_ops);
    DiagRun<T> run(n);
    std::vector<PassGate> lg;
    std::vector<PhaseSplit> sp;
    std::vector<int> fold_into, folded_from, next;
    std::vector<char> absorbed, zr_done;
    for (const auto &st : steps) {
        double frac = 0;
        for (int gi : st.gates) frac += low[gi].pass_fraction;
        if (!st.merged || frac <= 1.0) {
            for (int gi : st.gates) {
                PlainLaunch l;
                l.gate = gi;
                prog.launches.push_back(l);
            }
            continue;
        }
        // Virtual positions: lane position S-3+k holds qubit st.lanes[k], and
        // that qubit's own position holds the one it displaced.
        std::vector<int> vpos(n);
        for (int q = 0; q < n; q++) vpos[q] = q;
        PlainLaunch l;
        for (int k = 0; k < kPassLaneHi; k++) {
            const int u = S - kPassLaneHi + k;
            const int off = k - (kPassLaneHi - moves);   // st.lanes covers the top `moves` positions
            const int w = off >= 0 ? st.lanes[off] : u;
            if (w != u) std::swap(vpos[u], vpos[w]);
        }
        l.v2l.assign(n, 0);
        for (int q = 0; q < n; q++) l.v2l[vpos[q]] = q;
        // exactly kh register qubits: pad with qubits outside the lane positions
        std::vector<int> regs;
        for (int q : st.regs) regs.push_back(vpos[q]);
        for (int q = 0; q < n && (int)regs.size() < kh; q++)
            if (vpos[q] >= S && std::find(regs.begin(), regs.end(), vpos[q]) == regs.end()) regs.push_back(vpos[q]);
        std::sort(regs.begin(), regs.end());
        l.merged = true;
        l.op_begin = (int)ops.size();
        lg.clear();
        for (int gi : st.gates) lg.emplace_back(low[gi], vpos);
        // next[2 i + x]: the next gate on gate i's x-th target; head[q]: the
        // first one on q (kept at or after the gate being encoded)
        const int N = (int)lg.size();
        std::vector<int> head(n, N);
        next.assign(2 * N, N);
        for (int i = N; i-- > 0;)
            for (int x = 0; x < lg[i].k; x++) {
                next[2 * i + x] = head[lg[i].t[x]];
                head[lg[i].t[x]] = i;
            }
        auto next_on = [&](int i, int q) { return next[2 * i + (lg[i].t[0] == q ? 0 : 1)]; };
        const std::complex<double> one(1.0, 0.0);
        sp.assign(N, PhaseSplit{});
        bool any_split = false;
        if (e->phase_split)
            for (size_t i = 0; i < lg.size(); i++) {
                sp[i] = phase_split(lg[i]);
                any_split = any_split || sp[i].ok;
            }
        // complex<double>: a controlled phase (diagonal, only |11> not 1) whose
        // next gate on either qubit is a dense gate on a register slot or a
        // lane bit goes into that gate's op, with the other qubit as the control
        // (not into a split gate: its rotation runs as shears)
        fold_into.assign(N, -1);
        folded_from.assign(N, -1);
        if constexpr (sizeof(T) == 8) {
            auto in_regs = [&](int t) { return std::find(regs.begin(), regs.end(), t) != regs.end(); };
            for (size_t i = 0; i < lg.size(); i++) {
                const PassGate &d = lg[i];
                if (!(d.cls == OpClass::Diag && d.k == 2 && d.diag_active == 8u)) continue;
                const int j = std::min(next[2 * i], next[2 * i + 1]);   // the next gate on either qubit
                if (j == N) continue;
                const PassGate &u = lg[j];
                if (u.cls == OpClass::Dense && !u.cnot && folded_from[j] < 0 && !sp[j].ok &&
                    (in_regs(u.t[0]) || (u.t[0] >= VB && u.t[0] < S))) {
                    fold_into[i] = j;
                    folded_from[j] = (int)i;
                }
            }
        }
        // Phase split (phase_split above): each dense gate's rotation runs
        // as R; its phases wait per qubit in pend[] until a flush applies all
        // factors due -- placed just before the first gate that needs one, it
        // also takes, for every other resident qubit, the right factor of that
        // qubit's next gate and the one-qubit diagonals before it (all of them
        // diagonal, so they commute up to that gate).  The scalars collect in
        // gpass; the pass ends with a flush of what is left.
        auto resident = [&](int t) { return t < S || std::find(regs.begin(), regs.end(), t) != regs.end(); };
        std::vector<std::complex<double>> pend(n, one);
        absorbed.assign(N, 0);
        zr_done.assign(N, 0);
        std::complex<double> gpass = one;
        auto diag1 = [&](size_t j) {
            const PassGate &d = lg[j];
            return any_split && d.cls == OpClass::Diag && d.k == 1 && resident(d.t[0]) && d.m[0] != 0.0;
        };
        run.start(regs);
        // every factor due before gate `from` (see above), by position
        auto due = [&](int from, std::complex<double> *fac) {
            std::fill(fac, fac + n, one);
            auto take = [&](int q) {
                std::complex<double> f = pend[q];
                pend[q] = one;
                int &h = head[q];
                while (h < from) h = next_on(h, q);
                for (int j = h; j < N; j = next_on(j, q)) {
                    const PassGate &u = lg[j];
                    if (u.cls == OpClass::Diag) {
                        if (diag1(j) && !absorbed[j]) {
                            f *= u.m[1] / u.m[0];
                            gpass *= u.m[0];
                            absorbed[j] = 1;
                        }
                        continue;
                    }
                    if (u.cnot && u.t[1] == q) continue;   // a control: phases pass
                    if (sp[j].ok && !zr_done[j]) {
                        f *= sp[j].zr;
                        zr_done[j] = 1;
                    }
                    break;
                }
                fac[q] = f;
            };
            for (int p = 0; p < S; p++) take(p);
            for (int r : regs) take(r);
        };
        auto flush = [&](int from, bool last) {
            std::complex<double> fac[64];
            due(from, fac);
            l.flops_per_amp += emit_phases<T>(fac, regs, S, last ? gpass : one, ops);
        };
        // The diagonal gates that wait, before gate `from`: as tables when that
        // costs less than one op per gate -- then the phases due go along -- or
        // one op each.
        auto settle = [&](int from) {
            if (run.gates.empty()) return;
            if (tables && run.gates.size() > 1 && run.cost() < 0.9 * run.old_cost) {
                std::complex<double> fac[64];
                if (any_split) due(from, fac);
                l.flops_per_amp += run.emit(ops, any_split ? fac : nullptr);
            } else {
                for (const PassGate *d : run.gates) {
                    encode_pass_op<T>(*d, regs, ops);
                    l.flops_per_amp += executed_flops(ops.back());
                }
            }
            run.clear();
        };
        for (size_t i = 0; i < lg.size(); i++) {
            if (fold_into[i] >= 0) continue;   // applied inside the dense gate's op: no work of its own
            if (diag1(i)) {                    // a factor of its qubit's pending phase
                if (!absorbed[i]) {
                    pend[lg[i].t[0]] *= lg[i].m[1] / lg[i].m[0];
                    gpass *= lg[i].m[0];
                    absorbed[i] = 1;
                }
                continue;
            }
            // Rotations as shears (or scaled) for both types; CP(pi) as a sign
            // flip for complex<double> only: complex<float> keeps the diagonal
            // op, which measured faster there (FP32 arithmetic is cheap next to
            // the bit operations)
            constexpr bool kShears = true, kSigns = sizeof(T) == 8;
            if (kSigns && any_split && is_sign_cp(lg[i])) {   // CP(pi): a sign flip
                ops.push_back(sign_op<T>(lg[i], regs, S));
                continue;
            }
            if (lg[i].cls == OpClass::Diag) {
                if (tables && unit_diagonal(lg[i])) {
                    run.add(lg[i]);
                    continue;
                }
            } else if ((run.touched >> lg[i].t[0]) & 1) {
                settle(i);
            }
            if (lg[i].cnot) {
                if (pend[lg[i].t[0]] != one) flush(i, false);
                ops.push_back(cnot_op<T>(lg[i], regs));
                continue;
            }
            PassGate gi = lg[i];
            if (any_split && gi.cls == OpClass::Dense) {
                const int q = gi.t[0];
                std::complex<double> need = pend[q];
                if (sp[i].ok && !zr_done[i]) need *= sp[i].zr;
                if (need != one) flush(i, false);
                pend[q] = one;
                zr_done[i] = 1;
                if (sp[i].ok) {
                    pend[q] = sp[i].zl;
                    gpass *= sp[i].g;
                    const double c = sp[i].c, s = sp[i].s;
                    if (c == 1.0 && s == 0.0) continue;   // R = I
                    if (kShears && std::abs(c * c + s * s - 1.0) <= 1e-15) {   // a rotation: shears or scaled
                        double scale = 1.0;
                        ops.push_back(rotation_op<T>(c, s, q, regs, scale));
                        gpass *= scale;
                        l.flops_per_amp += executed_flops(ops.back());
                        continue;
                    }
                    // complex<float>, or a multiple of a rotation (a matrix that
                    // is not unitary): the real 2x2 product
                    gi.m[0] = c;
                    gi.m[1] = -s;
                    gi.m[2] = s;
                    gi.m[3] = c;
                }
            }
            encode_pass_op<T>(gi, regs, ops);
            if constexpr (sizeof(T) == 8) if (folded_from[i] >= 0) {
                const PassGate &d = lg[folded_from[i]];
                PassOp<T> &o = ops.back();
                const int ctl = gi.t[0] == d.t[0] ? d.t[1] : d.t[0];
                const auto it = std::find(regs.begin(), regs.end(), ctl);
                const bool lane_target = o.kind == PO_DENSE_LANE;
                o.kind = lane_target ? PO_DENSE_LANE_C : PO_DENSE_REG_C;
                if (it != regs.end()) { o.active = 0; o.b = (int)(it - regs.begin()); }
                else { o.active = ctl < S ? 1 : 2; o.b = ctl; }
                // A real gate stays real with a real phase.  A phase within one
                // ulp of the real axis counts as real: CP(pi) evaluates to
                // e^{i pi} = -1 + 1.2e-16 i, and leaving out that term changes
                // each amplitude by less than one ulp of its magnitude.
                const std::complex<double> ph = d.m[3];
                const bool ph_real = std::abs(ph.imag()) <= 0x1p-52 * std::abs(ph.real());
                const bool real = o.c == 15 && ph_real;
                o.c = real ? 15 : (!lane_target && o.coef[0].im == (T)0 ? 1 : 0);
                o.coef[kPassFoldPhase] = {(T)ph.real(), real ? (T)0 : (T)ph.imag()};
            }
            l.flops_per_amp += executed_flops(ops.back());
        }
        settle(N);
        if (any_split) flush(N, true);
        l.n_ops = (int)ops.size() - l.op_begin;
        for (int j = 0; j < kh; j++) l.hpos[j] = regs[j];
        prog.launches.push_back(l);
    }

    // op census of this program (sq_pass_census)
    e->pass_census.fill(0);
    for (size_t oi = 0; oi < ops.size(); oi++) {
        const PassOp<T> &o = ops[oi];
        int idx = -1;
        switch (o.kind) {
        case PO_DENSE_REG: idx = 0; break;
        case PO_DENSE_LANE: idx = o.a < 4 ? 1 : 2; break;
        case PO_DENSE_VEC: idx = 3; break;
        case PO_DIAG_FREE: idx = 4; break;
        case PO_DIAG_REG1: idx = 5; break;
        case PO_DIAG_REG2: idx = 6; break;
        case PO_PHASES: idx = 7; oi += o.c; break;   // past its coefficient records
        case PO_DIAG_TAB: idx = o.a < 0 ? 4 : 5; oi += o.c; break;   // past its tables
        case PO_CNOT: idx = o.b == 2 ? 3 : (o.b == 0 ? 0 : (o.a < 4 ? 1 : 2)); break;
        case PO_ROT_REG: idx = o.c == 1 ? 3 : 0; break;
        case PO_ROT_LANE: idx = o.a < 4 ? 1 : 2; break;
        case PO_SIGN: idx = o.b == 0 ? 4 : (__builtin_popcount((unsigned)o.b) == 1 ? 5 : 6); break;
        case PO_DENSE_REG_C:
        case PO_DENSE_LANE_C: {
            const int t = o.kind == PO_DENSE_REG_C ? 0 : (o.a < 4 ? 1 : 2);
            const int c = o.active == 0 ? (o.b == 0 ? 0 : 1) : (o.active == 1 ? 2 : 3);
            idx = 8 + 4 * t + c;
            break;
        }
        default: break;
        }
        if (idx >= 0) e->pass_census[idx]++;
    }

    // upload the program once (in stream order: earlier launches may still read the old one)
    const size_t bytes = ops.size() * sizeof(PassOp<T>) + 256;
    if (dst) {   // caller-owned buffer: never grown
        // (tables can take more records than the gates they stand for)
        if (ops.size() * sizeof(PassOp<T>) > dst_cap && tables)
            return build_plain_t<T>(e, gates, low, prog, dst, dst_cap, false);
        if (ops.size() * sizeof(PassOp<T>) > dst_cap)
            return e->fail(SQ_ERR_ARG, "the register-pass program (" + std::to_string(ops.size() * sizeof(PassOp<T>)) +
                                           " bytes) exceeds the " + std::to_string(dst_cap) + "-byte scratch");
        prog.d_ops = dst;
        if (!ops.empty()) {
            if (hipStreamSynchronize(e->stream) != hipSuccess) return e->fail(SQ_ERR_HIP, "stream sync");
            hipError_t he = hipMemcpy(dst, ops.data(), ops.size() * sizeof(PassOp<T>), hipMemcpyHostToDevice);
            if (he != hipSuccess) return e->hip_fail(he, "hipMemcpy(pass program to scratch)");
        }
        return SQ_OK;
    }
    if (!ops.empty()) {
        if (bytes > e->passprog_cap) {
            if (hipStreamSynchronize(e->stream) != hipSuccess) return e->fail(SQ_ERR_HIP, "stream sync");
            if (e->d_passprog) (void)hipFree(e->d_passprog);
            e->d_passprog = nullptr;
            e->passprog_cap = 0;
            hipError_t he = hipMalloc(&e->d_passprog, bytes * 2);
            if (he != hipSuccess) return e->hip_fail(he, "hipMalloc(pass program)");
            e->passprog_cap = bytes * 2;
        }
        if (int rc = e->upload(e->d_passprog, ops.data(), ops.size() * sizeof(PassOp<T>))) return rc;
    }
    prog.d_ops = e->d_passprog;
    return SQ_OK;
}

// Runs a program on the engine's current state buffer (e->n must be the
// program's n), and on e->d_state2 too when that is set (one launch covers
// both); its op records are at prog.d_ops.
template <typename T>
int run_plain_t(sq_engine *e, const PlainProgram &prog, const std::vector<LoweredGate> &low) {
    constexpr int VB = Traits<T>::VB;
    constexpr int S = VB + 6;
    const int n = e->n, kh = prog.kh;
    if (n != prog.n) return e->fail(SQ_ERR_ARG, "internal: pass program planned for another size");
    // one launch per gate: on each state in turn
    auto apply_one = [&](const LoweredGate &g) {
        int rc = e->apply_lowered(g);
        if (rc || !e->d_state2) return rc;
        std::swap(e->d_state, e->d_state2);
        rc = e->apply_lowered(g);
        std::swap(e->d_state, e->d_state2);
        return rc;
    };
    if (prog.per_gate) {
        for (const auto &g : low) {
            int rc = apply_one(g);
            if (rc) return rc;
        }
        return SQ_OK;
    }
    const PassOp<T> *dops = reinterpret_cast<const PassOp<T> *>(prog.d_ops);
    char nm[48];
    std::snprintf(nm, sizeof nm, "pass%d_%s", kh, e->dtype == SQ_C128 ? "c128" : "c64");
    const double vecs = e->d_state2 ? 2.0 : 1.0;
    const double bytes = 2.0 * e->amp_bytes() * std::ldexp(1.0, n) * vecs;
    for (const auto &l : prog.launches) {
        if (!l.merged) {
            int rc = apply_one(low[l.gate]);
            if (rc) return rc;
            continue;
        }
        if (l.n_ops == 0) continue;   // the kernel reads its first op unconditionally
        PassArgs<T> a{};
        a.s2 = reinterpret_cast<cx<T> *>(e->d_state2);
        a.ops = dops + l.op_begin;
        a.n_ops = l.n_ops;
        a.n_tile_bits = n - S - kh;
        a.n_tiles = 1ULL << a.n_tile_bits;
        if ((int)l.v2l.size() != n || a.n_tile_bits > kPassMaxTileBits) return e->fail(SQ_ERR_ARG, "internal: pass layout");
        // the qubit a virtual position stands for lies at its own index bit
        for (int j = 0; j < kh; j++) {
            a.hpos[j] = l.hpos[j];
            a.reg_pos[j] = l.v2l[l.hpos[j]];
        }
        for (int k = 0; k < 6; k++) {
            // the kernel's lane offset holds slot bits up to kPassMaxSlotBit only
            a.lane_pos[k] = l.v2l[VB + k] - VB;
            if (a.lane_pos[k] < 0 || a.lane_pos[k] > kPassMaxSlotBit)
                return e->fail(SQ_ERR_ARG, "internal: lane position out of range");
        }
        for (int v = S, k = 0; v < n; v++) {
            if (std::find(l.hpos, l.hpos + kh, v) != l.hpos + kh) continue;
            a.tile_pos[k++] = l.v2l[v];
        }
        int slot = e->stat_begin(nm, bytes, l.flops_per_amp * std::ldexp(1.0, n) * vecs);
        int rc;
        switch (kh) {
        case 1: rc = launch_pass<T, 1>(e, a); break;
        case 2: rc = launch_pass<T, 2>(e, a); break;
        case 3: rc = launch_pass<T, 3>(e, a); break;
        case 4: rc = launch_pass<T, 4>(e, a); break;
        case 5: rc = launch_pass<T, 5>(e, a); break;
        default: rc = e->fail(SQ_ERR_ARG, "internal: bad pass width");
        }
        e->stat_end(slot);
        if (rc) return rc;
    }
    return SQ_OK;
}

}  // namespace

int sq_engine::build_plain(const sq_gate *gates, const std::vector<LoweredGate> &low, PlainProgram &prog,
                           void *dst, size_t dst_cap) {
    return dtype == SQ_C128 ? build_plain_t<double>(this, gates, low, prog, dst, dst_cap, !keep_order)
                            : build_plain_t<float>(this, gates, low, prog, dst, dst_cap, !keep_order);
}

// The second state buffer of the out-of-place permutation pass, allocated
// once when a second copy of the state fits in HBM with room to spare.
// SQ_ERR_UNSUPPORTED (no error recorded) when it does not.
int sq_engine::ensure_alt() {
    if (d_alt) return SQ_OK;
    if (out_of_core() || !bitperm_ok) return SQ_ERR_UNSUPPORTED;
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) { (void)hipGetLastError(); return SQ_ERR_UNSUPPORTED; }
    if (free_b < state_bytes() + ((size_t)4 << 30)) return SQ_ERR_UNSUPPORTED;
    if (hipMalloc(&d_alt, state_bytes()) != hipSuccess) {
        (void)hipGetLastError();
        d_alt = nullptr;
        return SQ_ERR_UNSUPPORTED;
    }
    return SQ_OK;
}

int sq_engine::run_plain_program(const PlainProgram &prog, const std::vector<LoweredGate> &low) {
    return dtype == SQ_C128 ? run_plain_t<double>(this, prog, low) : run_plain_t<float>(this, prog, low);
}

// keep_order (complex64 gradients): CNOTs as H_t CZ H_t with exact 1/sqrt(2)
// coefficients instead of PO_CNOT.  A complex64 gradient carries the rounding
// of its forward sweep (1e-6) into FP64 results, and callers compare those
// between versions far more closely; so that sweep rounds as it always has.
bool sq_engine::expand_cnots(const sq_gate *gates, const std::vector<LoweredGate> &low,
                             std::vector<sq_gate> &g2, std::vector<LoweredGate> &l2) const {
    const int S = (dtype == SQ_C64 ? 1 : 0) + 6;
    if (sweep_mode != 0 || n < S + pass_qbits) return false;   // no register passes
    bool any = false;
    for (const auto &g : low) any = any || sq::cnot_target(g) >= 0;
    if (!any) return false;
    const double s = 0.70710678118654752440;
    g2.clear();
    l2.clear();
    for (size_t i = 0; i < low.size(); i++) {
        const int t = sq::cnot_target(low[i]);
        if (t < 0) {
            g2.push_back(gates[i]);
            l2.push_back(low[i]);
            continue;
        }
        LoweredGate h{};
        h.cls = OpClass::Dense;
        h.k = 1;
        h.t[0] = t;
        h.m[0] = h.m[1] = h.m[2] = s;
        h.m[3] = -s;
        h.pass_fraction = 1.0;
        h.name = "H (CNOT)";
        LoweredGate cz{};
        cz.cls = OpClass::Diag;
        cz.k = 2;
        cz.t[0] = low[i].t[0];
        cz.t[1] = low[i].t[1];
        cz.m[0] = cz.m[1] = cz.m[2] = 1.0;
        cz.m[3] = -1.0;
        cz.diag_active = 8u;
        cz.pass_fraction = 0.25;
        cz.name = "CZ (CNOT)";
        sq_gate gh = gates[i], gz = gates[i];
        gh.kind = SQ_GATE_U1;
        gh.nq = 1;
        gh.q[0] = t;
        gz.kind = SQ_GATE_CP;
        gz.q[0] = cz.t[0];
        gz.q[1] = cz.t[1];
        g2.insert(g2.end(), {gh, gz, gh});
        l2.insert(l2.end(), {h, cz, h});
    }
    return true;
}

// A SWAP (or VSWAP) in a plain list is half a pass of its own and ends the
// passes around it.  With register passes it costs nothing: the later gates
// take the swapped qubits, and one in-place permutation at the end puts the
// bits where the list leaves them (20-qubit QFT, ten SWAPs: 60 us -> 8 us).
bool sq_engine::relabel_swaps(const sq_gate *gates, const std::vector<LoweredGate> &low, std::vector<sq_gate> &g2,
                              std::vector<LoweredGate> &l2, std::vector<int> &sigma) const {
    const int S = (dtype == SQ_C64 ? 1 : 0) + 6;
    if (keep_order || sweep_mode != 0 || n < S + pass_qbits || lane_moves == 0) return false;   // lane_moves 0: data stays in its lanes
    bool any = false;
    for (const auto &g : low) any = any || g.cls == OpClass::Perm;
    if (!any) return false;
    sigma.resize(n);
    for (int p = 0; p < n; p++) sigma[p] = p;
    g2.clear();
    l2.clear();
    g2.reserve(low.size());
    l2.reserve(low.size());
    for (size_t i = 0; i < low.size(); i++) {
        if (low[i].cls == OpClass::Perm) {
            for (int j = 0; j < low[i].n_pairs; j++) std::swap(sigma[low[i].t[2 * j]], sigma[low[i].t[2 * j + 1]]);
            continue;
        }
        g2.push_back(gates[i]);
        for (int j = 0; j < gates[i].nq; j++) g2.back().q[j] = sigma[gates[i].q[j]];
        l2.push_back(low[i]);
        sq::relabel(l2.back(), sigma);
    }
    return true;
}

int sq_engine::run_plain(const sq_gate *gates, const std::vector<LoweredGate> &low, void *dst, size_t dst_cap) {
    std::vector<sq_gate> g1;
    std::vector<LoweredGate> l1;
    std::vector<int> sigma;
    const bool sw = relabel_swaps(gates, low, g1, l1, sigma);
    const sq_gate *g = sw ? g1.data() : gates;
    const std::vector<LoweredGate> *l = sw ? &l1 : &low;
    std::vector<sq_gate> g2;
    std::vector<LoweredGate> l2;
    if (keep_order && expand_cnots(g, *l, g2, l2)) {
        g = g2.data();
        l = &l2;
    }
    PlainProgram prog;
    int rc = build_plain(g, *l, prog, dst, dst_cap);
    if (!rc) rc = run_plain_program(prog, *l);
    if (rc || !sw) return rc;
    std::vector<int> perm(n);   // bit p is at sigma[p]: every bit moves home
    for (int p = 0; p < n; p++) perm[sigma[p]] = p;
    return bit_permute_in_place(perm);
}

int sq_engine::apply_plain(const sq_gate *gates, size_t n_gates, const std::vector<LoweredGate> &low) {
    if (low.size() != n_gates) return fail(SQ_ERR_ARG, "internal: lowered list of another size");
    return run_plain(gates, low, nullptr, 0);
}

// ---------------------------------------------------------------------------
// sq_apply_gates_noalloc: the plain sweep with its register-pass program in a
// fixed device array instead of the engine's growable buffer, so the call
// allocates nothing.  Every engine on a device shares that device's copy of
// the array; it keeps the last call's program.  Calls that overlap on one
// device (two host threads, or two engines on different streams) race on it.
// ---------------------------------------------------------------------------

namespace {

constexpr size_t kScratchBytes = (size_t)4 << 20;   // 32768 complex128 / 65536 complex64 op records
constexpr int kScratchDevices = 64;

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

std::mutex scratch_mu;
void *scratch_addr[kScratchDevices] = {};   // per device: the array's device address

}  // namespace

// Called by sq_create with the engine's device current.  The array's name is
// a host-side stand-in; its device address (one per device) comes from
// hipGetSymbolAddress, once per device.
int sq_engine::setup_scratch() {
    if (device < 0 || device >= kScratchDevices) return fail(SQ_ERR_ARG, "device ordinal beyond the scratch table");
    std::lock_guard<std::mutex> lock(scratch_mu);
    if (!scratch_addr[device]) {
        void *p = nullptr;
        const hipError_t he = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (he != hipSuccess || !p) return hip_fail(he != hipSuccess ? he : hipErrorInvalidValue, "hipGetSymbolAddress(scratch)");
        scratch_addr[device] = p;
    }
    d_scratch = scratch_addr[device];
    return SQ_OK;
}

extern "C" int sq_apply_gates_noalloc(sq_engine *e, const sq_gate *gates, uint64_t n) {
    if (!e || (!gates && n)) return SQ_ERR_ARG;
    if (e->out_of_core()) return e->fail(SQ_ERR_UNSUPPORTED, "sq_apply_gates_noalloc needs an HBM-resident state");
    if (!e->d_scratch) return e->fail(SQ_ERR_HIP, "scratch array not set up for this device");
    if (hipSetDevice(e->device) != hipSuccess) return e->fail(SQ_ERR_HIP, "hipSetDevice");
    // validate everything first so a bad line (or a program too large for the
    // scratch) leaves the state untouched
    if (int rc = e->lower_list(gates, n)) return rc;
    return e->run_plain(gates, e->ws_low, e->d_scratch, kScratchBytes);
}

extern "C" int sq_pass_census(sq_engine *e, int64_t *counts, int32_t cap, int32_t *n_out) {
    if (!e || (cap > 0 && !counts)) return SQ_ERR_ARG;
    const int32_t n = (int32_t)e->pass_census.size();
    if (n_out) *n_out = n;
    for (int32_t i = 0; i < std::min(cap, n); i++) counts[i] = e->pass_census[i];
    return cap < n ? SQ_ERR_ARG : SQ_OK;
}
