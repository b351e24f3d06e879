// sq_adjoint.hip -- energy and adjoint gradient of the hardware-efficient
// ansatz (layers x [RY on every qubit, RZ on every qubit, CNOT ring
// i -> (i+1) mod n]) for H = sum_i Z_i Z_{i+1 mod n}.  No reference
// counterpart: it reuses the engine's rotation matrices (RY, RZ as in
// circuit.cpp:2734-2795) and its state in HBM.
//
// Forward: the gates in order on the engine's state, saving an FP64 copy of
// the state after every `checkpoint_every` layers.  Backward (reverse sweep):
// lambda = H psi; for each gate from last to first, one pass over psi and
// lambda computes the parameter's derivative Im<lambda|P|psi> (FP64 block
// partials) and un-applies the gate to both.  At a checkpoint boundary psi is
// reset to the saved FP64 state, so rounding drift of the un-applied state
// (complex64) is bounded by checkpoint_every layers.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <unordered_map>
#include <vector>

#include "subquokka_hip.h"
#include "engine_internal.hpp"
#include "kernels/adjoint.hpp"
#include "kernels/hea.hpp"
#include "kernels/reduce.hpp"
#include "host/gate_lowering.hpp"

using sq::LoweredGate;
using namespace sqk;

namespace {

int ensure(sq_engine *e, void **buf, size_t *cap, size_t bytes, const char *what) {
    if (bytes <= *cap) return SQ_OK;
    if (*buf) hipFree(*buf);
    *buf = nullptr;
    *cap = 0;
    hipError_t he = hipMalloc(buf, bytes);
    if (he != hipSuccess) return e->hip_fail(he, what);
    *cap = bytes;
    return SQ_OK;
}

template <typename T>
int cnot(sq_engine *e, cx<T> *x, cx<T> *y, int c, int t) {
    AdjCnotArgs a{};
    a.n_quads = 1ULL << (e->n - 2);
    a.ctrl = c; a.targ = t;
    a.lo = std::min(c, t); a.hi = std::max(c, t);
    const double bytes = (y ? 2.0 : 1.0) * e->amp_bytes() * std::ldexp(1.0, e->n);   // half of each state
    int slot = e->stat_begin(y ? "adj_cnot2" : "cnot", bytes);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_cnot2<T>), e->grid_flat(a.n_quads, kBlock), kBlock, 0, e->stream, x, y, a);
    e->stat_end(slot);
    return e->check_launch("k_cnot2");
}

sq_gate rotation(int kind, int q, double theta) {
    sq_gate g{};
    g.kind = kind;
    g.nq = 1;
    g.q[0] = q;
    g.param = theta;
    return g;
}

template <typename T>
int forward(sq_engine *e, int layers, const double *theta, int ckpt_every, cx<double> *ckpt) {
    const int n = e->n;
    int rc = sq_init_zero(e);
    if (rc) return rc;
    cx<T> *psi = reinterpret_cast<cx<T> *>(e->d_state);
    for (int l = 0; l < layers; l++) {
        for (int half = 0; half < 2; half++)
            for (int q = 0; q < n; q++) {
                LoweredGate lg;
                rc = e->lower(rotation(half == 0 ? SQ_GATE_RY : SQ_GATE_RZ, q, theta[(size_t)l * 2 * n + half * n + q]), lg);
                if (!rc) rc = e->apply_lowered(lg);
                if (rc) return rc;
            }
        if (n > 1)
            for (int q = 0; q < n; q++) {
                rc = cnot<T>(e, psi, nullptr, q, (q + 1) % n);
                if (rc) return rc;
            }
        if (ckpt && ckpt_every > 0 && (l + 1) % ckpt_every == 0 && l + 1 < layers) {
            const int slot = (l + 1) / ckpt_every - 1;
            const uint64_t na = e->n_amps();
            hipLaunchKernelGGL(HIP_KERNEL_NAME(k_convert<T, double>), e->grid_for(na, kBlock), kBlock, 0, e->stream,
                               psi, ckpt + (size_t)slot * na, na);
            rc = e->check_launch("checkpoint");
            if (rc) return rc;
        }
    }
    return SQ_OK;
}

// States of at most one wave row: one launch per gate and per pair of rotations.
template <typename T>
int gradient_small(sq_engine *e, int layers, const double *theta, int ckpt_every, double *energy, double *grad) {
    const int n = e->n;
    const uint64_t na = e->n_amps();
    const int n_ckpt = (grad && ckpt_every > 0) ? std::max(0, (layers - 1) / ckpt_every) : 0;
    const unsigned grid = (unsigned)std::min<uint64_t>(kRedBlocks, std::max<uint64_t>(1, (na / 2 + kBlock - 1) / kBlock));
    const size_t n_params = (size_t)2 * n * layers;
    int rc = SQ_OK;
    if (grad) {
        rc = ensure(e, &e->d_aux, &e->aux_cap, e->state_bytes(), "hipMalloc(lambda)");
        if (!rc && n_ckpt)
            rc = ensure(e, &e->d_ckpt, &e->ckpt_cap, (size_t)n_ckpt * na * sizeof(cx<double>), "hipMalloc(checkpoints)");
        if (!rc) rc = ensure(e, &e->d_gradpart, &e->gradpart_cap, n_params * grid * sizeof(double), "hipMalloc(gradient partials)");
        if (rc) return rc;
    }
    cx<double> *ckpt = n_ckpt ? static_cast<cx<double> *>(e->d_ckpt) : nullptr;
    rc = forward<T>(e, layers, theta, ckpt_every, ckpt);
    if (rc) return rc;
    double v[2];
    rc = e->norm_zz(v);
    if (rc) return rc;
    if (energy) *energy = v[1];
    if (!grad) return SQ_OK;

    cx<T> *psi = reinterpret_cast<cx<T> *>(e->d_state);
    cx<T> *lam = reinterpret_cast<cx<T> *>(e->d_aux);
    double *part = static_cast<double *>(e->d_gradpart);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_apply_zz_ring<T>), e->grid_for(na, kBlock), kBlock, 0, e->stream, psi, lam, na, n);
    rc = e->check_launch("k_apply_zz_ring");
    if (rc) return rc;
    for (int l = layers - 1; l >= 0; l--) {
        if (ckpt && (l + 1) % ckpt_every == 0 && l + 1 < layers) {
            const int slot = (l + 1) / ckpt_every - 1;   // state after layer l
            hipLaunchKernelGGL(HIP_KERNEL_NAME(k_convert<double, T>), e->grid_for(na, kBlock), kBlock, 0, e->stream,
                               ckpt + (size_t)slot * na, psi, na);
            rc = e->check_launch("re-anchor");
            if (rc) return rc;
        }
        if (n > 1)
            for (int q = n - 1; q >= 0; q--) {
                rc = cnot<T>(e, psi, lam, q, (q + 1) % n);
                if (rc) return rc;
            }
        // each qubit's RZ then RY, qubits in reverse order (rotations on
        // different qubits commute)
        for (int q = n - 1; q >= 0; q--) {
            const size_t py = (size_t)l * 2 * n + q, pz = py + n;
            AdjRot2Args a{};
            a.n_pairs = na / 2;
            a.q = q;
            a.cz = std::cos(theta[pz] / 2);
            a.sz = std::sin(theta[pz] / 2);
            a.cy = std::cos(theta[py] / 2);
            a.sy = std::sin(theta[py] / 2);
            int slot = e->stat_begin("adj_rot2", 4.0 * e->amp_bytes() * (double)na);
            hipLaunchKernelGGL(HIP_KERNEL_NAME(k_adj_rot2<T>), grid, kBlock, 0, e->stream, psi, lam, a, part + py * grid,
                               (uint64_t)n * grid);
            e->stat_end(slot);
            rc = e->check_launch("k_adj_rot2");
            if (rc) return rc;
        }
    }
    std::vector<double> h(n_params * grid);
    hipError_t he = hipMemcpyAsync(h.data(), part, h.size() * sizeof(double), hipMemcpyDeviceToHost, e->stream);
    if (he == hipSuccess) he = hipStreamSynchronize(e->stream);
    if (he != hipSuccess) return e->hip_fail(he, "gradient partials");
    for (size_t p = 0; p < n_params; p++) {
        double s = 0;
        for (unsigned b = 0; b < grid; b++) s += h[p * grid + b];
        grad[p] = s;
    }
    return SQ_OK;
}


// The ansatz as k_hea passes: qubit sets whose bits are resident together --
// the vector, the lanes and KH register bits first, then KH + 3 qubits at a
// time (KH in register slots, three in the movable lane positions) -- and, per
// layer, one pass per set for the rotations and one per set for the ring.
// The gates keep the list's order: RY on qubit 0, 1, ..., RZ on qubit 0, 1,
// ... (any position), CNOT 0 -> 1, 1 -> 2, ...; the reverse sweep the opposite.
struct HeaSet {
    std::vector<int> qubits;     // ascending
    std::vector<int> vpos;       // qubit -> virtual position
    HeaArgs layout{};
};
template <typename T> struct HeaPlan {
    static constexpr int VB = Traits<T>::VB, S = VB + 6;
    int n, kh;
    std::vector<HeaSet> sets;
    HeaPlan(int n_, int kh_) : n(n_), kh(kh_) {
        for (int q = 0; q < n;) {
            HeaSet st;
            const int cnt = std::min(n - q, sets.empty() ? S + kh : kh + kPassLaneHi);
            for (int i = 0; i < cnt; i++) st.qubits.push_back(q++);
            std::vector<int> &vpos = st.vpos;
            vpos.resize(n);
            for (int i = 0; i < n; i++) vpos[i] = i;
            std::vector<int> regs;
            if (sets.empty()) {
                for (int j = 0; j < kh; j++) regs.push_back(S + j);
            } else {
                // the lowest excess qubits take lane positions (runs stay long)
                const int moved = std::max(0, cnt - kh);
                for (int i = 0; i < moved; i++) std::swap(vpos[S - kPassLaneHi + i], vpos[st.qubits[i]]);
                for (int i = moved; i < cnt; i++) regs.push_back(vpos[st.qubits[i]]);
                for (int p = S; p < n && (int)regs.size() < kh; p++)
                    if (std::find(regs.begin(), regs.end(), p) == regs.end()) regs.push_back(p);
                std::sort(regs.begin(), regs.end());
            }
            std::vector<int> v2l(n);
            for (int i = 0; i < n; i++) v2l[vpos[i]] = i;
            HeaArgs &a = st.layout;
            a.n_tile_bits = n - S - kh;
            a.n_tiles = 1ULL << a.n_tile_bits;
            for (int j = 0; j < kh; j++) { a.hpos[j] = regs[j]; a.reg_pos[j] = v2l[regs[j]]; }
            for (int k = 0; k < 6; k++) a.lane_pos[k] = v2l[VB + k] - VB;
            for (int v = S, k = 0; v < n; v++)
                if (std::find(regs.begin(), regs.end(), v) == regs.end()) a.tile_pos[k++] = v2l[v];
            sets.push_back(std::move(st));
        }
    }
    // a lane's offset holds slot bits up to kPassMaxSlotBit
    bool fits() const {
        for (const auto &st : sets)
            for (int k = 0; k < 6; k++) if (st.layout.lane_pos[k] < 0 || st.layout.lane_pos[k] > kPassMaxSlotBit) return false;
        return n - S - kh <= kPassMaxTileBits;
    }
    void where(const HeaSet &st, int q, int32_t &w, int32_t &at) const {
        const int v = st.vpos[q];
        const int *e = st.layout.hpos + kh, *it = std::find(st.layout.hpos, e, v);
        w = it != e ? HW_SLOT : (v < VB ? HW_VEC : (v < S ? HW_LANE : HW_TILE));
        at = it != e ? (int32_t)(it - st.layout.hpos) : v;
    }
    HeaOp target(const HeaSet &st, int kind, int q) const {   // a gate whose qubit is resident
        HeaOp o{};
        o.kind = kind;
        where(st, q, o.where, o.at);
        if (o.where == HW_LANE) o.at -= VB;
        return o;
    }
    HeaOp cnot(const HeaSet &st, int c, int t) const {
        HeaOp o = target(st, HO_CNOT, t);
        where(st, c, o.cwhere, o.cat);
        return o;
    }
};
struct HeaPass {
    size_t set, op_begin, n_ops;
    std::vector<int> slots;   // partial slots of its accumulators
    int restore = -1;         // checkpoint to re-anchor psi to before the pass
    int save = -1;            // checkpoint to take after the pass
};

template <typename T, int NV>
int launch_hea(sq_engine *e, int kh, const HeaArgs &a, unsigned grid) {
    cx<T> *psi = reinterpret_cast<cx<T> *>(e->d_state), *lam = reinterpret_cast<cx<T> *>(e->d_aux);
    const size_t lds = (size_t)a.n_acc * kBlock * sizeof(double);
    switch (kh) {
    case 1: hipLaunchKernelGGL(HIP_KERNEL_NAME(k_hea<T, 1, NV>), grid, kBlock, lds, e->stream, psi, lam, a); break;
    case 2: hipLaunchKernelGGL(HIP_KERNEL_NAME(k_hea<T, 2, NV>), grid, kBlock, lds, e->stream, psi, lam, a); break;
    case 3: hipLaunchKernelGGL(HIP_KERNEL_NAME(k_hea<T, 3, NV>), grid, kBlock, lds, e->stream, psi, lam, a); break;
    case 4: hipLaunchKernelGGL(HIP_KERNEL_NAME(k_hea<T, 4, NV>), grid, kBlock, lds, e->stream, psi, lam, a); break;
    default:
        if constexpr (NV == 1) { hipLaunchKernelGGL(HIP_KERNEL_NAME(k_hea<T, 5, NV>), grid, kBlock, lds, e->stream, psi, lam, a); break; }
        return e->fail(SQ_ERR_ARG, "internal: bad pass width");
    }
    return e->check_launch("k_hea");
}

template <typename T>
int gradient(sq_engine *e, int layers, const double *theta, int ckpt_every, double *energy, double *grad) {
    constexpr int VB = Traits<T>::VB, S = VB + 6;
    const int n = e->n;
    // register bits: as many as leave about 1024 waves, two at least; both
    // vectors of the reverse sweep: four (16 x 2 vectors a lane)
    const int most = n - S;
    if (most < 1) return gradient_small<T>(e, layers, theta, ckpt_every, energy, grad);
    const HeaPlan<T> fwd(n, std::min(most, std::max(2, std::min(5, most - 10))));
    const HeaPlan<T> rev(n, std::min(most, std::max(2, std::min(4, most - 10))));
    if (!fwd.fits() || !rev.fits()) return gradient_small<T>(e, layers, theta, ckpt_every, energy, grad);
    const uint64_t na = e->n_amps();
    const int n_ckpt = (grad && ckpt_every > 0) ? std::max(0, (layers - 1) / ckpt_every) : 0;
    const size_t n_params = (size_t)2 * n * layers;
    std::vector<HeaOp> ops;
    std::vector<HeaPass> up, down;
    auto open = [&](std::vector<HeaPass> &list, size_t set) { list.push_back({set, ops.size(), 0, {}}); };
    auto close = [&](std::vector<HeaPass> &list) {
        list.back().n_ops = ops.size() - list.back().op_begin;
        if (!list.back().n_ops) list.pop_back();
    };
    for (int l = 0; l < layers; l++) {
        const double *ty = theta + (size_t)l * 2 * n, *tz = ty + n;
        for (size_t k = 0; k < fwd.sets.size(); k++) {
            const HeaSet &st = fwd.sets[k];
            open(up, k);
            for (int q : st.qubits) {
                HeaOp o = fwd.target(st, HO_RY, q);
                o.c = std::cos(ty[q] / 2);
                o.s = std::sin(ty[q] / 2);
                ops.push_back(o);
            }
            for (int q = 0; k + 1 == fwd.sets.size() && q < n; q++) {   // after every RY: diagonal, any position
                HeaOp o{};
                o.kind = HO_RZ;
                fwd.where(st, q, o.where, o.at);
                o.c = std::cos(tz[q] / 2);
                o.s = std::sin(tz[q] / 2);
                ops.push_back(o);
            }
            close(up);
        }
        for (size_t k = 0; n > 1 && k < fwd.sets.size(); k++) {
            const HeaSet &st = fwd.sets[k];
            open(up, k);
            for (int t : st.qubits) if (t > 0) ops.push_back(fwd.cnot(st, t - 1, t));
            if (k + 1 == fwd.sets.size()) ops.push_back(fwd.cnot(st, n - 1, 0));   // bit 0 is resident in every set
            close(up);
        }
        if (n_ckpt && (l + 1) % ckpt_every == 0 && l + 1 < layers) up.back().save = (l + 1) / ckpt_every - 1;
    }
    for (int l = layers - 1; grad && l >= 0; l--) {
        const double *ty = theta + (size_t)l * 2 * n, *tz = ty + n;
        const size_t first = down.size();
        for (size_t k = rev.sets.size(); n > 1 && k-- > 0;) {
            const HeaSet &st = rev.sets[k];
            open(down, k);
            if (k + 1 == rev.sets.size()) ops.push_back(rev.cnot(st, n - 1, 0));
            for (size_t i = st.qubits.size(); i-- > 0;)
                if (st.qubits[i] > 0) ops.push_back(rev.cnot(st, st.qubits[i] - 1, st.qubits[i]));
            close(down);
        }
        for (size_t k = rev.sets.size(); k-- > 0;) {
            const HeaSet &st = rev.sets[k];
            open(down, k);
            for (size_t i = st.qubits.size(); i-- > 0;) {
                const int q = st.qubits[i];
                HeaOp o = rev.target(st, HO_ROT2, q);
                o.c = std::cos(ty[q] / 2);
                o.s = std::sin(ty[q] / 2);
                o.cz = std::cos(tz[q] / 2);
                o.sz = std::sin(tz[q] / 2);
                o.acc = (int32_t)down.back().slots.size();
                down.back().slots.push_back(l * 2 * n + q);
                down.back().slots.push_back(l * 2 * n + n + q);
                ops.push_back(o);
            }
            close(down);
        }
        if (n_ckpt && (l + 1) % ckpt_every == 0 && l + 1 < layers) down[first].restore = (l + 1) / ckpt_every - 1;
    }
    // buffers: partials [slot][block], their sums, the program
    const unsigned red_grid = (unsigned)std::min<uint64_t>(kRedBlocks, std::max<uint64_t>(1, rev.sets[0].layout.n_tiles * 64 / kBlock));
    const size_t part_bytes = grad ? n_params * red_grid * sizeof(double) : 0;
    const size_t out_bytes = (n_params * sizeof(double) + 255) / 256 * 256;
    const size_t prog_at = (part_bytes + out_bytes + 255) / 256 * 256;
    int rc = ensure(e, &e->d_gradpart, &e->gradpart_cap, prog_at + ops.size() * sizeof(HeaOp) + 256, "hipMalloc(gradient partials)");
    if (!rc && grad) rc = ensure(e, &e->d_aux, &e->aux_cap, e->state_bytes(), "hipMalloc(lambda)");
    if (!rc && n_ckpt)
        rc = ensure(e, &e->d_ckpt, &e->ckpt_cap, (size_t)n_ckpt * na * sizeof(cx<double>), "hipMalloc(checkpoints)");
    if (rc) return rc;
    double *part = static_cast<double *>(e->d_gradpart);
    double *d_out = reinterpret_cast<double *>(static_cast<char *>(e->d_gradpart) + part_bytes);
    const HeaOp *d_ops = reinterpret_cast<const HeaOp *>(static_cast<char *>(e->d_gradpart) + prog_at);
    cx<double> *ckpt = n_ckpt ? static_cast<cx<double> *>(e->d_ckpt) : nullptr;
    if ((rc = e->upload(const_cast<HeaOp *>(d_ops), ops.data(), ops.size() * sizeof(HeaOp)))) return rc;
    if ((rc = sq_init_zero(e))) return rc;
    cx<T> *psi = reinterpret_cast<cx<T> *>(e->d_state), *lam = reinterpret_cast<cx<T> *>(e->d_aux);
    for (const HeaPass &p : up) {
        HeaArgs a = fwd.sets[p.set].layout;
        a.ops = d_ops + p.op_begin;
        a.n_ops = (int)p.n_ops;
        const int slot = e->stat_begin("hea_fwd", 2.0 * e->amp_bytes() * (double)na);
        rc = launch_hea<T, 1>(e, fwd.kh, a, e->grid_flat(a.n_tiles, kBlock / 64));
        e->stat_end(slot);
        if (rc) return rc;
        if (p.save >= 0) {
            hipLaunchKernelGGL(HIP_KERNEL_NAME(k_convert<T, double>), e->grid_for(na, kBlock), kBlock, 0, e->stream,
                               psi, ckpt + (size_t)p.save * na, na);
            if ((rc = e->check_launch("checkpoint"))) return rc;
        }
    }
    double v[2];
    if ((rc = e->norm_zz(v))) return rc;
    if (energy) *energy = v[1];
    if (!grad) return SQ_OK;
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_apply_zz_ring<T>), e->grid_for(na, kBlock), kBlock, 0, e->stream, psi, lam, na, n);
    if ((rc = e->check_launch("k_apply_zz_ring"))) return rc;
    for (const HeaPass &p : down) {
        if (p.restore >= 0) {
            hipLaunchKernelGGL(HIP_KERNEL_NAME(k_convert<double, T>), e->grid_for(na, kBlock), kBlock, 0, e->stream,
                               ckpt + (size_t)p.restore * na, psi, na);
            if ((rc = e->check_launch("re-anchor"))) return rc;
        }
        HeaArgs a = rev.sets[p.set].layout;
        a.ops = d_ops + p.op_begin;
        a.n_ops = (int)p.n_ops;
        a.n_acc = (int)p.slots.size();
        if (a.n_acc > kHeaMaxAcc) return e->fail(SQ_ERR_ARG, "internal: too many terms in a pass");
        std::copy(p.slots.begin(), p.slots.end(), a.slot);
        a.part = part;
        const int slot = e->stat_begin(a.n_acc ? "hea_terms" : "hea_ring2", 4.0 * e->amp_bytes() * (double)na);
        rc = launch_hea<T, 2>(e, rev.kh, a, a.n_acc ? red_grid : e->grid_flat(a.n_tiles, kBlock / 64));
        e->stat_end(slot);
        if (rc) return rc;
    }
    if (!n_params) return SQ_OK;
    hipLaunchKernelGGL(k_sum_slots, (unsigned)((n_params + kBlock / 64 - 1) / (kBlock / 64)), kBlock, 0, e->stream,
                       (const double *)part, (uint64_t)red_grid, (int)n_params, d_out);
    if ((rc = e->check_launch("k_sum_slots"))) return rc;
    hipError_t he = hipMemcpyAsync(grad, d_out, n_params * sizeof(double), hipMemcpyDeviceToHost, e->stream);
    if (he == hipSuccess) he = hipStreamSynchronize(e->stream);
    return he == hipSuccess ? SQ_OK : e->hip_fail(he, "gradient sums");
}

}  // namespace

extern "C" int sq_hea_energy(sq_engine *e, int32_t layers, const double *theta, uint64_t n_theta, double *energy) {
    if (!e || layers < 0 || (layers && !theta)) return SQ_ERR_ARG;
    if (n_theta != (uint64_t)2 * e->n * layers)
        return e->fail(SQ_ERR_ARG, "theta must hold 2 * total_qbit * layers angles");
    if (e->out_of_core()) return e->fail(SQ_ERR_UNSUPPORTED, "the ansatz needs an HBM-resident state");
    if (hipSetDevice(e->device) != hipSuccess) return SQ_ERR_HIP;
    return e->dtype == SQ_C128 ? gradient<double>(e, layers, theta, 0, energy, nullptr)
                               : gradient<float>(e, layers, theta, 0, energy, nullptr);
}

extern "C" int sq_adjoint_grad_hea(sq_engine *e, int32_t layers, const double *theta, uint64_t n_theta,
                                   int32_t checkpoint_every, double *energy, double *grad) {
    if (!e || layers < 0 || (layers && (!theta || !grad)) || checkpoint_every < 0) return SQ_ERR_ARG;
    if (n_theta != (uint64_t)2 * e->n * layers)
        return e->fail(SQ_ERR_ARG, "theta must hold 2 * total_qbit * layers angles");
    if (e->n < 2) return e->fail(SQ_ERR_ARG, "the ansatz needs at least two qubits");
    if (e->out_of_core()) return e->fail(SQ_ERR_UNSUPPORTED, "the ansatz needs an HBM-resident state");
    if (hipSetDevice(e->device) != hipSuccess) return SQ_ERR_HIP;
    return e->dtype == SQ_C128 ? gradient<double>(e, layers, theta, checkpoint_every, energy, grad)
                               : gradient<float>(e, layers, theta, checkpoint_every, energy, grad);
}

// ---------------------------------------------------------------------------
// General parameterised circuits (sq_adjoint_grad).
// ---------------------------------------------------------------------------

namespace {

int adj_kind(int gate_kind) {
    switch (gate_kind) {
    case SQ_GATE_RX: return ADJ_RX;
    case SQ_GATE_RY: return ADJ_RY;
    case SQ_GATE_RZ: return ADJ_RZ;
    case SQ_GATE_P: return ADJ_P;
    case SQ_GATE_CP: return ADJ_CP;
    case SQ_GATE_RZZ: return ADJ_RZZ;
    default: return -1;
    }
}

// G^dag of a fixed gate as a gate line (rotations and phases with the angle
// negated, dense matrices conjugate-transposed, X Y Z SWAP themselves).
int adjoint_gate(const sq_gate &g, sq_gate &out) {
    out = g;
    switch (g.kind) {
    case SQ_GATE_X: case SQ_GATE_Y: case SQ_GATE_Z: case SQ_GATE_SWAP:
        return SQ_OK;
    case SQ_GATE_P: case SQ_GATE_RX: case SQ_GATE_RY: case SQ_GATE_RZ: case SQ_GATE_CP: case SQ_GATE_RZZ:
        out.param = -g.param;
        return SQ_OK;
    case SQ_GATE_H: {
        // the reference's H (circuit.cpp:247) as a dense matrix; it is real
        // and symmetric, so it is its own conjugate transpose
        const double c = 0.70710678118;
        out.kind = SQ_GATE_U1;
        const double m[8] = {c, 0, c, 0, c, 0, -c, 0};
        std::copy(m, m + 8, out.mat);
        return SQ_OK;
    }
    case SQ_GATE_U1:
    case SQ_GATE_U2: {
        const int d = g.kind == SQ_GATE_U1 ? 2 : 4;
        for (int r = 0; r < d; r++)
            for (int c = 0; c < d; c++) {
                out.mat[2 * (r * d + c)] = g.mat[2 * (c * d + r)];
                out.mat[2 * (r * d + c) + 1] = -g.mat[2 * (c * d + r) + 1];
            }
        return SQ_OK;
    }
    default:
        return SQ_ERR_UNSUPPORTED;
    }
}

// Applies a list of gates on the engine's state as register passes (the
// plain sweep), on psi (lambda_buffer = false) or on lambda.
int sweep_on(sq_engine *e, const std::vector<sq_gate> &gl, bool on_lambda) {
    if (gl.empty()) return SQ_OK;
    if (int rc = e->lower_list(gl.data(), gl.size())) return rc;
    if (on_lambda) std::swap(e->d_state, e->d_aux);
    const int rc = e->apply_plain(gl.data(), gl.size(), e->ws_low);
    if (on_lambda) std::swap(e->d_state, e->d_aux);
    return rc;
}

// The same list on psi and lambda at once: each register pass is one launch
// over both vectors (twice the waves, so small states fill the GPU better).
int sweep_both(sq_engine *e, const std::vector<sq_gate> &gl) {
    if (gl.empty()) return SQ_OK;
    if (int rc = e->lower_list(gl.data(), gl.size())) return rc;
    e->d_state2 = e->d_aux;
    const int rc = e->apply_plain(gl.data(), gl.size(), e->ws_low);
    e->d_state2 = nullptr;
    return rc;
}

// Register bits of a wave tile in the transform kernels: few enough that the
// tiles fill the GPU (1024 waves at 16 qubits and more), at most 2^4 rows.
int tile_rows_log2(int n) { return std::max(0, std::min(4, n - 16)); }

template <typename T> struct TransformLaunch {
    template <int KR> static void terms(sq_engine *e, unsigned grid, const cx<T> *psi, const cx<T> *lam, const DiagTermArgs &a, double *part) {
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_adj_diag_terms<T, KR>), grid, kBlock, 0, e->stream, psi, lam, a, part, (uint64_t)grid);
    }
    template <int KR> static void zterms(sq_engine *e, unsigned grid, const cx<T> *psi, cx<T> *lam, const ZTermArgs &a, double *part) {
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_apply_zterms<T, KR>), grid, kBlock, 0, e->stream, psi, lam, a, part);
    }
};

bool diagonal_kind(int kind) {
    return kind == SQ_GATE_Z || kind == SQ_GATE_P || kind == SQ_GATE_RZ || kind == SQ_GATE_CP || kind == SQ_GATE_RZZ;
}

// One step of the reverse sweep.
struct AdjStep {
    enum Kind { Inverse, Multi, Gate, Terms, Restore } kind;
    std::vector<sq_gate> gates;              // Inverse: applied to psi and lambda
    std::vector<uint64_t> group;             // Multi: its gates, in the sweep's order; Gate: one
    size_t slot = 0;                         // first partial slot
    std::vector<uint64_t> masks;             // Terms
    size_t blob_tile = 0, blob_low = 0;      // Terms: byte offsets of the mask arrays
    size_t segment = 0;                      // Restore
};

template <typename T>
int adjoint_general(sq_engine *e, const sq_gate *gates, const int32_t *param, uint64_t ng, const double *theta,
                    uint64_t n_theta, const sq_zterm *terms, uint64_t n_terms, int ckpt_every, double *energy,
                    double *grad) {
    const uint64_t na = e->n_amps();
    const int n = e->n, kr = tile_rows_log2(n), low_bits = 6 + kr;
    const bool tiles = n >= 6;   // the transform kernels work on whole waves
    // complex64: each gate is un-applied and its term taken where the list has
    // it, so that the FP32 rounding, and with it the gradient to all digits,
    // stays what it is (see keep_order)
    // Without register passes too (complex128: under 11 qubits): a run's gates would
    // be one launch each to un-apply, after the launch that takes the terms (MaxCut
    // gradient, 9 qubits, five layers: 2.54 ms as runs, 2.09 ms gate by gate).
    const bool runs = tiles && sizeof(T) == 8 && e->sweep_mode == 0 && n >= Traits<T>::VB + 6 + e->pass_qbits;
    struct KeepOrder {
        sq_engine *e;
        KeepOrder(sq_engine *x, bool on) : e(x) { e->keep_order = on; }
        ~KeepOrder() { e->keep_order = false; }
    } keep(e, sizeof(T) == 4);
    // the circuit with its angles, and the parameterised gates
    std::vector<sq_gate> circ(gates, gates + ng);
    std::vector<uint64_t> pgates;   // indices of parameterised gates, in order
    for (uint64_t i = 0; i < ng; i++) {
        if (param[i] < 0) continue;
        if ((uint64_t)param[i] >= n_theta) return e->fail(SQ_ERR_ARG, "parameter index beyond theta (gate " + std::to_string(i) + ")");
        if (adj_kind(circ[i].kind) < 0)
            return e->fail(SQ_ERR_ARG, "only RX RY RZ P CP RZZ take a parameter (gate " + std::to_string(i) + ")");
        circ[i].param = theta[param[i]];
        pgates.push_back(i);
    }
    for (uint64_t i = 0; i < ng; i++) {
        LoweredGate lg;
        int rc = e->lower(circ[i], lg);
        if (rc) { e->err += " (gate " + std::to_string(i) + ")"; return rc; }
        sq_gate inv;
        if (param[i] < 0 && adjoint_gate(circ[i], inv) != SQ_OK)
            return e->fail(SQ_ERR_UNSUPPORTED, "no adjoint for gate " + std::to_string(i));
    }
    // segments between FP64 checkpoints: every ckpt_every parameterised gates
    std::vector<uint64_t> seg_end;   // gate index where each segment ends (exclusive)
    if (grad && ckpt_every > 0)
        for (size_t k = ckpt_every; k < pgates.size(); k += ckpt_every) seg_end.push_back(pgates[k]);
    seg_end.push_back(ng);
    const size_t n_ckpt = grad && ckpt_every > 0 ? seg_end.size() : 0;   // states at the segment starts

    // The reverse sweep's steps.  Parameterised gates give gradient terms as
    // weighted sums of partial slots (slot 0: the energy):
    struct Term {
        int32_t param;
        size_t slot;
        double weight;
    };
    std::vector<Term> sums;
    std::vector<AdjStep> steps;
    size_t n_slots = 1;
    if (grad) {
        std::vector<sq_gate> inv_run;       // gates to un-apply before the next term is taken
        std::vector<uint64_t> group, run;   // pending one-qubit gates of one launch; pending diagonal gates (reverse order)
        auto flush = [&]() {
            if (inv_run.empty()) return;
            AdjStep st{AdjStep::Inverse};
            st.gates.swap(inv_run);
            steps.push_back(std::move(st));
        };
        auto launch_group = [&]() {
            if (group.empty()) return;
            flush();
            AdjStep st{AdjStep::Multi};
            st.slot = n_slots;
            // local bit b: the gate of slot + b, first the earliest in the circuit
            std::reverse(group.begin(), group.end());
            for (size_t b = 0; b < group.size(); b++) sums.push_back({param[group[b]], n_slots + b, 1.0});
            n_slots += group.size();
            st.group.swap(group);
            steps.push_back(std::move(st));
        };
        auto single = [&](uint64_t gi) {   // two-qubit gate, one launch
            flush();
            AdjStep st{AdjStep::Gate};
            st.slot = n_slots++;
            st.group = {gi};
            sums.push_back({param[gi], st.slot, 1.0});
            steps.push_back(std::move(st));
        };
        // Consecutive one-qubit parameterised gates on distinct qubits go to one
        // k_adj_multi launch: four for complex64 (171 VGPRs), three for complex128
        const size_t group_max = sizeof(T) == 4 ? 4 : 3;
        auto add_single_qubit = [&](uint64_t gi) {
            bool clash = group.size() == group_max;
            for (uint64_t m : group) clash = clash || circ[m].q[0] == circ[gi].q[0];
            if (clash) launch_group();
            group.push_back(gi);
        };
        // A run of diagonal gates: all of its terms by one read of psi and lambda,
        // then its gates join the next un-applies.  Runs that k_adj_multi takes in
        // one launch (one read and write) stay there.
        auto close_run = [&]() {
            if (run.empty()) return;
            std::vector<uint64_t> r;
            r.swap(run);
            size_t n_param = 0;
            bool one_qubit = true;
            for (uint64_t gi : r) {
                n_param += param[gi] >= 0;
                one_qubit = one_qubit && circ[gi].nq == 1 && param[gi] >= 0;
            }
            if (n_param == 0) {
                launch_group();
                for (uint64_t gi : r) {
                    sq_gate inv;
                    adjoint_gate(circ[gi], inv);
                    inv_run.push_back(inv);
                }
                return;
            }
            if (!runs || (one_qubit && r.size() <= group_max)) {
                for (uint64_t gi : r) {
                    if (param[gi] < 0) {
                        launch_group();
                        sq_gate inv;
                        adjoint_gate(circ[gi], inv);
                        inv_run.push_back(inv);
                    } else if (circ[gi].nq == 1) {
                        add_single_qubit(gi);
                    } else {
                        launch_group();
                        single(gi);
                    }
                }
                return;
            }
            launch_group();
            flush();
            std::vector<uint64_t> masks;
            std::vector<std::vector<std::pair<int32_t, double>>> weights;   // per mask: (parameter, weight)
            std::unordered_map<uint64_t, size_t> at;
            auto use = [&](uint64_t mask, int32_t p, double w) {
                auto it = at.emplace(mask, masks.size());
                if (it.second) { masks.push_back(mask); weights.emplace_back(); }
                weights[it.first->second].push_back({p, w});
            };
            for (uint64_t gi : r) {
                const sq_gate &g = circ[gi];
                const uint64_t a = 1ULL << g.q[0], b = g.nq > 1 ? 1ULL << g.q[1] : 0;
                if (param[gi] >= 0) switch (g.kind) {
                case SQ_GATE_RZ: use(a, param[gi], 1.0); break;
                case SQ_GATE_RZZ: use(a | b, param[gi], 1.0); break;
                // -2 Im <lambda|Pi|psi>, Pi = (1 - Z)/2 and (1 - Za)(1 - Zb)/4
                case SQ_GATE_P: use(0, param[gi], -1.0); use(a, param[gi], 1.0); break;
                default:
                    use(0, param[gi], -0.5);
                    use(a, param[gi], 0.5);
                    use(b, param[gi], 0.5);
                    use(a | b, param[gi], -0.5);
                    break;
                }
                sq_gate inv;
                adjoint_gate(g, inv);
                inv_run.push_back(inv);
            }
            std::vector<sq_gate> after;
            after.swap(inv_run);   // the launches come first
            for (size_t m0 = 0; m0 < masks.size(); m0 += kDiagTermMax) {
                AdjStep st{AdjStep::Terms};
                const size_t m1 = std::min(masks.size(), m0 + kDiagTermMax);
                st.masks.assign(masks.begin() + m0, masks.begin() + m1);
                st.slot = n_slots;
                for (size_t m = m0; m < m1; m++)
                    for (auto &w : weights[m]) sums.push_back({w.first, n_slots + (m - m0), w.second});
                n_slots += m1 - m0;
                steps.push_back(std::move(st));
            }
            inv_run.swap(after);
        };
        size_t seg = seg_end.size();   // segments left to sweep back
        for (uint64_t gi = ng; gi-- > 0;) {
            // entering the previous segment: psi is re-anchored to the FP64 copy
            // taken at this segment's end (the next one's start)
            while (seg > 1 && gi < seg_end[seg - 2]) {
                close_run();
                launch_group();
                flush();
                AdjStep st{AdjStep::Restore};
                st.segment = seg - 1;
                steps.push_back(std::move(st));
                seg--;
            }
            if (diagonal_kind(circ[gi].kind)) {
                run.push_back(gi);
                continue;
            }
            close_run();
            if (param[gi] < 0) {
                launch_group();
                sq_gate inv;
                adjoint_gate(circ[gi], inv);
                inv_run.push_back(inv);
                continue;
            }
            add_single_qubit(gi);
        }
        close_run();
        launch_group();
        flush();
    }

    // device buffers: partials, their sums, and the strings' and masks' arrays
    const unsigned grid = (unsigned)std::min<uint64_t>(kRedBlocks, std::max<uint64_t>(1, (na / 2 + kBlock - 1) / kBlock));
    std::vector<unsigned char> blob;
    auto put = [&](const void *p, size_t bytes) {
        const size_t at = (blob.size() + 7) / 8 * 8;
        blob.resize(at + bytes);
        if (bytes) std::memcpy(blob.data() + at, p, bytes);
        return at;
    };
    const uint64_t low_mask = (1ULL << low_bits) - 1;
    size_t z_low = 0, z_begin = 0, z_coef = 0, z_tile = 0, z_terms = 0;
    int n_low = 0;
    if (tiles) {
        std::vector<uint32_t> order(n_terms), low, begin;
        for (uint64_t t = 0; t < n_terms; t++) order[t] = (uint32_t)t;
        std::stable_sort(order.begin(), order.end(), [&](uint32_t x, uint32_t y) {
            return (terms[x].mask & low_mask) < (terms[y].mask & low_mask);
        });
        std::vector<double> coef;
        std::vector<uint64_t> tile;
        for (uint32_t t : order) {
            const uint32_t l = (uint32_t)(terms[t].mask & low_mask);
            if (low.empty() || low.back() != l) { low.push_back(l); begin.push_back((uint32_t)coef.size()); }
            coef.push_back(terms[t].coef);
            tile.push_back(terms[t].mask >> low_bits);
        }
        begin.push_back((uint32_t)coef.size());
        n_low = (int)low.size();
        z_low = put(low.data(), low.size() * sizeof(uint32_t));
        z_begin = put(begin.data(), begin.size() * sizeof(uint32_t));
        z_coef = put(coef.data(), coef.size() * sizeof(double));
        z_tile = put(tile.data(), tile.size() * sizeof(uint64_t));
    } else {
        std::vector<ZTerm> ht(n_terms);
        for (uint64_t t = 0; t < n_terms; t++) ht[t] = {terms[t].coef, terms[t].mask};
        z_terms = put(ht.data(), n_terms * sizeof(ZTerm));
    }
    for (auto &st : steps) {
        if (st.kind != AdjStep::Terms) continue;
        std::vector<uint64_t> tile;
        std::vector<uint32_t> low;
        for (uint64_t m : st.masks) {
            tile.push_back(m >> low_bits);
            low.push_back((uint32_t)(m & low_mask));
        }
        st.blob_tile = put(tile.data(), tile.size() * sizeof(uint64_t));
        st.blob_low = put(low.data(), low.size() * sizeof(uint32_t));
    }
    const size_t part_bytes = n_slots * grid * sizeof(double), out_bytes = (n_slots * sizeof(double) + 255) / 256 * 256;
    int rc = grad ? ensure(e, &e->d_aux, &e->aux_cap, e->state_bytes(), "hipMalloc(lambda)") : SQ_OK;
    if (!rc && n_ckpt)
        rc = ensure(e, &e->d_ckpt, &e->ckpt_cap, n_ckpt * na * sizeof(cx<double>), "hipMalloc(checkpoints)");
    if (!rc) rc = ensure(e, &e->d_gradpart, &e->gradpart_cap, part_bytes + out_bytes + blob.size() + 256,
                         "hipMalloc(gradient partials)");
    if (rc) return rc;
    double *part = static_cast<double *>(e->d_gradpart);
    double *d_out = reinterpret_cast<double *>(static_cast<char *>(e->d_gradpart) + part_bytes);
    char *d_blob = static_cast<char *>(e->d_gradpart) + part_bytes + out_bytes;
    if ((rc = e->upload(d_blob, blob.data(), blob.size()))) return rc;
    cx<double> *ckpt = n_ckpt ? static_cast<cx<double> *>(e->d_ckpt) : nullptr;
    auto save = [&](size_t slot) {
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_convert<T, double>), e->grid_for(na, kBlock), kBlock, 0, e->stream,
                           reinterpret_cast<const cx<T> *>(e->d_state), ckpt + slot * na, na);
        return e->check_launch("checkpoint");
    };
    auto restore = [&](size_t slot) {
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_convert<double, T>), e->grid_for(na, kBlock), kBlock, 0, e->stream,
                           ckpt + slot * na, reinterpret_cast<cx<T> *>(e->d_state), na);
        return e->check_launch("re-anchor");
    };
    // forward: segment by segment as register passes, an FP64 copy of the
    // state at each segment's start
    uint64_t begin = 0;
    for (size_t sgi = 0; sgi < seg_end.size(); sgi++) {
        if (ckpt && (rc = save(sgi))) return rc;
        if ((rc = sweep_on(e, std::vector<sq_gate>(circ.begin() + begin, circ.begin() + seg_end[sgi]), false))) return rc;
        begin = seg_end[sgi];
    }
    {
        const cx<T> *psi = reinterpret_cast<const cx<T> *>(e->d_state);
        cx<T> *lam = grad ? reinterpret_cast<cx<T> *>(e->d_aux) : nullptr;
        if (tiles) {
            const ZTermArgs a{1ULL << (n - low_bits), n_low, reinterpret_cast<const uint32_t *>(d_blob + z_low),
                              reinterpret_cast<const uint32_t *>(d_blob + z_begin),
                              reinterpret_cast<const double *>(d_blob + z_coef),
                              reinterpret_cast<const uint64_t *>(d_blob + z_tile)};
            switch (kr) {
            case 0: TransformLaunch<T>::template zterms<0>(e, grid, psi, lam, a, part); break;
            case 1: TransformLaunch<T>::template zterms<1>(e, grid, psi, lam, a, part); break;
            case 2: TransformLaunch<T>::template zterms<2>(e, grid, psi, lam, a, part); break;
            case 3: TransformLaunch<T>::template zterms<3>(e, grid, psi, lam, a, part); break;
            default: TransformLaunch<T>::template zterms<4>(e, grid, psi, lam, a, part); break;
            }
        } else {
            hipLaunchKernelGGL(HIP_KERNEL_NAME(k_apply_zterms_small<T>), grid, kBlock, 0, e->stream, psi, lam,
                               reinterpret_cast<const ZTerm *>(d_blob + z_terms), (int)n_terms, na, part);
        }
        if ((rc = e->check_launch("k_apply_zterms"))) return rc;
    }
    // reverse sweep
    for (const auto &st : steps) {
        cx<T> *psi = reinterpret_cast<cx<T> *>(e->d_state);
        cx<T> *lam = reinterpret_cast<cx<T> *>(e->d_aux);
        double *dst = part + st.slot * grid;
        switch (st.kind) {
        case AdjStep::Inverse:
            if ((rc = sweep_both(e, st.gates))) return rc;
            break;
        case AdjStep::Restore:
            if ((rc = restore(st.segment))) return rc;
            break;
        case AdjStep::Multi: {
            const int M = (int)st.group.size();
            AdjMultiArgs a{};
            a.n_items = na >> M;
            for (int b = 0; b < M; b++) {
                const sq_gate &g = circ[st.group[b]];
                a.kind[b] = adj_kind(g.kind);
                a.q[b] = g.q[0];
                const double ang = a.kind[b] == ADJ_P ? g.param : g.param / 2;
                a.c[b] = std::cos(ang);
                a.s[b] = std::sin(ang);
            }
            std::copy(a.q, a.q + M, a.qs);
            std::sort(a.qs, a.qs + M);
            const int slot = e->stat_begin("adj_multi", 4.0 * e->amp_bytes() * (double)na);
            switch (M) {
            case 1: hipLaunchKernelGGL(HIP_KERNEL_NAME(k_adj_multi<T, 1>), grid, kBlock, 0, e->stream, psi, lam, a, dst, (uint64_t)grid); break;
            case 2: hipLaunchKernelGGL(HIP_KERNEL_NAME(k_adj_multi<T, 2>), grid, kBlock, 0, e->stream, psi, lam, a, dst, (uint64_t)grid); break;
            case 3: hipLaunchKernelGGL(HIP_KERNEL_NAME(k_adj_multi<T, 3>), grid, kBlock, 0, e->stream, psi, lam, a, dst, (uint64_t)grid); break;
            default: hipLaunchKernelGGL(HIP_KERNEL_NAME(k_adj_multi<T, 4>), grid, kBlock, 0, e->stream, psi, lam, a, dst, (uint64_t)grid); break;
            }
            e->stat_end(slot);
            if ((rc = e->check_launch("k_adj_multi"))) return rc;
            break; }
        case AdjStep::Gate: {
            const sq_gate &g = circ[st.group[0]];
            AdjGateArgs a{};
            a.kind = adj_kind(g.kind);
            a.n_items = na;
            a.q0 = g.q[0];
            a.q1 = g.q[1];
            const double ang = a.kind == ADJ_CP ? g.param : g.param / 2;
            a.c = std::cos(ang);
            a.s = std::sin(ang);
            // every block writes its partial (zero when it has no items)
            const int slot = e->stat_begin("adj_gate", 4.0 * e->amp_bytes() * (double)na);
            hipLaunchKernelGGL(HIP_KERNEL_NAME(k_adj_gate<T>), grid, kBlock, 0, e->stream, psi, lam, a, dst);
            e->stat_end(slot);
            if ((rc = e->check_launch("k_adj_gate"))) return rc;
            break; }
        case AdjStep::Terms: {
            const DiagTermArgs a{1ULL << (n - low_bits), reinterpret_cast<const uint64_t *>(d_blob + st.blob_tile),
                                 reinterpret_cast<const uint32_t *>(d_blob + st.blob_low), (int)st.masks.size()};
            const int slot = e->stat_begin("adj_diag_terms", 2.0 * e->amp_bytes() * (double)na);
            switch (kr) {
            case 0: TransformLaunch<T>::template terms<0>(e, grid, psi, lam, a, dst); break;
            case 1: TransformLaunch<T>::template terms<1>(e, grid, psi, lam, a, dst); break;
            case 2: TransformLaunch<T>::template terms<2>(e, grid, psi, lam, a, dst); break;
            case 3: TransformLaunch<T>::template terms<3>(e, grid, psi, lam, a, dst); break;
            default: TransformLaunch<T>::template terms<4>(e, grid, psi, lam, a, dst); break;
            }
            e->stat_end(slot);
            if ((rc = e->check_launch("k_adj_diag_terms"))) return rc;
            break; }
        }
    }
    if (ckpt && (rc = restore(0))) return rc;   // the state the call started from, exactly
    hipLaunchKernelGGL(k_sum_slots, (unsigned)((n_slots + kBlock / 64 - 1) / (kBlock / 64)), kBlock, 0, e->stream,
                       (const double *)part, (uint64_t)grid, (int)n_slots, d_out);
    if ((rc = e->check_launch("k_sum_slots"))) return rc;
    std::vector<double> h(n_slots);
    hipError_t he = hipMemcpyAsync(h.data(), d_out, n_slots * sizeof(double), hipMemcpyDeviceToHost, e->stream);
    if (he == hipSuccess) he = hipStreamSynchronize(e->stream);
    if (he != hipSuccess) return e->hip_fail(he, "gradient sums");
    if (energy) *energy = h[0];
    if (!grad) return SQ_OK;
    std::fill(grad, grad + n_theta, 0.0);
    for (const Term &t : sums) grad[t.param] += t.weight * h[t.slot];
    return SQ_OK;
}

}  // namespace

extern "C" int sq_expect_z(sq_engine *e, const sq_zterm *terms, uint64_t n_terms, double *out) {
    if (!e || (!terms && n_terms) || !out) return SQ_ERR_ARG;
    if (e->out_of_core()) return e->fail(SQ_ERR_UNSUPPORTED, "the observable needs an HBM-resident state");
    if (hipSetDevice(e->device) != hipSuccess) return SQ_ERR_HIP;
    return e->dtype == SQ_C128 ? adjoint_general<double>(e, nullptr, nullptr, 0, nullptr, 0, terms, n_terms, 0, out, nullptr)
                               : adjoint_general<float>(e, nullptr, nullptr, 0, nullptr, 0, terms, n_terms, 0, out, nullptr);
}

extern "C" int sq_adjoint_grad(sq_engine *e, const sq_gate *gates, const int32_t *param, uint64_t n_gates,
                               const double *theta, uint64_t n_theta, const sq_zterm *terms, uint64_t n_terms,
                               int32_t checkpoint_every, double *energy, double *grad) {
    if (!e || (!gates && n_gates) || (!param && n_gates) || (!theta && n_theta) || (!terms && n_terms) ||
        checkpoint_every < 0 || (!grad && n_theta))
        return SQ_ERR_ARG;
    if (e->out_of_core()) return e->fail(SQ_ERR_UNSUPPORTED, "the adjoint gradient needs an HBM-resident state");
    if (hipSetDevice(e->device) != hipSuccess) return SQ_ERR_HIP;
    double dummy = 0;
    double *g = grad ? grad : &dummy;
    return e->dtype == SQ_C128
               ? adjoint_general<double>(e, gates, param, n_gates, theta, n_theta, terms, n_terms, checkpoint_every, energy, g)
               : adjoint_general<float>(e, gates, param, n_gates, theta, n_theta, terms, n_terms, checkpoint_every, energy, g);
}
