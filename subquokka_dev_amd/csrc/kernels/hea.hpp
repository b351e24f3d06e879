// hea.hpp -- passes of the hardware-efficient ansatz (RY on every qubit, RZ on
// every qubit, CNOT ring) over a wave's registers.
//
// One launch per gate (k_dense, k_diag, k_cnot2) and one per qubit in the
// reverse sweep (k_adj_rot2) each read and write the whole state.  A pass here
// holds 2^KH x 64 16-byte vectors of psi (and, in the reverse sweep, of
// lambda) as the register passes do (pass.hpp: the same virtual positions,
// with three movable lane positions) and runs every gate of the layer whose
// target is resident.  The gates keep the order of the list and the
// arithmetic of those kernels, operation by operation: only the sums over
// amplitudes (FP64) are added in another order, so complex64 results keep all
// their digits.
// What bounds it (24 qubits, complex64: the state is cache-resident): the
// passes without terms run at the cache's rate, the ones with terms at FP64
// issue (the terms' products).
#pragma once
#include "common.hpp"
#include "pass.hpp"

namespace sqk {

enum HeaOpKind : int32_t {
    HO_RY = 0,     // x0' = c x0 - s x1, x1' = s x0 + c x1
    HO_RZ = 1,     // times (c, -s) where the bit is 0, (c, s) where it is 1; any position
    HO_CNOT = 2,   // exchange along the target where the control is 1
    HO_ROT2 = 3,   // reverse sweep: the qubit's RZ and RY terms, both un-applied
};
enum HeaWhere : int32_t { HW_SLOT = 0, HW_LANE = 1, HW_VEC = 2, HW_TILE = 3 };

// 64 bytes, read with one batch of scalar loads (32-bit and 64-bit fields at
// their own alignment).
struct alignas(64) HeaOp {
    int32_t kind;
    int32_t where, at;      // target: register slot, lane bit, vector bit or tile position
    int32_t cwhere, cat;    // HO_CNOT's control
    int32_t acc;            // HO_ROT2: accumulator of the RY term (the RZ term's is the next)
    int32_t pad[2];
    double c, s;            // RY / RZ: cos, sin of the half angle; ROT2: RY's
    double cz, sz;          // ROT2: RZ's
};
static_assert(sizeof(HeaOp) == 64, "one scalar fetch per op");
struct HeaRec {
    pass_v16i w;
    __device__ explicit HeaRec(const HeaOp *p) {
        typedef SQK_AS_CONST const pass_v16i cpv;
        w = *(cpv *)p;
    }
    __device__ int i(int k) const { return w[k]; }
    __device__ double d(int k) const {
        const int b = 8 + 2 * k;
        return __builtin_bit_cast(double, (uint64_t)(uint32_t)w[b] | ((uint64_t)(uint32_t)w[b + 1] << 32));
    }
};

constexpr int kHeaMaxAcc = 24;   // two terms per resident qubit: 2 (VB + 6 + 4) at most
struct HeaArgs {
    const HeaOp *ops;
    uint64_t n_tiles;
    int n_ops;
    int n_tile_bits;
    int hpos[kPassMaxKH];
    int lane_pos[6];
    int reg_pos[kPassMaxKH];
    int tile_pos[kPassMaxTileBits];
    int n_acc;
    int slot[kHeaMaxAcc];    // partial slot of each accumulator
    double *part;            // [slot][block]
};

// a' = c a + t b with one product rounded first, as k_dense's two steps do
template <typename T> __device__ inline cx<T> hea_first(T m, cx<T> a) { return {m * a.re, m * a.im}; }
template <typename T> __device__ inline cx<T> hea_then(cx<T> acc, T m, cx<T> a) {
    return {fmaT(m, a.re, acc.re), fmaT(m, a.im, acc.im)};
}
template <typename T> __device__ inline void hea_ry(cx<T> &x0, cx<T> &x1, T c, T s) {
    const cx<T> a = hea_then(hea_first(c, x0), -s, x1), b = hea_then(hea_first(s, x0), c, x1);
    x0 = a;
    x1 = b;
}

// Phase products with k_diag's and k_adj_rot2's roundings (which product of a
// sum is rounded before the FMA), written out so that they do not depend on
// how a compiler contracts them here.
template <typename T> __device__ inline cx<T> hea_phase(cx<T> x, T c, T s) {   // k_diag: x (c, s)
    return {fmaT(x.re, c, -(x.im * s)), fmaT(x.im, c, x.re * s)};
}
template <typename T> __device__ inline cx<T> hea_unphase0(cx<T> x, T c, T s) {   // x (c, s)
    return {fmaT(x.re, c, -(x.im * s)), fmaT(x.re, s, x.im * c)};
}
template <typename T> __device__ inline cx<T> hea_unphase1(cx<T> x, T c, T s) {   // x (c, -s)
    return {fmaT(x.re, c, x.im * s), fmaT(x.im, c, -(x.re * s))};
}

// k_adj_rot2's arithmetic on one pair of psi and lambda.
template <typename T>
__device__ inline void hea_rot2(cx<T> &x0, cx<T> &x1, cx<T> &l0, cx<T> &l1, T cz, T sz, T cy, T sy, double &ry, double &rz) {
    {
        const double x0r = x0.re, x0i = x0.im, x1r = x1.re, x1i = x1.im;
        const double l0r = l0.re, l0i = l0.im, l1r = l1.re, l1i = l1.im;
        rz += (l0r * x0i - l0i * x0r) - (l1r * x1i - l1i * x1r);
        x0 = hea_unphase0(x0, cz, sz);
        x1 = hea_unphase1(x1, cz, sz);
        l0 = hea_unphase0(l0, cz, sz);
        l1 = hea_unphase1(l1, cz, sz);
    }
    {
        const double x0r = x0.re, x0i = x0.im, x1r = x1.re, x1i = x1.im;
        const double l0r = l0.re, l0i = l0.im, l1r = l1.re, l1i = l1.im;
        ry += (l1r * x0r + l1i * x0i) - (l0r * x1r + l0i * x1i);
        const cx<T> a = {fmaT(cy, x0.re, sy * x1.re), fmaT(cy, x0.im, sy * x1.im)};
        const cx<T> b = {fmaT(cy, x1.re, -(sy * x0.re)), fmaT(cy, x1.im, -(sy * x0.im))};
        x0 = a;
        x1 = b;
        const cx<T> d = {fmaT(cy, l0.re, sy * l1.re), fmaT(cy, l0.im, sy * l1.im)};
        const cx<T> e = {fmaT(cy, l1.re, -(sy * l0.re)), fmaT(cy, l1.im, -(sy * l0.im))};
        l0 = d;
        l1 = e;
    }
}

template <typename T, int MASK> __device__ inline cx<T> hea_partner(cx<T> x, int lane) {
    return {lane_partner<MASK>(x.re, lane), lane_partner<MASK>(x.im, lane)};
}

// One op on a register slot J of NV vectors.
template <typename T, int J, int NV, int R, int E>
__device__ inline void hea_slot(Pack<T> (&v)[NV][R], const HeaRec &rec, int kind, const bool (&on)[E], int cslot, double &ry,
                                double &rz) {
    if (kind == HO_RY) {
        const T c = (T)rec.d(0), s = (T)rec.d(1);
#pragma unroll
        for (int r = 0; r < R; r++)
            if (!((r >> J) & 1))
#pragma unroll
                for (int e = 0; e < E; e++) hea_ry(v[0][r].e[e], v[0][r | (1 << J)].e[e], c, s);
    } else if (kind == HO_ROT2) {
        if constexpr (NV == 2) {
            const T cz = (T)rec.d(2), sz = (T)rec.d(3), cy = (T)rec.d(0), sy = (T)rec.d(1);
#pragma unroll
            for (int r = 0; r < R; r++)
                if (!((r >> J) & 1))
#pragma unroll
                    for (int e = 0; e < E; e++)
                        hea_rot2(v[0][r].e[e], v[0][r | (1 << J)].e[e], v[1][r].e[e], v[1][r | (1 << J)].e[e], cz, sz, cy, sy, ry, rz);
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; r++) {
            if ((r >> J) & 1) continue;
            if (cslot >= 0 && !((r >> cslot) & 1)) continue;   // wave-uniform
#pragma unroll
            for (int k = 0; k < NV; k++)
#pragma unroll
                for (int e = 0; e < E; e++) {
                    const cx<T> p = v[k][r].e[e], o = v[k][r | (1 << J)].e[e];
                    v[k][r].e[e] = csel(on[e], o, p);
                    v[k][r | (1 << J)].e[e] = csel(on[e], p, o);
                }
        }
    }
}

// One op on lane bit MASK: every lane computes its own side of the pair.
template <typename T, int MASK, int NV, int R, int E>
__device__ inline void hea_lane(Pack<T> (&v)[NV][R], const HeaRec &rec, int kind, int lane, const bool (&on)[E], int cslot,
                                double &ry, double &rz) {
    const bool hi = (lane & MASK) != 0;
    if (kind == HO_RY) {
        // row of this lane: (c, -s) or (s, c)
        const T c = (T)rec.d(0), s = (T)rec.d(1), m0 = hi ? s : c, m1 = hi ? c : -s;
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int e = 0; e < E; e++) {
                const cx<T> x = v[0][r].e[e], p = hea_partner<T, MASK>(x, lane);
                v[0][r].e[e] = hea_then(hea_first(m0, csel(hi, p, x)), m1, csel(hi, x, p));
            }
    } else if (kind == HO_ROT2) {
        if constexpr (NV == 2) {
            const T cz = (T)rec.d(2), sz = (T)rec.d(3), cy = (T)rec.d(0), sy = (T)rec.d(1);
            const T t = hi ? -sy : sy;   // cy x0 + sy x1, cy x1 - sy x0: own value first
            double az = 0.0, ay = 0.0;
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int e = 0; e < E; e++) {
                    cx<T> x = v[0][r].e[e], l = v[1][r].e[e];
                    az += (double)l.re * (double)x.im - (double)l.im * (double)x.re;
                    x = csel(hi, hea_unphase1(x, cz, sz), hea_unphase0(x, cz, sz));
                    l = csel(hi, hea_unphase1(l, cz, sz), hea_unphase0(l, cz, sz));
                    const cx<T> xp = hea_partner<T, MASK>(x, lane), lp = hea_partner<T, MASK>(l, lane);
                    ay += (double)l.re * (double)xp.re + (double)l.im * (double)xp.im;
                    v[0][r].e[e] = {fmaT(cy, x.re, t * xp.re), fmaT(cy, x.im, t * xp.im)};
                    v[1][r].e[e] = {fmaT(cy, l.re, t * lp.re), fmaT(cy, l.im, t * lp.im)};
                }
            rz += hi ? -az : az;
            ry += hi ? ay : -ay;
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (cslot >= 0 && !((r >> cslot) & 1)) continue;
#pragma unroll
            for (int k = 0; k < NV; k++)
#pragma unroll
                for (int e = 0; e < E; e++) {
                    const cx<T> x = v[k][r].e[e], p = hea_partner<T, MASK>(x, lane);
                    v[k][r].e[e] = csel(on[e], p, x);
                }
        }
    }
}

// One op inside the complex64 vector.
template <typename T, int NV, int R>
__device__ inline void hea_vec(Pack<T> (&v)[NV][R], const HeaRec &rec, int kind, bool on, int cslot, double &ry, double &rz) {
    if (kind == HO_RY) {
#pragma unroll
        for (int r = 0; r < R; r++) hea_ry(v[0][r].e[0], v[0][r].e[1], (T)rec.d(0), (T)rec.d(1));
    } else if (kind == HO_ROT2) {
        if constexpr (NV == 2)
#pragma unroll
            for (int r = 0; r < R; r++)
                hea_rot2(v[0][r].e[0], v[0][r].e[1], v[1][r].e[0], v[1][r].e[1], (T)rec.d(2), (T)rec.d(3), (T)rec.d(0),
                         (T)rec.d(1), ry, rz);
    } else {
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (cslot >= 0 && !((r >> cslot) & 1)) continue;
#pragma unroll
            for (int k = 0; k < NV; k++) {
                const cx<T> p = v[k][r].e[0], o = v[k][r].e[1];
                v[k][r].e[0] = csel(on, o, p);
                v[k][r].e[1] = csel(on, p, o);
            }
        }
    }
}

template <typename T, int KH, int NV>
__global__ void __launch_bounds__(kBlock) k_hea(cx<T> *__restrict__ psi, cx<T> *__restrict__ lam, const HeaArgs a) {
    constexpr int VB = Traits<T>::VB, S = VB + 6, E = 1 << VB, R = 1 << KH;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // accumulator k of this lane: private, so no barrier until the end
    double *acc = reinterpret_cast<double *>(lds_raw) + wv * 64 + lane;
    for (int k = 0; k < a.n_acc; k++) acc[k * kBlock] = 0.0;
    uint64_t bid = blockIdx.x;
    if ((gridDim.x & 7) == 0) bid = (bid & 7) * (gridDim.x >> 3) + (bid >> 3);   // an eighth of the tiles per XCD
    uint32_t slot = 0;
#pragma unroll
    for (int k = 0; k < 6; k++) slot |= (uint32_t)((lane >> k) & 1) << a.lane_pos[k];
    slot &= (1u << (kPassMaxSlotBit + 1)) - 1;
    uint64_t hb[KH];
#pragma unroll
    for (int j = 0; j < KH; j++) hb[j] = 1ULL << a.reg_pos[j];
    for (uint64_t t = bid * (kBlock / 64) + wv; t < a.n_tiles; t += (uint64_t)gridDim.x * (kBlock / 64)) {
        uint64_t pt = 0;
#pragma unroll
        for (int k = 0; k < kPassMaxTileBits; k++)
            if (k < a.n_tile_bits) pt |= ((t >> k) & 1) << a.tile_pos[k];
        uint64_t tb = t << S;
#pragma unroll
        for (int j = 0; j < KH; j++) tb = insert_zero(tb, a.hpos[j]);
        const uint64_t base = tb + ((uint64_t)lane << VB);   // virtual index of register 0
        Pack<T> v[NV][R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            pass_ld<T>(row_ptr<T, KH>(psi, pt, hb, r) + slot, v[0][r]);
            if constexpr (NV == 2) pass_ld<T>(row_ptr<T, KH>(lam, pt, hb, r) + slot, v[1][r]);
        }
        for (int op = 0; op < a.n_ops; op++) {
            const HeaRec rec(a.ops + op);
            const int kind = rec.i(0), where = rec.i(1), at = rec.i(2);
            if (kind == HO_RZ) {
                if constexpr (NV == 1) {
                    const T c = (T)rec.d(0), s = (T)rec.d(1);
#pragma unroll
                    for (int r = 0; r < R; r++)
#pragma unroll
                        for (int e = 0; e < E; e++) {
                            const bool b = where == HW_SLOT ? ((r >> at) & 1) != 0 : (((base + e) >> at) & 1) != 0;
                            v[0][r].e[e] = hea_phase(v[0][r].e[e], c, b ? s : -s);
                        }
                }
                continue;
            }
            bool on[E];
            int cslot = -1;
#pragma unroll
            for (int e = 0; e < E; e++) on[e] = true;
            if (kind == HO_CNOT) {
                const int cw = rec.i(3), ca = rec.i(4);
                if (cw == HW_TILE && !((tb >> ca) & 1)) continue;   // the wave's control is 0
                if (cw == HW_SLOT) cslot = ca;
#pragma unroll
                for (int e = 0; e < E; e++) on[e] = cw == HW_SLOT || (((base + e) >> ca) & 1) != 0;
            }
            double ry = 0.0, rz = 0.0;
            if (where == HW_VEC) {
                if constexpr (E == 2) hea_vec<T, NV, R>(v, rec, kind, on[0], cslot, ry, rz);
            } else {
                switch (where * 8 + at) {
                case 0: hea_slot<T, 0, NV, R, E>(v, rec, kind, on, cslot, ry, rz); break;
                case 1: if constexpr (KH > 1) hea_slot<T, 1, NV, R, E>(v, rec, kind, on, cslot, ry, rz); break;
                case 2: if constexpr (KH > 2) hea_slot<T, 2, NV, R, E>(v, rec, kind, on, cslot, ry, rz); break;
                case 3: if constexpr (KH > 3) hea_slot<T, 3, NV, R, E>(v, rec, kind, on, cslot, ry, rz); break;
                case 4: if constexpr (KH > 4) hea_slot<T, 4, NV, R, E>(v, rec, kind, on, cslot, ry, rz); break;
                case 8: hea_lane<T, 1, NV, R, E>(v, rec, kind, lane, on, cslot, ry, rz); break;
                case 9: hea_lane<T, 2, NV, R, E>(v, rec, kind, lane, on, cslot, ry, rz); break;
                case 10: hea_lane<T, 4, NV, R, E>(v, rec, kind, lane, on, cslot, ry, rz); break;
                case 11: hea_lane<T, 8, NV, R, E>(v, rec, kind, lane, on, cslot, ry, rz); break;
                case 12: hea_lane<T, 16, NV, R, E>(v, rec, kind, lane, on, cslot, ry, rz); break;
                case 13: hea_lane<T, 32, NV, R, E>(v, rec, kind, lane, on, cslot, ry, rz); break;
                default: break;
                }
            }
            if (kind == HO_ROT2) {
                const int k = rec.i(5);
                acc[k * kBlock] += ry;
                acc[(k + 1) * kBlock] += rz;
            }
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            pass_st<T>(row_ptr<T, KH>(psi, pt, hb, r) + slot, v[0][r]);
            if constexpr (NV == 2) pass_st<T>(row_ptr<T, KH>(lam, pt, hb, r) + slot, v[1][r]);
        }
    }
    if (a.n_acc == 0) return;
    __syncthreads();
    const double *all = reinterpret_cast<const double *>(lds_raw);
    for (int k = wv; k < a.n_acc; k += kBlock / 64) {   // one wave per accumulator
        double x = 0.0;
        for (int w = 0; w < kBlock / 64; w++) x += all[k * kBlock + w * 64 + lane];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
        if (lane == 0) a.part[(uint64_t)a.slot[k] * gridDim.x + blockIdx.x] = x;
    }
}

}  // namespace sqk
