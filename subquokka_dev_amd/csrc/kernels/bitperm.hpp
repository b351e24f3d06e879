// bitperm.hpp -- passes that move index bit q of the state to bit p[q] (any
// permutation of the index bits, out of place; an involution, in place).
//
// A workgroup owns the 2^tb amplitudes that share the values of every bit
// outside a set T of tile bits.  T holds the low c bits and the bits that
// land on them, so both sides are read and written in runs of 2^c amplitudes.
// The tile goes through LDS: read in source order, written in destination
// order.  Both sides are read and written once: one pass of HBM traffic
// whatever the permutation.
//
// HBM-bound: the tile is small (2^10 amplitudes at most, c = 5: runs of 512
// bytes in complex128), so ten workgroups share a CU, and a thread's address
// is its own bits' part (computed once) plus a uniform part per iteration.
// Slots are XOR-folded over the bank bits, since a destination run reads LDS
// with a power-of-two stride.
#pragma once
#include "common.hpp"

namespace sqk {

constexpr int kPermMaxTile = 12;   // tile bits the argument arrays hold
constexpr int kPermTile = 10;      // tile bits a launch aims at
constexpr int kPermMaxBits = 40;
constexpr int kBlockBits = 8;      // log2(kBlock)

struct BitPermArgs {
    int tb;                             // tile bits
    int n_other;                        // the other bits: log2 of the workgroup count
    int ld_src[kPermMaxTile];           // source bit of load-order bit k (k < c: bit k itself)
    int st_loc[kPermMaxTile];           // load-order position of the bit that store-order bit k carries
    int st_dst[kPermMaxTile];           // destination bit of store-order bit k (k < c: bit k itself)
    int other_src[kPermMaxBits];        // the bits outside the tile, ascending: where they are read
    int other_dst[kPermMaxBits];        // and where they are written
};

__device__ inline uint32_t perm_slot(uint32_t i) { return i ^ ((i >> 5) & 31u); }

// Positions of the bits of x (from bit `from` on) given by pos[].
__device__ inline uint64_t perm_spread(uint32_t x, const int *pos, int from, int to) {
    uint64_t o = 0;
    for (int k = from; k < to; k++) o |= (uint64_t)((x >> k) & 1) << pos[k];
    return o;
}

template <typename T>
__global__ void __launch_bounds__(kBlock) k_bitperm(const cx<T> *__restrict__ src, cx<T> *__restrict__ dst,
                                                    const BitPermArgs a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    cx<T> *lds = reinterpret_cast<cx<T> *>(lds_raw);
    const uint64_t w = blockIdx.x;
    uint64_t sb = 0, db = 0;   // the tile's fixed bits, read and written (uniform)
    for (int k = 0; k < a.n_other; k++) {
        const uint64_t b = (w >> k) & 1;
        sb |= b << a.other_src[k];
        db |= b << a.other_dst[k];
    }
    const uint32_t cnt = 1u << a.tb, tid = threadIdx.x;
    const int lo = a.tb < kBlockBits ? a.tb : kBlockBits;
    const uint64_t so = sb + perm_spread(tid, a.ld_src, 0, lo);
    for (uint32_t i = tid; i < cnt; i += kBlock) lds[perm_slot(i)] = src[so + perm_spread(i - tid, a.ld_src, lo, a.tb)];
    __syncthreads();
    const uint64_t d = db + perm_spread(tid, a.st_dst, 0, lo);
    const uint32_t i0 = (uint32_t)perm_spread(tid, a.st_loc, 0, lo);
    for (uint32_t j = tid; j < cnt; j += kBlock)
        dst[d + perm_spread(j - tid, a.st_dst, lo, a.tb)] = lds[perm_slot(i0 | (uint32_t)perm_spread(j - tid, a.st_loc, lo, a.tb))];
}

// In place, for a permutation that is its own inverse (other_dst and st_dst as
// above): the workgroup of tile x exchanges it with the tile x's fixed bits
// move to; the lower one of the two does the work.
template <typename T>
__global__ void __launch_bounds__(kBlock) k_bitswap(cx<T> *__restrict__ s, cx<T> *__restrict__ s2, const BitPermArgs a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    cx<T> *lds = reinterpret_cast<cx<T> *>(lds_raw);
    uint64_t w = blockIdx.x;
    if (w >> a.n_other) {   // the second state's tiles
        w &= (1ULL << a.n_other) - 1;
        s = s2;
    }
    uint64_t sb = 0, db = 0;
    for (int k = 0; k < a.n_other; k++) {
        const uint64_t b = (w >> k) & 1;
        sb |= b << a.other_src[k];
        db |= b << a.other_dst[k];
    }
    if (db < sb) return;
    const bool two = db != sb;
    const uint32_t cnt = 1u << a.tb, tid = threadIdx.x;
    const int lo = a.tb < kBlockBits ? a.tb : kBlockBits;
    const uint64_t so = perm_spread(tid, a.ld_src, 0, lo);
    for (uint32_t i = tid; i < cnt; i += kBlock) {
        const uint64_t off = so + perm_spread(i - tid, a.ld_src, lo, a.tb);
        lds[perm_slot(i)] = s[sb + off];
        if (two) lds[cnt + perm_slot(i)] = s[db + off];
    }
    __syncthreads();
    const uint64_t d = perm_spread(tid, a.st_dst, 0, lo);
    const uint32_t i0 = (uint32_t)perm_spread(tid, a.st_loc, 0, lo);
    for (uint32_t j = tid; j < cnt; j += kBlock) {
        const uint64_t off = d + perm_spread(j - tid, a.st_dst, lo, a.tb);
        const uint32_t i = perm_slot(i0 | (uint32_t)perm_spread(j - tid, a.st_loc, lo, a.tb));
        s[db + off] = lds[i];
        if (two) s[sb + off] = lds[cnt + i];
    }
}

}  // namespace sqk
