// pa_order.h -- the workgroup -> (unit, block) order of the MFMA pass kernels: which
// (batch, head) unit and which block of it a workgroup runs.  Plain integer arithmetic with
// no HIP dependency, so that a host program can check it (tests/test_order.py).
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define PA_HD __host__ __device__ __forceinline__
#else
#define PA_HD inline
#endif

namespace pa {

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own L2).  Map the
// hardware id to a logical id so that every XCD runs a contiguous range of logical ids --
// consecutive logical ids share a head, so its K/V stay in that XCD's L2.
constexpr int kNumXcd = 8;
PA_HD int xcd_remap(int bid, int nblocks) {
    const int per = nblocks / kNumXcd, rem = nblocks % kNumXcd;
    const int x = bid % kNumXcd, slot = bid / kNumXcd;
    return (x < rem) ? x * (per + 1) + slot : rem * (per + 1) + (x - rem) * per + slot;
}

// The unit (batch-major, head-minor) of the j-th of the nu units that XCD x runs.  Where the
// heads split evenly over the XCDs in runs of whole groups (`group` consecutive heads share
// their K / V: GQA), each XCD takes heads [x * hpx, (x + 1) * hpx) of every batch row, so that
// work that differs by batch row (padding masks) is spread over all XCDs; otherwise the XCD's
// units are consecutive.
PA_HD int xcd_unit(int x, int j, int nu, int heads, int group) {
    if (heads % (kNumXcd * group) == 0) {
        const int hpx = heads / kNumXcd;
        return (j / hpx) * heads + x * hpx + j % hpx;
    }
    return x * nu + j;
}

// (unit, rank) of workgroup bid of a grid of nblocks = units x nblk workgroups.
// heavy (causal grids, work per block falling with its rank): every XCD runs whole units and
// dispatches the heaviest blocks of all its units first, so the light blocks fill the end of
// the kernel.  Otherwise each unit's blocks are consecutive on one XCD.  When the XCD ranges
// do not hold whole units, the order is unit by unit.  heads: units per batch row; group: see
// xcd_unit.
PA_HD void block_map(int bid, int nblocks, int nblk, int heads, int group, bool heavy,
                     int& unit, int& rank) {
    const int lid = xcd_remap(bid, nblocks);
    const int per = nblocks / kNumXcd;
    if (nblocks % kNumXcd == 0 && per % nblk == 0) {
        const int x = lid / per, k = lid % per, nu = per / nblk;
        if (heavy) {
            unit = xcd_unit(x, k % nu, nu, heads, group);
            rank = k / nu;
        } else {
            unit = xcd_unit(x, k / nblk, nu, heads, group);
            rank = k % nblk;
        }
    } else {
        unit = lid / nblk;
        rank = lid % nblk;
    }
}

// Whether a workgroup of 128 rows gets two groups of four waves, which share the `chain` positions that
// each row walks (forward and dQ: keys; dK/dV: queries of every head of the group).  Two groups halve
// the chain and fill a CU that has one workgroup, at the price of merging their sums; a CU holds
// one such workgroup where it holds two or three of one group, so beyond one workgroup per CU
// only long chains of causal grids, whose last rows run alone, still gain: how far depends on the
// workgroups of an XCD (32 CUs), and on whether the XCDs hold whole units (units not a multiple
// of 8 run unit by unit, and an XCD may end with a unit of its own).
// Measured on passes of heads x length at d = 64, us with one group / two, forward and backward:
//   causal, up to 256 workgroups: 16 x 512 15.0 / 10.8 and 29.7 / 28.6, 16 x 256 10.3 / 8.5 and 20.8 / 21.7,
//   8 x 4096 74 / 40 and 147 / 117; 16 x 128 7.5 / 7.3 and 16.4 / 18.7;
//   causal, more: 80 x 512 15.3 / 14.0 and 34 / 40, 48 x 900 two 1.19 and 0.94 times as fast, 32 x 1200 1.59
//   and 1.15, 40 x 1200 1.30 and 0.97, 16 x 4096 1.53 and 1.12, 20 x 2560 1.11 and 0.91, 24 x 2816 1.31 and
//   0.98, 128 x 384 12.4 / 14.1 and 30 / 40, 40 x 2048 1.05 and 0.83, 48 x 2048 0.96 and 0.83;
//   not causal: 16 x 512 15.1 / 10.5 and 27.8 / 27.7, 21 x 768 19.3 / 12.4 and 35.8 / 34.5, 32 x 1024 23.9 /
//   15.9 and 47.8 / 45.5, 40 x 1024 23.9 / 27.4 and 63 / 80, 8 x 4096 76 / 44 and 144 / 131.
// d = 128 (forward, and dQ with the one dK/dV): 16 x 256 11.1 / 11.7 and 35.0 / 34.8, 64 x 384 14.6 / 14.3 and
//   46.9 / 45.2, causal 106 x 384 22.1 / 24.2 and 71.7 / 71.4, 80 x 512 20.2 / 23.3 and 63.7 / 66.2, 53 x 768
//   31.9 / 30.4 and 105 / 98; 16 x 4096 99 / 83 and 327 / 286.
PA_HD bool two_wave_groups(bool fwd, int dim, bool causal, int64_t units, int rows, int64_t chain) {
    const int64_t per_unit = (rows + 127) / 128, wgs = units * per_unit;
    if (dim == 128) {
        if (!fwd && wgs <= 256) return chain > 192;
        return chain >= (causal && wgs > 256 ? 768 : 384);
    }
    if (wgs <= 256) return fwd ? causal || chain > 128 : chain >= (causal ? 448 : 576);
    if (!causal) return false;
    const int64_t xcd = (units + kNumXcd - 1) / kNumXcd * per_unit;  // workgroups of the fullest XCD
    const bool even = units % kNumXcd == 0;
    if (fwd) {
        if (xcd <= 48) return chain >= (xcd <= 40 ? 512 : 768);
        if (chain >= 2048) return wgs < 768;
        return even && xcd <= 72 && chain >= (xcd <= 64 ? 768 : 1536);
    }
    if (xcd <= 48) return chain > 1024;
    return xcd <= 64 && chain >= 2048 && (even || units <= 2 * kNumXcd);
}

}  // namespace pa
