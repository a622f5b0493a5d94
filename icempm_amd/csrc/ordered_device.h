// ordered_device.h -- device pieces of ORDERED mode that the node fold
// (kernels.hip) and the exact particle pass (particles_exact.hip) share: the
// points' records and cell lists, and the fold of the indenter force.  Built
// without FMA contraction in both.
#pragma once

#include "internal.h"

namespace icempm {

// What a point's contributions follow from, 64 bytes.
struct PointRec {
    double2 f, a, b, mv;   // offset in its cell, affine momentum (rows), momentum
};

// A point's record, and its entry in the list of its base cell.
static __device__ __forceinline__ void point_record(const KParams &k, const PointLists &L, int pt, double px, double py,
                                                    double vx, double vy, double F00, double F01, double F10, double F11,
                                                    double B00, double B01, double B10, double B11) {
    int bx, by;
    double fx0, fx1, w0, w1, w2;
    if (!stencil(px, k.h_inv, bx, fx0, w0, w1, w2) || !stencil(py, k.h_inv, by, fx1, w0, w1, w2)) {
        flag_error(k);
        return;
    }
    // the cell's list first: the place in it is on its way while the stress is made
    if (bx >= k.gridX - 2 || by >= k.gridY - 2) flag_error(k);   // nodes outside the grid take nothing
    const bool in = bx < k.gridX && by < k.gridY;
    const int at = in ? bx + by * k.gridX : 0;
    int *cell = reinterpret_cast<int *>(L.cells + at);
    int slot = 0;
    if (in) slot = atomicAdd(cell, 1);
    double t00, t01, t11;
    kirchhoff(F00, F01, F10, F11, k.mu, k.kappa, t00, t01, t11);
    const double m = k.mass;
    const double sc = k.dt * k.vol * k.Dinv;
    L.rec[pt] = PointRec{make_double2(fx0, fx1), make_double2(m * B00 - sc * t00, m * B01 - sc * t01),
                       make_double2(m * B10 - sc * t01, m * B11 - sc * t11), make_double2(vx * m, vy * m)};
    if (!in) return;
    if (slot < kCellCap)
        L.bucket[kCellCap * (size_t)at + slot] = pt;
    else
        L.next[pt] = atomicExch(cell + 1, pt + 1);
}

// ORDERED indenter force: each bin, and the substep's total, summed in node
// order by one thread each over the nodes in contact.  One workgroup: it looks
// only at the w x h nodes around the disc, and leaves those in contact in LDS,
// 256 nodes at a time.  In a run it is one more workgroup of the G2P (a launch of
// its own takes 4.5 us).
constexpr int kFoldBlock = 256, kFoldBinsMax = 1024;   // bins and the total
struct BinsLds {
    int bin[kFoldBlock], wave[kFoldBlock / 64];
    double f0[kFoldBlock], f1[kFoldBlock];
};
static __device__ void fold_bins(const BinsFold &B, BinsLds &L) {
    constexpr int kPer = kFoldBinsMax / kFoldBlock;
    const int t = threadIdx.x, nb = B.nb;
    double a0[kPer], a1[kPer];
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const int b = t + kFoldBlock * q;
        a0[q] = b < nb ? B.bins[2 * b] : 0.0;
        a1[q] = b < nb ? B.bins[2 * b + 1] : 0.0;
    }
    const long nodes = (long)B.w * B.h;
    for (long first = 0; first < nodes; first += kFoldBlock) {
        const long e = first + t;
        int b = -1, idx = 0;
        if (e < nodes) {
            idx = B.x0 + (int)(e % B.w) + (B.y0 + (int)(e / B.w)) * B.gx;
            b = B.nodeBin[idx];
        }
        const unsigned long long hit = __ballot(b >= 0);
        if ((t & 63) == 0) L.wave[t >> 6] = __popcll(hit);
        __syncthreads();
        int at = __popcll(hit & ((1ull << (t & 63)) - 1ull)), count = 0;
        for (int q = 0; q < kFoldBlock / 64; ++q) {
            if (q < t >> 6) at += L.wave[q];
            count += L.wave[q];
        }
        if (b >= 0) {
            L.bin[at] = b;
            L.f0[at] = B.nodeF[2 * (size_t)idx];
            L.f1[at] = B.nodeF[2 * (size_t)idx + 1];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            const int mine = t + kFoldBlock * q;
            if (mine <= nb)
                for (int c = 0; c < count; ++c)
                    if (mine == nb || L.bin[c] == mine) {
                        a0[q] += L.f0[c];
                        a1[q] += L.f1[c];
                    }
        }
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const int b = t + kFoldBlock * q;
        if (b < nb) {
            B.bins[2 * b] = a0[q];
            B.bins[2 * b + 1] = a1[q];
        } else if (b == nb && B.hist2) {
            B.hist2[0] = a0[q];
            B.hist2[1] = a1[q];
        }
    }
}

}  // namespace icempm
