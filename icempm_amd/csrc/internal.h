// internal.h -- launchers shared between the translation units of
// libicempm_hip.so.  Not part of the C ABI.
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "../host/parameters_sim.h"
#include "host_guard.h"
#include "mpm_device.h"

namespace icempm {

// Geometry of the shared-memory window that one P2G / G2P workgroup uses:
// a chunk of at most kChunk consecutive particles whose base cells lie in
// one cell row at build time; the window spans kWinX x kWinY grid nodes from
// the chunk's minimum base cell.
constexpr int kChunk = 256;
constexpr int kWinX = 128;
constexpr int kWinY = 4;

// ---- kernels.hip ------------------------------------------------------------
hipError_t launch_fill_f64(double *p, size_t n, double v, hipStream_t s);
hipError_t launch_fill_i32(int *p, size_t n, int v, hipStream_t s);

// ORDERED mode: where a particle pass leaves the points' records, and the
// indenter force that one workgroup folds (see ordered_device.h).
struct PointRec;
struct PointLists {
    PointRec *rec;   // null: none
    int *bucket;
    int2 *cells;
    int *next;
};
struct BinsFold {
    double *bins;    // null: nothing to do
    const int *nodeBin;
    const double *nodeF;
    double *hist2;
    int nb, gx, x0, y0, w, h;
};
struct PassExtra {
    PointLists lists;
    BinsFold force;
};

// ---- particles_exact.hip / particles_fast.hip ---------------------------------
// The particle pass.  do_g2p: gather from gridV (velocities in rows 1-2) and
// update the particles; do_p2g: scatter the (updated) particles into gridOut
// (mass, momentum).  gridV and gridOut may be the same buffer only when one
// of the two passes is off.  exact:: is built without FMA contraction
// (ORDERED mode), fast:: with it (FAST mode).  kind selects the kernel
// variant: 0 workgroup windows (shared-memory gather and scatter), 1 wavefront
// windows (direct gather, per-wavefront scatter), 2 as 1 with the stencil
// order rotated per lane.
namespace exact {
hipError_t launch_particles(const KParams &k, bool do_g2p, bool do_p2g, const double *gridV,
                            double *gridOut, const int *chunkStart, int nChunks, int recordPQ,
                            hipStream_t s, int kind);
// The G2P of an ORDERED substep (kind 1 or 2) with what the next one needs.
hipError_t launch_g2p_records(const KParams &k, const double *gridV, const int *chunkStart, int nChunks,
                              int recordPQ, hipStream_t s, int kind, const PassExtra &extra);
}
namespace fast {
hipError_t launch_particles(const KParams &k, bool do_g2p, bool do_p2g, const double *gridV,
                            double *gridOut, const int *chunkStart, int nChunks, int recordPQ,
                            hipStream_t s, int kind);
}

// Grid update.  ordered: write each node's contact force and bin to
// nodeBin/nodeF for a later ordered fold; otherwise accumulate into k.bins
// and hist2 (if not null) with atomics.  zeroGrid (may be null): a second
// grid whose 3 rows are cleared in the same pass.
hipError_t launch_update(const KParams &k, double *grid, double ix, double iy, double *hist2,
                         double *zeroGrid, bool ordered, int *nodeBin, double *nodeF,
                         hipStream_t s);

// ORDERED mode: contributions in particle order per node.  cells[0] and cells[1]
// (in turn, see flip) count the points of every base cell and chain those past
// kCellCap; the one not in use is zero.
constexpr int kCellCap = 16;
struct OrderedScratch {
    double *rec = nullptr;       // 8 doubles per particle
    int *next = nullptr;         // chain of a crowded cell: point + 1, or 0
    int *bucket = nullptr;       // kCellCap points per cell
    int2 *cells[2] = {};         // {points, first of the chain + 1} per cell
    int flip = 0;
    int *nodeBin = nullptr;      // gridTotal
    double *nodeF = nullptr;     // 2 per node
    size_t nPts = 0, nGrid = 0, cleared = 0;
};
// The points' records and cell lists for the next fold, in the list not in use.
PointLists ordered_lists(const OrderedScratch &o);
// Makes them; padGrid (may be null): the padding of its rows is cleared.
hipError_t ordered_records(const KParams &k, const OrderedScratch &o, double *padGrid, hipStream_t s);
// The P2G of the records into grid; update: with the grid update, for an
// indenter at (ix, iy).
hipError_t ordered_fold(const KParams &k, double *grid, OrderedScratch &o, bool update, double ix, double iy,
                        hipStream_t s);
// The contact forces of the last update, with the indenter where it was: as
// arguments of a fold, and folded by a launch of its own.
BinsFold ordered_force(const KParams &k, const OrderedScratch &o, double *hist2, double ix, double iy);
hipError_t ordered_fold_forces(const KParams &k, OrderedScratch &o, double *hist2, double ix, double iy,
                               hipStream_t s);

hipError_t launch_hello(int *flag, hipStream_t s);
hipError_t launch_copy(const double *src, double *dst, size_t n_doubles, hipStream_t s);

// ---- batch.hip: the batches' substep kernel for one case ------------------------
// One launch per substep: grid update, G2P and the next P2G, FP64, exact return
// map; v, Bp, P and Q are not recorded.  It runs on a copy of the points in
// band order, which enter makes and leave takes back.  Three grids rotate: a
// substep reads in (mass and momentum of its P2G), adds the next P2G to out,
// which must be zero, and clears the third.
namespace single {
constexpr size_t kRecBytes = 48, kCaseBytes = 512;   // of a chunk record and of the case's constants
constexpr size_t copy_bytes(size_t pp) { return pp * (7 * sizeof(double) + 3); }
struct Run {
    const void *cp;          // the case's constants (device)
    void *bounds;            // 16 bytes: the box of touched nodes
    double *pts;             // 16 rows x pp
    size_t pp, gp;
    int n, gx, gy;
    const int *perm;         // slot -> point
    const int *starts;       // nChunks + 1 first slots
    void *recs;              // nChunks records, made by enter
    int nChunks;
    bool inOrder;            // the layout of their points, chosen by plan
    double *rows;            // the copy
    double *bins;
    int *err;
    hipStream_t stream;
};
// The case's constants, the indenter starting at (x0, y0), in out (kCaseBytes);
// false where the kernel does not take the case.
bool case_constants(const icy::SimParams &P, double x0, double y0, void *out);
// The points' band order as they are (in vals; keys, keys2, vals2: scratch of n
// ints, tmp: of radix_tmp_ints(n)) and its chunks' first slots; sets r.inOrder.
hipError_t plan(Run &r, int *keys, int *vals, int *keys2, int *vals2, int *tmp, std::vector<int> &starts);
// The points of the slots, from that order.
hipError_t slots(const Run &r, const int *sorted, int *perm);
hipError_t enter(const Run &r);
hipError_t leave(const Run &r);
// hist2: this substep's force (added to); t: its time; step: its index in the run.
hipError_t substep(const Run &r, const double *in, double *out, double *clear, double *hist2, double t, int step);
}  // namespace single

// ---- sort.hip -----------------------------------------------------------------
// Exclusive scan of n ints (in and out may alias).  tmp must hold
// scan_tmp_ints(n) ints.
size_t scan_tmp_ints(size_t n);
hipError_t exclusive_scan(const int *in, int *out, size_t n, int *tmp, hipStream_t s);

// Stable LSD radix sort of (key, value) pairs by signed 32-bit key.
// Buffers: keys/vals (in, out), keys2/vals2 (scratch of n), tmp of
// radix_tmp_ints(n) ints.  The result ends in keys/vals.
size_t radix_tmp_ints(size_t n);
hipError_t radix_sort_pairs(int *keys, int *vals, int *keys2, int *vals2, size_t n, int *tmp,
                            hipStream_t s);

// key_i of the particles in a point SoA
hipError_t launch_point_keys(const double *pts, size_t pp, int n, double hinv, int gridX,
                             int *keys, int *vals, hipStream_t s);
// key_i of raw float (x, y) pairs
hipError_t launch_raw_keys(const float *xy, int n, double hinv, int gridX, int *keys, int *vals,
                           hipStream_t s);
// dst = src permuted: dst slot k <- src slot perm[k], for all 16 rows
hipError_t launch_permute_points(const double *src, double *dst, size_t pp, int n,
                                 const int *perm, hipStream_t s);
hipError_t launch_permute_raw(const float *xy, const int16_t *g, float *xy2, int16_t *g2, int n,
                              const int *perm, hipStream_t s);

}  // namespace icempm
