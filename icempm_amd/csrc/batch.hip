// batch.hip -- many independent indentation cases of uneven size advanced
// together: one launch per substep does the grid update, the G2P and the next
// P2G of every case, and the substep loop is captured once in a HIP graph and
// replayed.
//
// Storage (per batch, cases contiguous, each case in band order):
//   F64 variant    positions: 2 rows of double; vel(2) Fe(4) Bp(4) Jp_inv(1):
//                  11 rows of double
//   F32 variant    positions: 48-bit fixed point over the case's grid width,
//                  3 rows of u32 (x high 32 bits, y high 32 bits, both low
//                  16-bit halves); vel(2) Fe-I(4) Bp(4) Jp_inv-1(1): 11 rows
//                  of float.  Fe and Jp_inv are stored as their deviations
//                  from 1 so that float keeps them to ~1e-12 absolute.
//   crushed        1 byte per point
//   grain          i16 per point, only when a case has GrainVariability != 0
//   grids          three grids of 3 rows of double per node (mass, momentum),
//                  cases concatenated: a substep reads one, scatters into the
//                  next and clears the third
// All arithmetic is FP64 in both variants (the return map included); the F32
// variant only stores less: a fused pass moves 49 B per point instead of 97 B.
// A case's NACC strengths are uniform (constants per case) or vary per grain
// id as GetParametersForGrain makes them (gpu_implementation5.cu:97-111).
#include <algorithm>
#include <atomic>
#include <chrono>
#include <climits>
#include <cmath>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <string>
#include <system_error>
#include <thread>
#include <type_traits>
#include <vector>

#include "../../include/icempm.h"
#include "../host/parameters_sim.h"
#include "internal.h"
#include "mlp_device.h"

namespace icempm {
namespace batch {

// The substep kernel's device functions, without contraction for the batches and
// with it for a single case, as their particle passes have always been built.  It
// matters: without contraction det F = F00 F11 - F10 F01 and J^2 - 1 round twice
// more at 1e-16 in every substep, of a strain of 1e-5, and the in-cell offset x /
// h - base at the size of x / h, not of the offset.  Over 2,500 substeps of 2,400
// points that set the uncontracted Bp apart from the particle pass's by half of
// a run's scatter (2e-10 of its norm in the median, 2e-9 in some inputs);
// contracted, the means of 24 runs agree to what 24 runs can show.
struct PlainMath {
#include "fast_math.inc"
};
}  // namespace batch
}  // namespace icempm

#pragma clang fp contract(fast)

namespace icempm {
namespace batch {

struct FusedMath {
#include "fast_math.inc"
};

struct CaseParams {
    double dt, vol, mass, h, h_inv, Dinv, mu, kappa, gravity, indRsq, indV;
    double ics, its, iss, tanPhi, dpThr, x0, y0;
    double pmax, msq, betaPmax, onePlus2Beta, slope;   // NACC constants of the case's material (grain 0)
    double grainVar;        // GrainVariability: 0 = the constants above hold for every point
    // FP32 storage: a coordinate is a 48-bit integer u with x / h = u 2^-F,
    // F = 48 - the bits a cell index of the case needs: the quantum in metres
    // (h 2^-F) and its inverse, and in cell units 2^-F, 2^(16 - F), 2^F
    double posQ, posInvQ, cellQ, cellQ16, cellInvQ;
    double gxInv;           // 1 / gx: a node's row from its index
    double scm;             // dt V_p D^-1 / m_p: the stress term of the affine momentum per unit mass
    double vmax;            // the speed limit, half a cell per substep
    double dtCells;         // dt / h
    int gx, gy, gridTotal, nPts, ptOffset, gridOffset;
    int nbins, binOffset;   // indenter force bins: n_indenter_subdivisions, first double in the bin array
};

#ifndef ICEMPM_BATCH_CHAINS
#define ICEMPM_BATCH_CHAINS 2   // independent chains of a batched run (groups of cases)
#endif

// Point rows.  FP64 storage: positions FP64.  FP32 storage: positions as
// 48-bit fixed point in units of h 2^-F, the cell index in the top 48 - F
// bits (F = 48 - the bits of the larger grid dimension: a quantum of at most
// ~2 gx h / 2^48, ~2e-14 m for a 3 m grid; a substep moves a point by ~1e-6
// m, which an FP32 coordinate could not resolve, and 32 bits -- a quantum of
// ~7e-10 m -- rounded each displacement by ~1e-4 of itself, enough to move
// the force history of a fracturing case by ~1%); the base cell and in-cell
// offset of a stencil are exact functions of the integer.  The other values
// FP32.
template <bool F32>
struct Rows {
    using V = typename std::conditional<F32, float, double>::type;
    using P = typename std::conditional<F32, unsigned int, double>::type;
    // FP64: rows x, y.  FP32: one 16-byte record per slot, {high 32 bits of
    // x, of y, the two low 16-bit halves, the crushed flag | grain id << 16}
    // (one load and one store per pass; the crushed and grain rows are then
    // unused)
    static constexpr int kPosRows = F32 ? 4 : 2;
    P *pos;            // kPosRows values per slot
    V *rest;           // 11 rows: vel(2) Fe(4) Bp(4) Jp(1)
    unsigned char *crushed;
    short *grain;      // null when every case is uniform
    size_t pitch;
};

constexpr double kFix48Max = 281474976710655.0;   // 2^48 - 1

// Element i of a row through a 32-bit byte offset from the row's start: the
// row start is wavefront-uniform (scalar registers), so the access takes the
// scalar-base + 32-bit vector-offset form, with no 64-bit address arithmetic
// per lane.  Rows hold < 2^29 elements (finalize refuses larger batches), so
// i * sizeof(T) < 2^32.
template <class T>
static __device__ __forceinline__ T *at(T *row, unsigned i) {
    using B = typename std::conditional<std::is_const<T>::value, const char, char>::type;
    return reinterpret_cast<T *>(reinterpret_cast<B *>(row) + i * (unsigned)sizeof(T));
}

// FP32 storage: a coordinate as 48-bit fixed point, u = hi 2^16 + lo, in
// metres (round to nearest; below 0 to 0, above 2^48 - 1 quanta and NaN to
// 2^48 - 1, past the grid's edge, where the next stencil check flags them).
// Every step is exact in FP64 except the scalings by posQ / posInvQ.
static __host__ __device__ inline double fix48_get(unsigned int hi, unsigned int lo, const CaseParams &cp) {
    return ((double)hi * 65536.0 + (double)lo) * cp.posQ;
}
static __host__ __device__ inline void fix48_put(double x, const CaseParams &cp, unsigned int &hi, unsigned int &lo) {
    double u = rint(x * cp.posInvQ);
    u = (u >= 0.0 && u <= kFix48Max) ? u : (u < 0.0 ? 0.0 : kFix48Max);
    const double uh = floor(u * (1.0 / 65536.0));
    hi = (unsigned int)uh;
    lo = (unsigned int)(u - uh * 65536.0);
}
// The same in cell units (xr = x / h = u 2^-F): exact both ways, the
// scalings being powers of 2.  fix_put_cells returns u.
static __device__ __forceinline__ double fix_cells(unsigned int hi, unsigned int lo, const CaseParams &cp) {
    return fma((double)hi, cp.cellQ16, (double)lo * cp.cellQ);
}
static __device__ __forceinline__ double fix_put_cells(double xr, const CaseParams &cp, unsigned int &hi,
                                                       unsigned int &lo) {
    // clamped (NaN to the top), then u + 2^52: its low 48 mantissa bits are u,
    // rounded to nearest even as rint would
    const double top = kFix48Max * cp.cellQ;
    const double c = xr >= 0.0 ? fmin(xr, top) : (xr < 0.0 ? 0.0 : top);
    const double s = fma(c, cp.cellInvQ, 0x1p52);
    const unsigned long long b = __builtin_bit_cast(unsigned long long, s);
    hi = (unsigned int)(b >> 16);
    lo = (unsigned int)b & 0xFFFFu;
    return s - 0x1p52;
}
// The quadratic B-spline stencil (gpu_implementation5.cu:185-193) of a
// coordinate in cell units: base cell floor(xr - 0.5), 0 below xr = 0.5 (as
// the truncation of the FP64 form gives), and offset fx = xr - base, both
// exact for the xr of a record.
static __device__ __forceinline__ void stencil_cells(double xr, int &base, double &fx, double &w0, double &w1,
                                                     double &w2) {
    const double b = fmax(floor(xr - 0.5), 0.0);
    base = (int)b;
    fx = xr - b;
    const double v0 = 1.5 - fx, v1 = fx - 1.0, v2 = fx - 0.5;
    w0 = 0.5 * v0 * v0;
    w1 = 0.75 - v1 * v1;
    w2 = 0.5 * v2 * v2;
}

// Point position of slot pt (both storage formats) as FP64; store it back,
// and the value the stored form holds.
static __device__ __forceinline__ void pos_load(const double *pos, size_t pp, int pt, const CaseParams &,
                                                double &x, double &y) {
    const unsigned u = (unsigned)pt;
    x = *at(pos, u);
    y = *at(pos + pp, u);
}
typedef unsigned int prec4 __attribute__((ext_vector_type(4)));
// FP32 storage: the slot's record, its coordinates in metres; returns its
// last word (crushed flag in bits 0-7, grain id in bits 16-31)
static __device__ __forceinline__ unsigned pos_load(const unsigned int *pos, size_t, int pt, const CaseParams &cp,
                                                    double &x, double &y) {
    const prec4 v = reinterpret_cast<const prec4 *>(pos)[pt];
    x = fix48_get(v.x, v.z & 0xFFFFu, cp);
    y = fix48_get(v.y, v.z >> 16, cp);
    return v.w;
}
// FP64 storage: stores (x, y), through the L2 (a wavefront's 512 B of a row
// straddle cache lines that the neighbouring wavefronts complete: measured
// 6% faster than non-temporal stores).  The FP32 record streams
// non-temporally (measured faster that way).
static __device__ __forceinline__ void pos_store(double *pos, size_t pp, int pt, double x, double y) {
    const unsigned u = (unsigned)pt;
    *at(pos, u) = x;
    *at(pos + pp, u) = y;
}

// FP32 storage keeps a point's Fe - I as one 16-byte record in the space of
// rest rows 2-5 (one float4 per point, one load and one store per pass
// instead of four of each); FP64 storage keeps the four rows.
typedef float fe4 __attribute__((ext_vector_type(4)));
static __device__ __forceinline__ fe4 *fe_rec(float *R, size_t pp) { return reinterpret_cast<fe4 *>(R + pp * 2); }
static __device__ __forceinline__ const fe4 *fe_rec(const float *R, size_t pp) {
    return reinterpret_cast<const fe4 *>(R + pp * 2);
}

static __device__ __forceinline__ void wsync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Band order of a case's base cells: the rows in pairs (bands, a last odd
// row alone), a band column by column with the two cells of a column
// together.  Consecutive cells then cover two rows: a wavefront's 64 points
// (16 cells at 4 per cell) lie in 2 x 8 cells, whose stencils touch 4 x 10
// grid nodes, where 1 x 16 cells of a row-major order touch 3 x 18.  The
// keys of a case are a bijection onto [0, gx * gy).
static __host__ __device__ inline int band_key(int x, int y, int gx, int gy) {
    const int band = y >> 1;
    const int rows = (gy - 2 * band) < 2 ? 1 : 2;
    return band * 2 * gx + x * rows + (y & 1);
}
static __host__ __device__ inline void band_cell(int key, int gx, int gy, int &x, int &y) {
    const int band = key / (2 * gx);
    const int w = key - band * 2 * gx;
    const int rows = (gy - 2 * band) < 2 ? 1 : 2;
    x = w / rows;
    y = 2 * band + w % rows;
}

static __device__ __forceinline__ KParams kp_of(const CaseParams &c, int *err) {
    KParams k{};
    k.err = err;
    k.gridX = c.gx;
    k.gridY = c.gy;
    k.dt = c.dt; k.vol = c.vol; k.mass = c.mass; k.h = c.h; k.h_inv = c.h_inv; k.Dinv = c.Dinv;
    k.mu = c.mu; k.kappa = c.kappa; k.gravity = c.gravity; k.indRsq = c.indRsq; k.indV = c.indV;
    k.ics = c.ics; k.its = c.its; k.iss = c.iss; k.tanPhi = c.tanPhi; k.dpThr = c.dpThr;
    k.grainVar = c.grainVar;
    return k;
}

// Return map of crushed points: the exact Drucker-Prager map, the exact map
// while recording (trial, projected) pairs, or the learned map with the
// exact one as fallback.  kMapSingle: the exact map of a single case (FusedMath).
enum { kMapExact = 0, kMapHarvest = 1, kMapLearned = 2, kMapSingle = 3 };

struct LearnArgs {
    const unsigned short *wbf;   // MLP weights, BF16 bits
    const float *pf;             // MLP parameters, FP32 (biases)
    mlpdev::Norm norm;
    double tol;                  // accepted when the yield residual is <= tol
    float *hx, *ht;              // harvest: inputs (n x 5), targets (n x 3)
    unsigned long long *hcount;
    int hcap;
    // [accepted, fell back, inside the surface, tension accepted, tension fell
    // back, shear accepted, shear fell back] (the last four: map kernel only)
    unsigned long long *stats;
    int branches;                // kMapTension | kMapShear: branches the network proposes for
};

constexpr int kMapStats = 7;
enum { kMapTension = 1, kMapShear = 2 };

// A crushed point whose projection is deferred to the map kernel: its trial
// elastic deformation (FP64) and Jp_inv, and where it lives.
struct MapEntry {
    int pt, cs;
    double F[4];
    double Jp;
    double x[2], v[2], B[4];   // position, velocity and Bp for its P2G
};

// Queue of deferred points of one pass (learned map only).
struct MapQueue {
    MapEntry *q;
    unsigned int *count;   // appended by the particle pass
    int cap;
};

// The branch of the exact map (Wolper_Drucker_Prager, gpu_implementation5.cu:48-94)
// a crushed trial state falls in, decided exactly: the tension branch, the
// shear projection onto q = q_lim, or inside the surface (the map is the
// identity there).  qlim is set for the shear branch.
enum { kBrInside = 0, kBrTension = 1, kBrShear = 2 };
static __device__ __forceinline__ int map_branch(const KParams &k, const Trial &r, double Jp, double &qlim) {
    qlim = 0;
    if (r.p < -k.dpThr || Jp < 1) return kBrTension;
    qlim = (r.p > k.ics) ? 0.0 : fmin((r.p + k.dpThr) * k.tanPhi, k.iss);
    return (r.q >= qlim) ? kBrShear : kBrInside;
}

// Raw features of a crushed point for the map: log s0, log s1, log Jp_inv,
// a hardening variable the reference does not have (0), and the yield-state
// flag: 1 in the tension branch, 0 in the shear branch.
static __device__ __forceinline__ void map_features(const Trial &r, double Jp, int br, double f[5]) {
    f[0] = log(r.svd.s0);
    f[1] = log(r.svd.s1);
    f[2] = log(Jp);
    f[3] = 0.0;
    f[4] = (br == kBrTension) ? 1.0 : 0.0;
}

// Yield residual of a proposed projected state (s0, s1, Jpn), as stress
// errors relative to the case's strengths:
//  tension  the state must be isotropic at p = -p_thr:
//           max(|p(s) + p_thr| / pmax, q(s) / qmax, |Jpn / Jp_exact - 1|)
//  shear    the deviator (scaled with the trial J, as the map scales it)
//           must sit at q_lim and the mean of s^2 must be kept:
//           max(|q~(s) - q_lim| / qmax, kappa |mean s^2 - mean s_tr^2| / pmax)
static __device__ __forceinline__ double yield_residual(const KParams &k, const Trial &r, double Jp, int br,
                                                        double qlim, double s0, double s1, double Jpn) {
    const double a = s0 * s0, b = s1 * s1;
    if (br == kBrTension) {
        const double Je_new = sqrt(-2. * -k.dpThr / k.kappa + 1.);
        const double Jn = s0 * s1;
        const double pn = -(k.kappa / 2.) * (Jn * Jn - 1.);
        const double qn = (k.mu / Jn) * fabs(a - b);
        double res = fabs(pn + k.dpThr) / k.ics;
        res = fmax(res, qn / k.iss);
        res = fmax(res, fabs(Jpn / (Jp * (Je_new / r.Je)) - 1.));
        return res;
    }
    const double qt = (k.mu / r.Je) * fabs(a - b);
    const double dm = 0.5 * (a + b) - 0.5 * (r.ss0 + r.ss1);
    return fmax(fabs(qt - qlim) / k.iss, k.kappa * fabs(dm) / k.ics);
}

// A chunk: the up to 256 points of a workgroup and the box of grid nodes their
// stencils touch.  The workgroup keeps the box in the record, renewing it every
// kBoxEvery substeps (points move far less than a cell in that time; one that
// has left it takes the general paths).
struct __attribute__((aligned(16))) ChunkRec {
    int beg;          // first slot
    unsigned shape;   // points in band order: their number; else lanes per row | rows with one lane more << 8 | rows << 16
    int cs, gofs;     // the case and its first grid node
    unsigned dims;    // GridX | GridY << 16
    unsigned org;     // the box: first column | first row << 16
    unsigned ext;     // columns | rows << 8 | tile stride << 16 | FP64: window stride << 24 (0: no box)
    unsigned inv;     // ceil(2^16 / columns): a node's row from its index in the box
    unsigned win[4];  // FP32: the windows: first column | first row << 8 (both from the box's) | columns << 16 | rows << 24
};
constexpr int kBoxEvery = 8;

// The points of a chunk, in one of two layouts.
//
// In order (FP32 storage, workgroups of fewer than four wavefronts, dense clouds):
// in band order, 64 a wavefront.  The four lanes of a quad mostly hold the points of
// a cell and add up their contributions before these reach the window (FP32: the
// wavefront's, which keeps the sums of a node in the order quad, wavefront, grid).
//
// In rows (FP64 storage otherwise): in rows of a wavefront each, as few as hold them
// and filled evenly; slot s holds the point that band order puts at chunk_point(s,
// shape).  Consecutive points go to the same lane of consecutive rows, so that the
// 64 lanes of a wavefront hold different cells, at four points a cell, and their LDS
// atomics, 27 a point into one window for the workgroup, go to different nodes (four
// lanes of one cell at one node take five times as long).
//
// Rows take fewer instructions (8 cases FP64, 671 thousand points: 22.6
// us a substep, 25.0 in order; 1.6 million points FP64: 50 and 51), but
// add the terms in another order.  FP64 points differ by rounding then; the
// rounding of FP32 storage and the yield branches carry a study's points past 1e-5
// of the other order's within 4000 substeps in most runs, where two runs of one
// order mostly agree to the bit.  Chunks of 64 points are kept in order: in one row
// their cells' points are neighbours anyway (32 cases, 6.98 million points: 242 us,
// 480 with an LDS atomic for each of a point's 27 sums).  So are those of clouds
// with more than kDensePoints a cell, of which a row holds several a cell.  us a
// substep of 960 thousand points FP64 in rows and in order: 26.9 and 29.2 at 4 a
// cell, 39.0 and 41.3 at 5.5, 40.8 and 39.7 at 6, 53 and 35 at 9, 75 and 32 at 16,
// 123 and 30 at 49 (the grid update and pass before: 41, 42, 41, 39, 37 and 37).
constexpr double kDensePoints = 5.75;
static __host__ __device__ inline unsigned chunk_shape(int n) {
    const int rows = (n + 63) / 64;
    return (unsigned)(n / rows) | (unsigned)(n % rows) << 8 | (unsigned)rows << 16;
}
static __host__ __device__ inline int chunk_count(unsigned shape) {
    return (int)((shape & 0xFFu) * (shape >> 16) + (shape >> 8 & 0xFFu));
}
static __host__ __device__ inline int chunk_point(int slot, unsigned shape) {
    const int lanes = (int)(shape & 0xFFu), more = (int)(shape >> 8 & 0xFFu), rows = (int)(shape >> 16);
    const int wide = more * (lanes + 1);   // slots of the rows with one lane more
    const int row = slot < wide ? slot / (lanes + 1) : more + (slot - wide) / lanes;
    return rows * (slot - row * lanes - (row < more ? row : more)) + row;
}

// LDS of a workgroup: the windows of its P2G (three sums per node), the tile of
// node velocities its G2P reads, and a patch per wavefront for the velocities of
// kPatch points outside the box.  64 points in band order, four to a cell, touch
// 10 x 4 nodes and 256 points 34 x 4; the space (25.6 KB with a window per
// wavefront, 19.6 KB with one) holds more rows, for points that have moved out
// of their band.  Workgroups of one or two wavefronts, for chunks of at most 64
// or 128 points, have room for the box of a chunk's two rows and no more, so that
// as many wavefronts fit a CU.
constexpr int kWaveWin = 160;            // of a wavefront's window (FP32): nodes x row stride
constexpr int box_space(int waves) { return waves == 4 ? 384 : 240; }   // of the tile, and of the window (FP64)
constexpr int kWinCols = 40;
constexpr int kPatch = 7;                // x 9 nodes: one load round of a wavefront
constexpr int kChunkCols = 58;           // base cells a chunk may span: 60 columns of nodes
static_assert(4 * (kChunkCols + 2) <= box_space(1), "the box of two rows of cells fits");

// The row stride of a wavefront's window: rows next to each other lie on
// different LDS banks (a row of S doubles shifts them by 2 S of 64).
static __device__ __forceinline__ int win_stride(int w) { return w <= 16 ? 20 : (w <= 32 ? 36 : kWinCols); }

// The box of the base cells [x0, x1] x [y0, y1] as a record's org, ext and
// inv; false if it does not fit the space (of box_space).  A tile row of T 16-byte entries, T
// = 8 mod 16, and a window row of S doubles, S = 16 mod 32, put the two cell
// rows of a band on different LDS banks; a taller box packs its rows.
static __device__ __forceinline__ bool set_box(ChunkRec &r, int x0, int y0, int x1, int y1, int space) {
    const int w = x1 + 3 - x0, h = y1 + 3 - y0;
    if (w > 128 || h > 128 || w * h > space) return false;
    int T = ((w + 7) >> 4) * 16 + 8, S = ((w + 15) >> 5) * 32 + 16;
    if (T * h > space) T = w;
    if (S * h > space) S = w;
    r.org = (unsigned)x0 | (unsigned)y0 << 16;
    r.ext = (unsigned)w | (unsigned)h << 8 | (unsigned)T << 16 | (unsigned)S << 24;
    r.inv = 65535u / (unsigned)w + 1u;
    return true;
}
// A wavefront's window in that box: the stencils of the base cells
// [x0, x1] x [y0, y1] of its points, as far as they lie in the box and the
// window has room.
static __device__ __forceinline__ unsigned win_of(const ChunkRec &r, int x0, int y0, int x1, int y1) {
    const int ox = (int)(r.org & 0xFFFFu), oy = (int)(r.org >> 16);
    x0 = max(x0 - ox, 0);
    y0 = max(y0 - oy, 0);
    const int w = min(min(x1 - ox + 3, (int)(r.ext & 0xFFu)) - x0, kWinCols);
    const int h = min(min(y1 - oy + 3, (int)(r.ext >> 8 & 0xFFu)) - y0, kWaveWin / win_stride(w));
    return w < 3 || h < 3 ? 0u : (unsigned)x0 | (unsigned)y0 << 8 | (unsigned)w << 16 | (unsigned)h << 24;
}

// The velocity a node has after the grid update (gpu_implementation5.cu:
// 215-290) from its mass (not zero) and momentum: gravity, the speed limit,
// the indenter's contact, the walls.  Returns whether the indenter touches
// it; d is then the velocity the contact takes from it and n the unit normal.
// 1/m comes from rcp_nr.
static __device__ __forceinline__ bool node_velocity(const CaseParams &cp, double ind_x, double mass, double p0,
                                                     double p1, int ix, int iy, double &v0, double &v1, double &d0,
                                                     double &d1, double &n0, double &n1) {
    const double rm = rcp_nr(mass);
    v0 = p0 * rm;
    v1 = p1 * rm;
    v1 = v1 - cp.dt * cp.gravity;
    const double vsq = v0 * v0 + v1 * v1;
    if (vsq > cp.vmax * cp.vmax) {
        const double s = cp.vmax / sqrt(vsq);
        v0 = v0 * s;
        v1 = v1 * s;
    }
    bool hit = false;
    n0 = ix * cp.h - ind_x;
    n1 = iy * cp.h - cp.y0;
    const double z = n0 * n0 + n1 * n1;
    if (z < cp.indRsq) {
        const double V = cp.indV, r0 = v0 - V, r1 = v1;
        if (z > 0) {
            const double nz = sqrt(z);
            n0 = n0 / nz;
            n1 = n1 / nz;
        }
        const double vnr = r0 * n0 + r1 * n1;
        if (vnr < 0) {
            d0 = v0;
            d1 = v1;
            v0 = V + (r0 - n0 * vnr);
            v1 = r1 - n1 * vnr;
            d0 -= v0;
            d1 -= v1;
            hit = true;
        }
    }
    if (iy <= 2) {
        v0 = 0;
        v1 = 0;
    } else if (iy >= cp.gy - 3 && v1 > 0) {
        v1 = 0;
    }
    if (ix <= 2 && v0 < 0)
        v0 = 0;
    else if (ix >= cp.gx - 3 && v0 > 0)
        v0 = 0;
    return hit;
}

// The grid side of a substep: the workgroups after the particle ones each
// take kNodeBlk nodes of one case.  They clear the grid that the next
// substep scatters into and add up the indenter's force; nothing else of the
// grid update is left to them, since every workgroup makes the velocities of
// its own box.  bounds holds, per case, the box of all nodes that the P2G has
// ever touched since the run's fresh start (columns and rows of the least and
// greatest, widened by the passes): outside it (and a border of one) the
// grids are still zero.
constexpr int kNodeBlk = 1024;
struct NodeWork {
    const int2 *blocks;   // {case, first node} per workgroup (null: one case's, in order)
    double *clear;        // the grid to clear
    double *hist;         // this substep's force, 2 per case
    double *bins;
};

template <int kWaves>
static __device__ __forceinline__ void node_part(const NodeWork &nw, int block, const CaseParams *__restrict__ cases,
                                                 const double *__restrict__ grid, size_t gpitch, const int4 *bounds,
                                                 double t, double *lds) {
    constexpr int kParts = 4 / kWaves, kNodes = kNodeBlk / kParts;   // smaller workgroups take a part of a block
    int2 nb = nw.blocks ? nw.blocks[block / kParts] : make_int2(0, block / kParts * kNodeBlk);
    if constexpr (kParts > 1) nb.y += block % kParts * kNodes;
    const CaseParams &cp = cases[nb.x];
    const int4 bd = bounds[nb.x];
    const int x0 = bd.x - 1, y0 = bd.y - 1, x1 = bd.z + 1, y1 = bd.w + 1;
    // rows of the block: (node + 0.5) / gx lies >= 0.5 / gx >= 2^-17 from an
    // integer and is computed to within 2^-23, so its floor is the row
    const int first = (int)(((double)nb.y + 0.5) * cp.gxInv);
    const int last = (int)(((double)min(nb.y + kNodes, cp.gridTotal) - 0.5) * cp.gxInv);
    if ((kParts > 1 && nb.y >= cp.gridTotal) || bd.z < 0 || last < y0 || first > y1) return;   // uniform: nothing was ever touched here
    if (threadIdx.x < 3) lds[threadIdx.x] = 0;
    __syncthreads();
    const double ind_x = cp.x0 + t * cp.indV;
#pragma unroll
    for (int q = 0; q < kNodes; q += 64 * kWaves) {
        const int local = nb.y + q + (int)threadIdx.x;
        const int iy = (int)(((double)local + 0.5) * cp.gxInv), ix = local - iy * cp.gx;
        if (local >= cp.gridTotal || ix < x0 || ix > x1 || iy < y0 || iy > y1) continue;
        const size_t idx = (size_t)cp.gridOffset + local;
        nw.clear[idx] = 0;
        nw.clear[gpitch + idx] = 0;
        nw.clear[2 * gpitch + idx] = 0;
        const double c0 = ix * cp.h - ind_x, c1 = iy * cp.h - cp.y0;
        if (c0 * c0 + c1 * c1 < cp.indRsq) {
            const double mass = grid[idx];
            if (mass != 0) {
                double v0, v1, d0, d1, n0, n1;
                if (node_velocity(cp, ind_x, mass, grid[gpitch + idx], grid[2 * gpitch + idx], ix, iy, v0, v1, d0, d1,
                                  n0, n1)) {
                    const double f0 = d0 * mass / cp.dt, f1 = d1 * mass / cp.dt;
                    atomicAdd(&lds[0], f0);
                    atomicAdd(&lds[1], f1);
                    lds[2] = 1;
                    // the force's angular bin (gpu_implementation5.cu:262-269:
                    // atan2 of (x, y) of the unit normal, then + pi, scaled)
                    double angle = atan2(n0, n1);
                    angle += kPi;
                    angle *= cp.nbins / (2 * kPi);
                    int kb = (int)angle;
                    kb = max(kb, 0);
                    kb = min(kb, cp.nbins - 1);
                    unsafeAtomicAdd(&nw.bins[cp.binOffset + 2 * kb], f0);
                    unsafeAtomicAdd(&nw.bins[cp.binOffset + 2 * kb + 1], f1);
                }
            }
        }
    }
    __syncthreads();
    if (threadIdx.x == 0 && lds[2] != 0) {
        unsafeAtomicAdd(&nw.hist[2 * nb.x], lds[0]);
        unsafeAtomicAdd(&nw.hist[2 * nb.x + 1], lds[1]);
    }
}

// Node e of a box of the given width: its column and row.
static __device__ __forceinline__ void box_node(unsigned e, unsigned inv, unsigned w, unsigned &col, unsigned &row) {
    row = e * inv >> 16;
    col = e - row * w;
}

// Widens a case's box of touched nodes to the stencils of base cells
// [x0, x1] x [y0, y1].  Mostly it holds them already: the atomics of every
// workgroup on the few cases' boxes would take longer than the substep.
static __device__ __forceinline__ void widen_bounds(int4 *bounds, int cs, int x0, int y0, int x1, int y1) {
    int *b = reinterpret_cast<int *>(&bounds[cs]);
    const auto get = [&](int i) { return __hip_atomic_load(b + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
    if (x0 >= get(0) && y0 >= get(1) && x1 + 2 <= get(2) && y1 + 2 <= get(3)) return;
    atomicMin(b, x0);
    atomicMin(b + 1, y0);
    atomicMax(b + 2, x1 + 2);
    atomicMax(b + 3, y1 + 2);
}

// Quad-level P2G.  A DPP read of a double from another lane of the quad
// (quad_perm control CTRL; every lane of the quad must be active, so no
// lane keeps an old value and none is needed)
template <int CTRL>
static __device__ __forceinline__ double quad_dpp(double v) {
    const long long b = __builtin_bit_cast(long long, v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, true);
    return __builtin_bit_cast(double, (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
constexpr int kQuadXor1 = 0xB1, kQuadXor2 = 0x4E, kQuadXor3 = 0x1B;   // quad_perm 1032, 2301, 3210
// whether the four lanes of this lane's quad hold the same key (all lanes
// of the wavefront active)
static __device__ __forceinline__ bool quad_uniform(unsigned key) {
    const int k = (int)key;
    return k == __builtin_amdgcn_mov_dpp(k, kQuadXor1, 0xF, 0xF, true) &&
           k == __builtin_amdgcn_mov_dpp(k, kQuadXor2, 0xF, 0xF, true) &&
           k == __builtin_amdgcn_mov_dpp(k, kQuadXor3, 0xF, 0xF, true);
}
// One component's ten node values of a quad lane (step 1 layout, below)
// summed over the quad and added to the window row Wc.
static __device__ __forceinline__ void quad_component(int lane, const double (&K)[5], const double (&D)[4], int eA,
                                                      int eB, int eC, double *Wc) {
    const int sy = (lane >> 1) & 1;
    double k[5];
#pragma unroll
    for (int s = 0; s < 4; ++s) k[s] = K[s] + quad_dpp<kQuadXor1>(D[s]);
    k[4] = K[4] + quad_dpp<kQuadXor1>(K[4]);
    // step 2: the partners across bit 1 split slots (0, 1) and (2, 3)
    const double x01 = sy ? k[0] : k[1], y01 = sy ? k[1] : k[0];
    const double x23 = sy ? k[2] : k[3], y23 = sy ? k[3] : k[2];
    atomicAdd(&Wc[eA], y01 + quad_dpp<kQuadXor2>(x01));
    atomicAdd(&Wc[eB], y23 + quad_dpp<kQuadXor2>(x23));
    const double k4 = k[4] + quad_dpp<kQuadXor2>(k[4]);
    if ((lane & 3) == 0) atomicAdd(&Wc[eC], k4);
}
// The P2G of a quad whose four points share their base cell, into the
// window (e0: the base's element): node (i, j) of the stencil gets
// W (v + A d), W = wx_i wy_j, d = ((i, j) - f) h, summed over the four
// points.  Step 1 pairs lanes across lane bit 0 (sx): slot s < 3 holds node
// (2 sx, s), kept, and (2 - 2 sx, s), sent to the partner; slot 3 node
// (1, sx), kept, and (1, 1 - sx), sent; slot 4 node (1, 2) on both.  After
// it a lane holds pair sums of five (sx = 0) or four (sx = 1) nodes.  Step 2
// pairs lanes across bit 1 (sy): of slots 0 and 1 the lane keeps slot sy,
// of slots 2 and 3 slot 2 + sy, and lane 0 of the quad keeps slot 4.  Each
// lane then adds two or three of the nine node sums per row: 6-9 LDS
// atomics instead of 27, the nodes of one instruction still distinct
// within the quad.
static __device__ __forceinline__ void quad_scatter(int lane, int e0, int S, double h, double fx0, double fx1, double wx0,
                                                    double wx1, double wx2, double wy0, double wy1, double wy2,
                                                    double vx, double vy, double A00, double A01, double A10,
                                                    double A11, double *W0, double *W1, double *W2) {
    const int sx = lane & 1, sy = (lane >> 1) & 1;
    const double dx0 = (0.0 - fx0) * h, dx1 = (1.0 - fx0) * h, dx2 = (2.0 - fx0) * h;
    const double dy0 = (0.0 - fx1) * h, dy1 = (1.0 - fx1) * h, dy2 = (2.0 - fx1) * h;
    const double xa0 = vx + A00 * dx0, xa1 = vx + A00 * dx1, xa2 = vx + A00 * dx2;
    const double xb0 = vy + A10 * dx0, xb1 = vy + A10 * dx1, xb2 = vy + A10 * dx2;
    const double ya0 = A01 * dy0, ya1 = A01 * dy1, ya2 = A01 * dy2;
    const double yb0 = A11 * dy0, yb1 = A11 * dy1, yb2 = A11 * dy2;
    // the kept and sent columns of slots 0-2, and the kept and sent rows of slot 3
    const double wxK = sx ? wx2 : wx0, xaK = sx ? xa2 : xa0, xbK = sx ? xb2 : xb0;
    const double wxD = sx ? wx0 : wx2, xaD = sx ? xa0 : xa2, xbD = sx ? xb0 : xb2;
    const double wyK = sx ? wy1 : wy0, yaK = sx ? ya1 : ya0, ybK = sx ? yb1 : yb0;
    const double wyD = sx ? wy0 : wy1, yaD = sx ? ya0 : ya1, ybD = sx ? yb0 : yb1;
    const double wy[3] = {wy0, wy1, wy2}, ya[3] = {ya0, ya1, ya2}, yb[3] = {yb0, yb1, yb2};
    double WK[5], WD[4];
#pragma unroll
    for (int s = 0; s < 3; ++s) {
        WK[s] = wxK * wy[s];
        WD[s] = wxD * wy[s];
    }
    WK[3] = wx1 * wyK;
    WD[3] = wx1 * wyD;
    WK[4] = wx1 * wy2;
    // the nodes a lane adds: slot sy's node (2 sx, sy); slot 2 + sy's node,
    // (2 sx, 2) or (1, sx); slot 4's node (1, 2)
    const int eA = e0 + 2 * sx + sy * S;
    const int eB = e0 + (sy ? 1 + sx * S : 2 * sx + 2 * S);
    const int eC = e0 + 1 + 2 * S;
    quad_component(lane, WK, WD, eA, eB, eC, W0);
    double K[5], D[4];
#pragma unroll
    for (int s = 0; s < 3; ++s) {
        K[s] = WK[s] * (xaK + ya[s]);
        D[s] = WD[s] * (xaD + ya[s]);
    }
    K[3] = WK[3] * (xa1 + yaK);
    D[3] = WD[3] * (xa1 + yaD);
    K[4] = WK[4] * (xa1 + ya2);
    quad_component(lane, K, D, eA, eB, eC, W1);
#pragma unroll
    for (int s = 0; s < 3; ++s) {
        K[s] = WK[s] * (xbK + yb[s]);
        D[s] = WD[s] * (xbD + yb[s]);
    }
    K[3] = WK[3] * (xb1 + ybK);
    D[3] = WD[3] * (xb1 + ybD);
    K[4] = WK[4] * (xb1 + yb2);
    quad_component(lane, K, D, eA, eB, eC, W2);
}


// One substep over all cases: grid update, G2P of this substep and P2G of
// the next (G2P false: a run's first P2G alone).  gridIn holds the masses and
// momenta of the last P2G; every workgroup turns the nodes of its box into
// velocities in LDS (a node a thread), its wavefronts gather from there, move
// their points, sum their contributions in a window of their own and add it to
// gridOut with one atomic per node and component; the workgroups from pGroups
// on do the rest of the grid update (node_part).
//
// What bounds it: at 7 million points in FP32 storage the memory (647 MB a
// substep, 131 us at a copy's rate, of which 123 to 194 MB are atomic requests of
// 64 bytes) and the vector units (660 instructions per 64 points, half of them
// FP64 at 4 cycles each, 108 us), which overlap in part; below ~100 thousand
// points the launch and one chain of memory latencies (3.9 us).  Against a grid
// update of its own and a particle pass that gathered from global memory and
// found each wavefront's window anew, a substep of 32 cases / 6.98 million points
// went from 193 to 168 us (FP32 storage, points in mid-run; of cases at rest in
// their load order both take 165 to 179), of 12 cases / 81 thousand points from
// 18.4 to 8.2, of 8 cases / 671 thousand points from 35 to 21 (FP64, strengths
// per grain).  Making a node's velocity in each of the ~2 workgroups that need it
// costs ~50 instructions per 64 points; it saves a launch, the velocities' trip
// through memory and the gathers' 6 to 18 loads a point.  Four or five wavefronts
// per SIMD are equally fast, six (80 registers) slower.  The grid's workgroups
// come last: spread among the others their writes slow these down (1.6 million
// points FP64 47 us against 44).
//
// The records, the grid and the point rows lead the arguments, which the
// kernel receives preloaded in SGPRs.
//
// tAt: where a batch has the substep's time (its runs are captured); null: t0.
// step: the box is renewed where it is a multiple of kBoxEvery.
//
// kWaves: wavefronts of a workgroup, for chunks of at most 64 kWaves points.  Fewer
// than four only where a caller asks for smaller chunks.  us a substep in chunks of
// 256, 128 and 64: 32 cases / 6.98 million points 178, 178 and 189 (FP32), 210, 224
// and 242 (FP64); 12 cases / 81 thousand points 8.2, 8.1 and 9.4, 7.5, 8.1 and 8.4.
// With four wavefronts for all of them 176, 233 and 356, 212, 287 and 486; 8.1, 8.1
// and 10.5, 7.5, 8.2 and 13.
template <bool F32, bool G2P, int RMAP, int kWaves, bool kInOrder>
__global__ __launch_bounds__(64 * kWaves, kWaves == 1 ? 4 : 5) void k_batch_substep(
    ChunkRec *__restrict__ recs, const double *__restrict__ gridIn, int nChunks, int pGroups,
    typename Rows<F32>::P *pos, typename Rows<F32>::V *rest, size_t gpitch, const CaseParams *__restrict__ cases,
    unsigned char *crushedRow, size_t pitch, double *__restrict__ gridOut, int4 *bounds, int *__restrict__ err,
    const short *__restrict__ grains, typename Rows<F32>::V *jpRow, const double *__restrict__ tAt, double t0, int step,
    NodeWork nw, LearnArgs la, MapQueue mq, int storeVB, int joint) {
    static_assert(kInOrder || (!F32 && kWaves == 4), "rows are FP64 storage's, four to a workgroup");
    using M = typename std::conditional<RMAP == kMapSingle, FusedMath, PlainMath>::type;
    constexpr int kWin = box_space(kWaves), kTile = kWin;
    constexpr int kWindows = 3 * (F32 ? kWaves * kWaveWin : kWin);   // doubles
    __shared__ __attribute__((aligned(16))) double smem[kWindows + 2 * kTile + kWaves * (2 * 9 + 1) * kPatch];
    if constexpr (G2P) {
        if ((int)blockIdx.x >= pGroups) {
            node_part<kWaves>(nw, (int)blockIdx.x - pGroups, cases, gridIn, gpitch, bounds, tAt ? *tAt : t0, smem);
            return;
        }
    }
    const Rows<F32> S{pos, rest, crushedRow, nullptr, pitch};
    // neighbouring chunks on one XCD (workgroups go round the 8 XCDs)
    const int chunk = (blockIdx.x & 7) * (pGroups >> 3) + (blockIdx.x >> 3);
    if (chunk >= nChunks) return;
    const int lane = threadIdx.x & 63, row = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const ChunkRec rec = recs[chunk];
    // FP32 storage: a wavefront issues its loads, and later its window flush,
    // at raised priority, computes at the base one (measured: -2.6% per
    // substep; FP64 storage measured slower with it)
    if constexpr (F32) __builtin_amdgcn_s_setprio(2);
    const CaseParams &cp = cases[rec.cs];
    const KParams k = kp_of(cp, err);
    const size_t pp = S.pitch;
    const int gx = (int)(rec.dims & 0xFFFFu), gy = (int)(rec.dims >> 16);
    const double *__restrict__ gI = gridIn + rec.gofs;
    double *__restrict__ gO = gridOut + rec.gofs;
    using V = typename Rows<F32>::V;
    V *__restrict__ R = S.rest;
    constexpr double fe0 = F32 ? 1.0 : 0.0;   // stored Fe = Fe - fe0 * I, Jp_inv - fe0
    // the wavefront's points: lanes of them (none past the last one)
    int lanes, first;
    if constexpr (kInOrder) {
        lanes = (int)rec.shape - row * 64;
        first = row * 64;
    } else {
        const int lanesRow = (int)(rec.shape & 0xFFu), more = (int)(rec.shape >> 8 & 0xFFu);
        lanes = row < (int)(rec.shape >> 16) ? lanesRow + (row < more ? 1 : 0) : 0;
        first = row * lanesRow + min(row, more);
    }
    const bool valid = lane < lanes;
    const int pt = rec.beg + first + lane;
    const unsigned u = (unsigned)pt;
    // the box with the tile
    const int ox = (int)(rec.org & 0xFFFFu), oy = (int)(rec.org >> 16);
    const int bw = (int)(rec.ext & 0xFFu), bh = (int)(rec.ext >> 8 & 0xFFu), tS = (int)(rec.ext >> 16 & 0xFFu);
    const unsigned nodes = (unsigned)(bw * bh);
    // base cells whose stencil lies in the box and in the grid: [ox, ox + fw) x [oy, oy + fh)
    const unsigned fw = (unsigned)max(min(bw, gx - ox) - 2, 0), fh = (unsigned)max(min(bh, gy - oy) - 2, 0);
    // the window: FP64 storage, the box; FP32, the wavefront's part of it
    int wx = ox, wy = oy, ww = bw, wh = bh, wS = (int)(rec.ext >> 24);
    unsigned ww2 = fw, wh2 = fh;
    double *W0 = smem;
    constexpr int kWinSize = F32 ? kWaveWin : kWin;
    if constexpr (F32) {
        const unsigned win = recs[chunk].win[row];
        wx += (int)(win & 0xFFu);
        wy += (int)(win >> 8 & 0xFFu);
        ww = (int)(win >> 16 & 0xFFu);
        wh = (int)(win >> 24);
        wS = win_stride(ww);
        ww2 = (unsigned)max(min(ww, gx - wx) - 2, 0);
        wh2 = (unsigned)max(min(wh, gy - wy) - 2, 0);
        W0 += row * 3 * kWaveWin;
    }
    double *W1 = W0 + kWinSize, *W2 = W1 + kWinSize;
    // lanes map onto a wavefront's window 16, 32 or 64 columns at a time
    const int wsh = ww <= 16 ? 4 : (ww <= 32 ? 5 : 6);
    const int wcol = lane & ((1 << wsh) - 1), wrow0 = lane >> wsh, wstep = 64 >> wsh;
    double2 *tile = reinterpret_cast<double2 *>(smem + kWindows);
    const double ind_x = cp.x0 + (G2P ? (tAt ? *tAt : t0) : 0.0) * cp.indV;

    // The state of the points, read once per substep.  FP32 records
    // non-temporally, so the grid keeps the L2 (167 us for 6.98 million points,
    // 178 without); FP64 rows, whose wavefronts' 512 B straddle cache lines that
    // the neighbours complete, through it (1.6 million points 44 us, 50
    // non-temporally).  A lane without a point reads the chunk's first one and
    // computes along with the others; only its stores and sums are left out.
    prec4 pr;
    fe4 fr;
    double px, py, F00, F01, F10, F11;
    unsigned char crushed = 0;
    short grain = 0;
    const unsigned us = valid ? u : (unsigned)rec.beg;
    if constexpr (F32) {
        pr = __builtin_nontemporal_load(reinterpret_cast<const prec4 *>(S.pos) + us);
        fr = __builtin_nontemporal_load(fe_rec(R, pp) + us);
    } else {
        pos_load(S.pos, pp, (int)us, cp, px, py);
        F00 = (*at(R + pp * 2, us));
        F01 = (*at(R + pp * 3, us));
        F10 = (*at(R + pp * 4, us));
        F11 = (*at(R + pp * 5, us));
        crushed = (*at(S.crushed, us));
        if (cp.grainVar != 0) grain = (*at(grains, us));
    }

    if constexpr (F32) {
        if (wcol < ww) {
            for (int r = wrow0; r < wh; r += wstep) {
                const int e = r * wS + wcol;
                W0[e] = 0;
                W1[e] = 0;
                W2[e] = 0;
            }
        }
    }
    // the box's velocities (FP32 storage rounds them to FP32)
    if constexpr (G2P || !F32) {
        for (unsigned e = threadIdx.x; e < nodes; e += 64 * kWaves) {
            unsigned c, r;
            box_node(e, rec.inv, (unsigned)bw, c, r);
            if constexpr (!F32) {
                const unsigned w = r * (unsigned)wS + c;
                W0[w] = 0;
                W1[w] = 0;
                W2[w] = 0;
            }
            if constexpr (!G2P) continue;
            const int X = ox + (int)c, Y = oy + (int)r;
            const bool in = X < gx && Y < gy;
            const unsigned node = in ? (unsigned)(X + Y * gx) : 0u;
            const double mass = *at(gI, node), m0 = *at(gI + gpitch, node), m1 = *at(gI + 2 * gpitch, node);
            double n0, n1, e0, e1, e2, e3;
            node_velocity(cp, ind_x, mass, m0, m1, X, Y, n0, n1, e0, e1, e2, e3);
            if constexpr (F32) {
                n0 = (double)(float)n0;
                n1 = (double)(float)n1;
            }
            const bool moves = in && mass != 0;   // a node without mass has no velocity
            tile[r * (unsigned)tS + c] = make_double2(moves ? n0 : 0.0, moves ? n1 : 0.0);
        }
    }
    if constexpr (F32) __builtin_amdgcn_s_setprio(0);
    if constexpr (G2P || !F32) __syncthreads();

    // the base cells of the points, for the box (when it is renewed)
    int cellx = -1, celly = -1;
    if (lanes > 0) {
        double vx, vy;
        double B00, B01, B10, B11;   // Bp
        double t00, t01, t11;        // the Kirchhoff stress
        bool defer = false;          // learned map: projection and P2G done by the map kernel
        if constexpr (G2P) {
            double Jp = 1;
            if constexpr (F32) {   // the record's coordinates in cell units
                px = fix_cells(pr.x, pr.z & 0xFFFFu, cp);
                py = fix_cells(pr.y, pr.z >> 16, cp);
                crushed = (unsigned char)(pr.w & 0xFFu);
                grain = (short)(pr.w >> 16);
                F00 = fe0 + (double)fr.x;
                F01 = (double)fr.y;
                F10 = (double)fr.z;
                F11 = fe0 + (double)fr.w;
            }
            int bx = 0, by = 0;
            double fx0 = 0, fx1 = 0, wx0 = 0, wx1 = 0, wx2 = 0, wy0 = 0, wy1 = 0, wy2 = 0;
            bool ok = valid;
            if constexpr (F32) {   // a record always has a stencil
                stencil_cells(px, bx, fx0, wx0, wx1, wx2);
                stencil_cells(py, by, fx1, wy0, wy1, wy2);
            } else {
                const bool st = M::stencil(px, cp.h_inv, bx, fx0, wx0, wx1, wx2) &&
                                M::stencil(py, cp.h_inv, by, fx1, wy0, wy1, wy2);
                ok = valid && st;
                if (valid && !st) flag_error(k);
            }
            // the node velocities: in the tile, or for a point outside the box
            // in the wavefront's patch, where 9 lanes a point put them
            const int lx0 = bx - ox, ly0 = by - oy;
            const bool inTile = (unsigned)lx0 < fw && (unsigned)ly0 < fh;
            const double2 *line = tile + (inTile ? ly0 * tS + lx0 : 0);
            int ls = tS;
            bool slow = ok && !inTile;
            if (const unsigned long long om = __ballot(slow)) {
                double2 *patch = tile + kTile + row * 9 * kPatch;
                int2 *cells = reinterpret_cast<int2 *>(tile + kTile + kWaves * 9 * kPatch) + row * kPatch;
                const int rank = __popcll(om & ((1ull << lane) - 1ull));
                if (slow && rank < kPatch) cells[rank] = make_int2(bx, by);
                wsync();
                const int e = lane, o = e / 9, n = e - 9 * o;
                if (e < 9 * min(__popcll(om), kPatch)) {
                    const int2 cell = cells[o];
                    const int X = cell.x + n % 3, Y = cell.y + n / 3;
                    double n0 = 0, n1 = 0;
                    if (X >= gx || Y >= gy) {
                        flag_error(k);
                    } else {
                        const unsigned node = (unsigned)(X + Y * gx);
                        const double mass = *at(gI, node), m0 = *at(gI + gpitch, node), m1 = *at(gI + 2 * gpitch, node);
                        double e0, e1, e2, e3;
                        if (mass != 0) node_velocity(cp, ind_x, mass, m0, m1, X, Y, n0, n1, e0, e1, e2, e3);
                    }
                    if constexpr (F32) {
                        n0 = (double)(float)n0;
                        n1 = (double)(float)n1;
                    }
                    patch[e] = make_double2(n0, n1);
                }
                wsync();
                if (slow && rank < kPatch) {
                    line = patch + 9 * rank;
                    ls = 3;
                    slow = false;
                }
            }
            double v0 = 0, v1 = 0, b00 = 0, b01 = 0, b10 = 0, b11 = 0;   // v and Bp
            const double c4 = 4. * cp.h_inv;
            {
                const double wyd0 = wy0 * (0 - fx1), wyd1 = wy1 * (1 - fx1), wyd2 = wy2 * (2 - fx1);
                const double wxs[3] = {wx0, wx1, wx2};
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    const double2 a = line[i], b = line[ls + i], c = line[2 * ls + i];
                    const double s0 = wy0 * a.x + wy1 * b.x + wy2 * c.x;
                    const double s1 = wy0 * a.y + wy1 * b.y + wy2 * c.y;
                    const double t0 = wyd0 * a.x + wyd1 * b.x + wyd2 * c.x;
                    const double t1 = wyd0 * a.y + wyd1 * b.y + wyd2 * c.y;
                    const double wxd = wxs[i] * (i - fx0);
                    v0 += wxs[i] * s0;
                    v1 += wxs[i] * s1;
                    b00 += wxd * s0;
                    b10 += wxd * s1;
                    b01 += wxs[i] * t0;
                    b11 += wxs[i] * t1;
                }
            }
            if (slow) {
                // more points outside the box than the patch holds: node by node
                v0 = v1 = b00 = b01 = b10 = b11 = 0;
#pragma unroll 1
                for (int e = 0; e < 9; ++e) {
                    const int i = e % 3, j = e / 3, X = bx + i, Y = by + j;
                    if (X >= gx || Y >= gy) {
                        flag_error(k);
                        continue;
                    }
                    const unsigned node = (unsigned)(X + Y * gx);
                    const double mass = *at(gI, node);
                    if (mass == 0) continue;
                    double n0, n1, e0, e1, e2, e3;
                    node_velocity(cp, ind_x, mass, *at(gI + gpitch, node), *at(gI + 2 * gpitch, node), X, Y, n0, n1,
                                  e0, e1, e2, e3);
                    if constexpr (F32) {
                        n0 = (double)(float)n0;
                        n1 = (double)(float)n1;
                    }
                    const double w = sel3(i, wx0, wx1, wx2) * sel3(j, wy0, wy1, wy2);
                    v0 += w * n0;
                    v1 += w * n1;
                    b00 += w * n0 * (i - fx0);
                    b01 += w * n0 * (j - fx1);
                    b10 += w * n1 * (i - fx0);
                    b11 += w * n1 * (j - fx1);
                }
            }
            b00 *= c4; b01 *= c4; b10 *= c4; b11 *= c4;
            B00 = b00; B01 = b01; B10 = b10; B11 = b11;
            const double dt = cp.dt;
            const double dtp = F32 ? cp.dtCells : dt;   // FP32 storage: cell units
            px += v0 * dtp;
            py += v1 * dtp;
            const double M00 = 1.0 + dt * b00, M01 = dt * b01, M10 = dt * b10, M11 = 1.0 + dt * b11;
            const double n00 = M00 * F00 + M01 * F10, n01 = M00 * F01 + M01 * F11;
            const double n10 = M10 * F00 + M11 * F10, n11 = M10 * F01 + M11 * F11;
            F00 = n00; F01 = n01; F10 = n10; F11 = n11;
            vx = v0; vy = v1;
            // p and q^2 of the trial state (q itself is never needed here:
            // every test compares it with a non-negative limit)
            const InvSq iv = M::invariants_sq(F00, F01, F10, F11, cp.mu, cp.kappa);
            const unsigned char crushed0 = crushed;
            if (cp.grainVar != 0) {   // GetParametersForGrain's strengths (case-uniform branch)
                if (crushed == 0) crushed = M::fails_sq(k, grain, iv.p, iv.q2) ? 1 : 0;
            } else {
                // tension line q > slope (p + 3e6), slope >= 0 and p + 3e6 >= 0 there
                const double ql = cp.slope * (iv.p - -3e6);
                const bool ft = (iv.p < -3e6) || (iv.q2 > ql * ql);
                const bool fc = cp.onePlus2Beta * iv.q2 + cp.msq * (iv.p + cp.betaPmax) * (iv.p - cp.pmax) > 0;
                if (crushed == 0 && (iv.p < 0 ? ft : fc)) crushed = 1;
            }
            // ---- return map (convergent: the learned map runs wavefront-wide) ----
            // The trial SVD only for crushed points (few: the wavefront mostly
            // skips it); p and q for the NACC test came from the invariants.
            // Jp_inv matters only to the map, so only crushed points load it.
            const bool crushedOk = ok && crushed == 1;
            if (crushedOk) Jp = fe0 + (double)*at(jpRow, u);
            const double Jp0 = Jp;
            if constexpr (RMAP == kMapExact || RMAP == kMapSingle) {
                if (crushedOk && M::dp_projects_sq(k, iv.p, iv.q2, Jp))
                    M::dp_return(k, M::compute_pq_fast(F00, F01, F10, F11, cp.mu, cp.kappa), F00, F01, F10, F11, Jp);
            } else if constexpr (RMAP == kMapHarvest) {
                Trial r{};
                if (crushedOk) r = compute_pq_fast(F00, F01, F10, F11, cp.mu, cp.kappa);
                double f[5] = {0, 0, 0, 0, 0}, t[3] = {0, 0, 0};
                bool usable = false;
                if (crushedOk) {
                    double qlim;
                    const int br = map_branch(k, r, Jp, qlim);
                    map_features(r, Jp, br, f);
                    dp_return(k, r, F00, F01, F10, F11, Jp);
                    if (br != kBrInside) {
                        const Trial rn = compute_pq(F00, F01, F10, F11, cp.mu, cp.kappa);
                        usable = r.svd.s1 > 0 && rn.svd.s1 > 0;
                        t[0] = log(rn.svd.s0) - f[0];
                        t[1] = log(rn.svd.s1) - f[1];
                        t[2] = log(Jp) - f[2];
                    }
                }
                // one counter update per wavefront
                const unsigned long long um = __ballot(usable);
                if (um) {
                    unsigned long long base = 0;
                    if (lane == 0) base = atomicAdd(la.hcount, (unsigned long long)__popcll(um));
                    base = __shfl(base, 0, 64);
                    const unsigned long long slot = base + (unsigned long long)__popcll(um & ((1ull << lane) - 1ull));
                    if (usable && slot < (unsigned long long)la.hcap) {
                        for (int q = 0; q < 5; ++q) la.hx[slot * 5 + q] = (float)f[q];
                        for (int q = 0; q < 3; ++q) la.ht[slot * 3 + q] = (float)t[q];
                    }
                }
            } else {
                // the branch is decided exactly; inside the surface the map is
                // the identity; points that project are queued for the map
                // kernel (network proposal, residual check, exact fallback) unless
                // their state is inverted, which takes the exact map here
                double qlim = 0;
                Trial r{};
                if (crushedOk) r = compute_pq_fast(F00, F01, F10, F11, cp.mu, cp.kappa);
                const int br = crushedOk ? map_branch(k, r, Jp, qlim) : kBrInside;
                const bool proj = crushedOk && br != kBrInside;
                // the network proposes only in the branches it is enabled for
                // (the autotuner switches off a branch whose proposals the yield
                // gate does not pass); the others take the exact map here
                const int bit = (br == kBrTension) ? kMapTension : kMapShear;
                defer = proj && r.svd.s1 > 0 && (la.branches & bit) != 0;
                if (proj && !defer) dp_return(k, r, F00, F01, F10, F11, Jp);
                const unsigned long long dm = __ballot(defer);
                if (dm) {
                    unsigned int base = 0;
                    if (lane == 0) base = atomicAdd(mq.count, (unsigned int)__popcll(dm));
                    base = __shfl(base, 0, 64);
                    const unsigned int slot = base + (unsigned int)__popcll(dm & ((1ull << lane) - 1ull));
                    if (defer) {
                        if (slot < (unsigned int)mq.cap) {
                            MapEntry &e = mq.q[slot];
                            e.pt = pt;
                            e.cs = rec.cs;
                            e.F[0] = F00; e.F[1] = F01; e.F[2] = F10; e.F[3] = F11;
                            e.Jp = Jp;
                            // the position at its stored precision, as the P2G here would take it
                            if constexpr (F32) {
                                unsigned int hi, lo;
                                e.x[0] = fix_put_cells(px, cp, hi, lo) * cp.posQ;
                                e.x[1] = fix_put_cells(py, cp, hi, lo) * cp.posQ;
                            } else {
                                e.x[0] = px;
                                e.x[1] = py;
                            }
                            e.v[0] = vx; e.v[1] = vy;
                            e.B[0] = B00; e.B[1] = B01; e.B[2] = B10; e.B[3] = B11;
                        } else {
                            flag_error(k);
                        }
                    }
                }
                const unsigned long long fb = __ballot(proj && !defer), ins = __ballot(crushedOk && !proj);
                if (lane == 0 && (fb | ins)) {
                    if (fb) atomicAdd(&la.stats[1], (unsigned long long)__popcll(fb));
                    if (ins) atomicAdd(&la.stats[2], (unsigned long long)__popcll(ins));
                }
            }
            if (ok) {
                // px, py become what the rows hold: the P2G takes them at their
                // stored precision
                if constexpr (F32) {
                    // a position outside the grid (or NaN) is an error here, as
                    // the next stencil of FP64 rows would report it; the fixed
                    // point clamps it
                    if (!(px >= 0.0 && px < (double)gx && py >= 0.0 && py < (double)gy)) flag_error(k);
                }
            }
            if constexpr (F32) {
                unsigned int hx, lx, hy, ly;
                px = fix_put_cells(px, cp, hx, lx) * cp.cellQ;
                py = fix_put_cells(py, cp, hy, ly) * cp.cellQ;
                const prec4 r = {hx, hy, lx | (ly << 16), (unsigned)crushed | ((unsigned)(unsigned short)grain << 16)};
                const fe4 f = {(float)(F00 - fe0), (float)F01, (float)F10, (float)(F11 - fe0)};
                if (ok) {
                    __builtin_nontemporal_store(r, reinterpret_cast<prec4 *>(S.pos) + u);
                    if (!defer) __builtin_nontemporal_store(f, fe_rec(R, pp) + u);
                }
                // a point the map left alone keeps the stress of its trial
                // state: the P2G takes it from the invariants, which describe F
                // before its rounding to the stored FP32 (~6e-8 of Fe - I).  A
                // crushed point's Fe is taken as the next substep reads it back.
                F00 = f.x; F01 = f.y; F10 = f.z; F11 = f.w;
            } else if (ok) {
                pos_store(S.pos, pp, pt, px, py);
                if (!defer) {   // as pos_store
                    *at(R + pp * 2, u) = (V)F00;
                    *at(R + pp * 3, u) = (V)F01;
                    *at(R + pp * 4, u) = (V)F10;
                    *at(R + pp * 5, u) = (V)F11;
                }
            }
            // v and Bp: a fused pass uses them at once (a deferred point's go
            // to the map kernel in its queue entry) and the next G2P
            // recomputes them before any use; the last pass of a run stores
            // them (storeVB), for readback, checkpoints and a P2G that
            // starts afresh
            if (storeVB && ok) {
                R[pt] = (V)vx;
                R[pp + pt] = (V)vy;
                R[pp * 6 + pt] = (V)B00;
                R[pp * 7 + pt] = (V)B01;
                R[pp * 8 + pt] = (V)B10;
                R[pp * 9 + pt] = (V)B11;
            }
            if (ok && Jp != Jp0 && !defer) *at(jpRow, u) = (V)(Jp - fe0);
            if (!F32 && ok && crushed != crushed0) *at(S.crushed, u) = crushed;   // FP32: in the record
            M::kirchhoff_from_inv(iv, t00, t01, t11);
            if (crushedOk) M::kirchhoff_rcp(fe0 + F00, F01, F10, fe0 + F11, cp.mu, cp.kappa, t00, t01, t11);
        } else {
            if constexpr (F32) {
                px = fix_cells(pr.x, pr.z & 0xFFFFu, cp);
                py = fix_cells(pr.y, pr.z >> 16, cp);
                F00 = fe0 + (double)fr.x;
                F01 = (double)fr.y;
                F10 = (double)fr.z;
                F11 = fe0 + (double)fr.w;
            }
            vx = (double)R[us];
            vy = (double)R[pp + us];
            B00 = (double)R[pp * 6 + us];
            B01 = (double)R[pp * 7 + us];
            B10 = (double)R[pp * 8 + us];
            B11 = (double)R[pp * 9 + us];
            kirchhoff_rcp(F00, F01, F10, F11, cp.mu, cp.kappa, t00, t01, t11);
        }

        // ---- P2G of the points as they now are ----
        int bx = 0, by = 0;
        double fx0 = 0, fx1 = 0, wx0 = 0, wx1 = 0, wx2 = 0, wy0 = 0, wy1 = 0, wy2 = 0;
        bool ok = valid;
        if constexpr (F32) {   // cell units
            stencil_cells(px, bx, fx0, wx0, wx1, wx2);
            stencil_cells(py, by, fx1, wy0, wy1, wy2);
        } else {
            const bool st = px == px && py == py && M::stencil(px, cp.h_inv, bx, fx0, wx0, wx1, wx2) &&
                            M::stencil(py, cp.h_inv, by, fx1, wy0, wy1, wy2);
            ok = valid && st;
            if (valid && !st) flag_error(k);
        }
        // the cells of the points in the grid (deferred ones, whose P2G is the
        // map kernel's, too: the next G2P gathers for them as well)
        if (ok && bx < gx && by < gy) {
            cellx = bx;
            celly = by;
        }
        const int lx0 = bx - wx, ly0 = by - wy;
        const bool inWin = ok && (unsigned)lx0 < ww2 && (unsigned)ly0 < wh2;
        const bool winFits = inWin && !defer;
        // Every point of a case has the same mass m: the window sums the
        // contributions per unit mass, W (v + (Bp - m^-1 dt V D^-1 tau) d),
        // and the flush multiplies by m once per node.
        const double h = cp.h;
        const double A00 = B00 - cp.scm * t00, A01 = B01 - cp.scm * t01;
        const double A10 = B10 - cp.scm * t01, A11 = B11 - cp.scm * t11;
        if constexpr (kInOrder) {
            // A quad of lanes whose four points share one base cell (in band
            // order most quads, until points cross into other cells) and whose
            // stencil lies in the window sums its contributions in registers
            // before they reach the window.  Every lane is active here.
            const bool quad = quad_uniform(winFits ? (unsigned)bx | (unsigned)by << 16 : 0xFFFF0000u | (unsigned)lane);
            if (quad) {
                quad_scatter(lane, ly0 * wS + lx0, wS, h, fx0, fx1, wx0, wx1, wx2, wy0, wy1, wy2, vx, vy, A00, A01, A10,
                             A11, W0, W1, W2);
            } else if (winFits) {
                const int e0 = ly0 * wS + lx0;
                // The four lanes of a quad (in band order mostly the points of
                // one cell) walk the 3 x 3 stencil from four different nodes,
                // so their LDS atomics never meet at one address: lane bit 0
                // shifts the columns, bit 1 the rows, by one.  Step k of an
                // axis visits node (k + s) mod 3 = s, 1 + s, 2 - 2 s; only the
                // weights need selecting, the offsets follow from the index.
                const int sx = lane & 1, sy = (lane >> 1) & 1;
                const int xe[3] = {sx, 1 + sx, 2 - 2 * sx};
                const int iy[3] = {sy, 1 + sy, 2 - 2 * sy};
                const int ye[3] = {iy[0] * wS, iy[1] * wS, iy[2] * wS};
                const double xw[3] = {sx ? wx1 : wx0, sx ? wx2 : wx1, sx ? wx0 : wx2};
                const double yw[3] = {sy ? wy1 : wy0, sy ? wy2 : wy1, sy ? wy0 : wy2};
                double xa[3], xb[3], ya[3], yb[3];
    #pragma unroll
                for (int q = 0; q < 3; ++q) {
                    const double dx = ((double)xe[q] - fx0) * h, dy = ((double)iy[q] - fx1) * h;
                    xa[q] = vx + A00 * dx;
                    xb[q] = vy + A10 * dx;
                    ya[q] = A01 * dy;
                    yb[q] = A11 * dy;
                }
    #pragma unroll
                for (int a = 0; a < 3; ++a)
    #pragma unroll
                    for (int b = 0; b < 3; ++b) {
                        const double W = xw[a] * yw[b];
                        const int e = e0 + xe[a] + ye[b];
                        atomicAdd(&W0[e], W);
                        atomicAdd(&W1[e], W * (xa[a] + ya[b]));
                        atomicAdd(&W2[e], W * (xb[a] + yb[b]));
                    }
            }
        } else if (winFits) {
            const double wxs[3] = {wx0, wx1, wx2}, wys[3] = {wy0, wy1, wy2};
            double *w0 = W0 + ly0 * wS + lx0, *w1 = w0 + wS, *w2 = w1 + wS;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const double dx = (i - fx0) * h, xa = vx + A00 * dx, xb = vy + A10 * dx;
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    double *w = (j == 0 ? w0 : (j == 1 ? w1 : w2)) + i;
                    const double W = wxs[i] * wys[j], dy = (j - fx1) * h;
                    atomicAdd(w, W);
                    atomicAdd(w + kWin, W * (xa + A01 * dy));
                    atomicAdd(w + 2 * kWin, W * (xb + A11 * dy));
                }
            }
        }
        // outside the window, or the stencil leaves the grid: the box of touched
        // nodes has to hold these (deferred points too, which the map kernel
        // scatters), and they are added node by node
        if (ok && !inWin) widen_bounds(bounds, rec.cs, bx, by, min(bx, gx), min(by, gy));
        if (ok && !inWin && !defer) {
            const double m = cp.mass;
#pragma unroll 1
            for (int e = 0; e < 9; ++e) {
                const int i = e % 3, j = e / 3, X = bx + i, Y = by + j;
                if (X >= gx || Y >= gy) {
                    flag_error(k);
                    continue;
                }
                const double W = sel3(i, wx0, wx1, wx2) * sel3(j, wy0, wy1, wy2);
                const double d0 = (i - fx0) * h, d1 = (j - fx1) * h;
                const unsigned node = (unsigned)(X + Y * gx);
                unsafeAtomicAdd(at(gO, node), W * m);
                unsafeAtomicAdd(at(gO + gpitch, node), W * (vx + (A00 * d0 + A01 * d1)) * m);
                unsafeAtomicAdd(at(gO + 2 * gpitch, node), W * (vy + (A10 * d0 + A11 * d1)) * m);
            }
        }
    }

    if (!F32 || joint)
        __syncthreads();
    else
        wsync();
    if constexpr (F32) __builtin_amdgcn_s_setprio(2);
    // the windows to the grid, three sums of a node in one LDS round trip; the
    // atomics address the rows from their scalar bases with 32-bit offsets
    const auto add = [&](int X, int Y, double a, double a1, double a2) {
        if (a != 0 && X < gx && Y < gy) {
            const unsigned node = (unsigned)(X + Y * gx);
            unsafeAtomicAdd(at(gO, node), a);
            unsafeAtomicAdd(at(gO + gpitch, node), a1);
            unsafeAtomicAdd(at(gO + 2 * gpitch, node), a2);
        }
    };
    const double m = cp.mass;   // the windows hold sums per unit mass
    if (!F32 || joint) {
        for (unsigned e = threadIdx.x; e < nodes; e += 64 * kWaves) {
            unsigned c, r;
            box_node(e, rec.inv, (unsigned)bw, c, r);
            double a, a1, a2;
            if constexpr (F32) {
                a = a1 = a2 = 0;
#pragma unroll
                for (int q = 0; q < kWaves; ++q) {
                    const unsigned win = rec.win[q], x = c - (win & 0xFFu), y = r - (win >> 8 & 0xFFu);
                    const unsigned w = win >> 16 & 0xFFu, h = win >> 24;
                    if (x < w && y < h) {
                        const double *W = smem + q * 3 * kWaveWin + y * (unsigned)win_stride((int)w) + x;
                        a += W[0] * m;
                        a1 += W[kWaveWin] * m;
                        a2 += W[2 * kWaveWin] * m;
                    }
                }
            } else {
                const double *W = W0 + r * (unsigned)wS + c;
                a = W[0] * m;
                a1 = W[kWin] * m;
                a2 = W[2 * kWin] * m;
            }
            add(ox + (int)c, oy + (int)r, a, a1, a2);
        }
    } else if (wcol < ww) {
        for (int r = wrow0; r < wh; r += wstep) {
            const int e = r * wS + wcol;
            add(wx + wcol, wy + r, W0[e] * m, W1[e] * m, W2[e] * m);
        }
    }
    if (step % kBoxEvery == 0) {
        // the box and the windows of the points as they now are
        const unsigned x0 = wave_min_u32((unsigned)cellx), y0 = wave_min_u32((unsigned)celly);
        const unsigned x1 = wave_max_u32((unsigned)(cellx + 1)), y1 = wave_max_u32((unsigned)(celly + 1));
        __syncthreads();   // the windows have been read
        unsigned *lim = reinterpret_cast<unsigned *>(smem);
        if (lane == 0) {
            lim[row] = x0;
            lim[4 + row] = y0;
            lim[8 + row] = x1;
            lim[12 + row] = y1;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned q0 = lim[0], q1 = lim[4], q2 = lim[8], q3 = lim[12];
            for (int q = 1; q < kWaves; ++q) {
                q0 = min(q0, lim[q]);
                q1 = min(q1, lim[4 + q]);
                q2 = max(q2, lim[8 + q]);
                q3 = max(q3, lim[12 + q]);
            }
            ChunkRec &out = recs[chunk];
            if (q2 == 0) {   // no point in the grid
                out.ext = 0;
                for (int q = 0; q < 4; ++q) out.win[q] = 0;
            } else if (set_box(out, (int)q0, (int)q1, (int)q2 - 1, (int)q3 - 1, kTile)) {
                for (int q = 0; q < kWaves; ++q)
                    out.win[q] = lim[8 + q] ? win_of(out, (int)lim[q], (int)lim[4 + q], (int)lim[8 + q] - 1,
                                                     (int)lim[12 + q] - 1)
                                            : 0u;
                widen_bounds(bounds, rec.cs, (int)q0, (int)q1, (int)q2 - 1, (int)q3 - 1);
            }
            // a point far from the others must not take the box away from them:
            // one that cannot hold all points stays where it was
        }
    }
}

// The boxes of the chunks' points as they are, a wavefront a chunk: what a
// run's first P2G, or a table rebuilt between two runs, starts from.
// starts (one case only, may be null): the chunks' first slots and the end, from
// which the rest of their records is made first.
template <bool F32>
__global__ __launch_bounds__(256) void k_chunk_boxes(ChunkRec *recs, int nChunks, const typename Rows<F32>::P *pos,
                                                     size_t pitch, const CaseParams *__restrict__ cases, int4 *bounds,
                                                     const int *__restrict__ starts, int waves, int inOrder) {
    const int ch = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, lane = threadIdx.x & 63;
    if (ch >= nChunks) return;
    ChunkRec rec = recs[ch];
    if (starts) {
        rec = ChunkRec{};
        rec.beg = starts[ch];
        rec.shape = inOrder ? (unsigned)(starts[ch + 1] - rec.beg) : chunk_shape(starts[ch + 1] - rec.beg);
        rec.dims = (unsigned)cases[0].gx | (unsigned)cases[0].gy << 16;
    }
    const CaseParams &cp = cases[rec.cs];
    const int count = inOrder ? (int)rec.shape : chunk_count(rec.shape), space = box_space(waves);
    int wx0[4], wy0[4], wx1[4], wy1[4];   // of each wavefront's points
    int fx = 0, fy = 0, x0 = INT_MAX, y0 = INT_MAX, x1 = -1, y1 = -1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int i = q * 64 + lane;
        int bx = -1, by = -1;
        if (i < count) {
            double f, a, b, c;
            if constexpr (F32) {
                const prec4 r = reinterpret_cast<const prec4 *>(pos)[rec.beg + i];
                stencil_cells(fix_cells(r.x, r.z & 0xFFFFu, cp), bx, f, a, b, c);
                stencil_cells(fix_cells(r.y, r.z >> 16, cp), by, f, a, b, c);
            } else {
                double x, y;
                pos_load(pos, pitch, rec.beg + i, cp, x, y);
                if (!stencil(x, cp.h_inv, bx, f, a, b, c) || !stencil(y, cp.h_inv, by, f, a, b, c)) bx = -1;
            }
        }
        const bool in = (unsigned)bx < (unsigned)cp.gx && (unsigned)by < (unsigned)cp.gy;
        if (q == 0) {
            fx = __builtin_amdgcn_readlane(in ? bx : 0, 0);
            fy = __builtin_amdgcn_readlane(in ? by : 0, 0);
        }
        wx0[q] = (int)min(wave_min_u32(in ? (unsigned)bx : 0xFFFFFFFFu), (unsigned)INT_MAX);
        wy0[q] = (int)min(wave_min_u32(in ? (unsigned)by : 0xFFFFFFFFu), (unsigned)INT_MAX);
        wx1[q] = (int)wave_max_u32(in ? (unsigned)bx + 1u : 0u) - 1;
        wy1[q] = (int)wave_max_u32(in ? (unsigned)by + 1u : 0u) - 1;
        x0 = min(x0, wx0[q]);
        y0 = min(y0, wy0[q]);
        x1 = max(x1, wx1[q]);
        y1 = max(y1, wy1[q]);
    }
    if (lane == 0) {
        // too wide a box (the points of a stale order): the cells of the first
        // point's surroundings
        rec.ext = 0;
        for (int q = 0; q < 4; ++q) rec.win[q] = 0;
        if (x0 <= x1) widen_bounds(bounds, rec.cs, x0, y0, x1, y1);
        if (x0 <= x1 && !set_box(rec, x0, y0, x1, y1, space)) {
            x0 = max(fx - 7, x0);
            x1 = min(fx + 7, x1);
            y0 = max(fy - 7, y0);
            y1 = min(fy + 7, y1);
            if (x0 <= x1 && y0 <= y1) (void)set_box(rec, x0, y0, x1, y1, space);
        }
        if (rec.ext) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (wx1[q] >= 0) rec.win[q] = win_of(rec, wx0[q], wy0[q], wx1[q], wy1[q]);
        }
        recs[ch] = rec;
    }
}

// P2G of a deferred point from the position, velocity and Bp its queue entry
// carries and the given Fe (rounded to the storage type first, as the pass
// continues from what it stores), straight to the grid with global atomics.
template <bool F32>
static __device__ void scatter_point(const MapEntry &e, const CaseParams &cp, const KParams &k,
                                     double F00, double F01, double F10, double F11,
                                     double *__restrict__ gridOut, size_t gpitch) {
    using V = typename Rows<F32>::V;
    constexpr double fe0 = F32 ? 1.0 : 0.0;
    const double px = e.x[0], py = e.x[1];
    const double vx = e.v[0], vy = e.v[1];
    const double B00 = e.B[0], B01 = e.B[1], B10 = e.B[2], B11 = e.B[3];
    if constexpr (F32) {
        F00 = fe0 + (double)(V)(F00 - fe0); F01 = (double)(V)F01;
        F10 = (double)(V)F10; F11 = fe0 + (double)(V)(F11 - fe0);
    }
    int bx, by;
    double fx0, fx1, wx0, wx1, wx2, wy0, wy1, wy2;
    if (!(px == px && py == py) || !stencil(px, cp.h_inv, bx, fx0, wx0, wx1, wx2) ||
        !stencil(py, cp.h_inv, by, fx1, wy0, wy1, wy2)) {
        flag_error(k);
        return;
    }
    {
        double t00, t01, t11;
        kirchhoff(F00, F01, F10, F11, cp.mu, cp.kappa, t00, t01, t11);
        const double m = cp.mass, h = cp.h;
        const double sc2 = cp.dt * cp.vol * cp.Dinv;
        const double A00 = m * B00 - sc2 * t00, A01 = m * B01 - sc2 * t01;
        const double A10 = m * B10 - sc2 * t01, A11 = m * B11 - sc2 * t11;
        const double mv0 = vx * m, mv1 = vy * m;
        double *__restrict__ gO = gridOut + cp.gridOffset;
        for (int a = 0; a < 3; ++a)
            for (int b = 0; b < 3; ++b) {
                const int X = bx + a, Y = by + b;
                if (X >= cp.gx || Y >= cp.gy) {
                    flag_error(k);
                    continue;
                }
                const double Wip = sel3(a, wx0, wx1, wx2) * sel3(b, wy0, wy1, wy2);
                const double d0 = (a - fx0) * h, d1 = (b - fx1) * h;
                const int node = X + Y * cp.gx;
                unsafeAtomicAdd(&gO[node], Wip * m);
                unsafeAtomicAdd(&gO[gpitch + node], Wip * (mv0 + (A00 * d0 + A01 * d1)));
                unsafeAtomicAdd(&gO[2 * gpitch + node], Wip * (mv1 + (A10 * d0 + A11 * d1)));
            }
    }
}

// The learned return map of the points a particle pass deferred: the MLP
// (one 16-row MFMA tile per wavefront and iteration, weights staged in
// shared memory) proposes the projected state of
// each queued point, the proposal is kept where its yield residual is <=
// tol and the exact FP64 map runs otherwise; then Fe and Jp_inv are stored
// and, when gridOut is given, the point's P2G contribution goes to the grid
// with global atomics (the pass left these points out of its P2G).  Resets
// the counter the next pass appends to.
template <bool F32>
__global__ __launch_bounds__(256) void k_batch_map(Rows<F32> S, const CaseParams *__restrict__ cases,
                                                  const MapEntry *__restrict__ q,
                                                  const unsigned int *__restrict__ qCount,
                                                  unsigned int *__restrict__ qCountNext,
                                                  double *__restrict__ gridOut, size_t gpitch,
                                                  int *__restrict__ err, LearnArgs la) {
    __shared__ mlpdev::InferScratch isc[4];
    __shared__ __attribute__((aligned(16))) unsigned short wsh[mlpdev::kParams];   // the weights, BF16
    using V = typename Rows<F32>::V;
    constexpr double fe0 = F32 ? 1.0 : 0.0;
    __shared__ unsigned int counts[kMapStats];
    if (blockIdx.x == 0 && threadIdx.x == 0) qCountNext[0] = 0u;
    const unsigned int n = qCount[0];
    if (blockIdx.x * 64u >= n) return;   // no entry for this block (uniform)
    static_assert(mlpdev::kParams % 8 == 0, "weights are staged 8 at a time");
    for (int x = threadIdx.x; x < mlpdev::kParams / 8; x += 256)
        reinterpret_cast<uint4 *>(wsh)[x] = reinterpret_cast<const uint4 *>(la.wbf)[x];
    if (threadIdx.x < kMapStats) counts[threadIdx.x] = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const size_t pp = S.pitch;
    V *__restrict__ R = S.rest;
    mlpdev::InferScratch &sc = isc[wv];
    // one 16-row tile per wavefront and iteration: lanes 0..15 own the entries
    for (unsigned int base = (blockIdx.x * 4 + wv) * 16u; base < n; base += gridDim.x * 64u) {
        const unsigned int i = base + lane;
        const bool have = lane < 16 && i < n;
        MapEntry e{};
        if (have) e = q[i];
        const CaseParams &cp = cases[have ? e.cs : 0];
        const KParams k = kp_of(cp, err);
        double F00 = have ? e.F[0] : 1.0, F01 = e.F[1], F10 = e.F[2], F11 = have ? e.F[3] : 1.0;
        double Jp = have ? e.Jp : 1.0;
        const Trial r = compute_pq_fast(F00, F01, F10, F11, cp.mu, cp.kappa);
        double qlim = 0;
        const int br = map_branch(k, r, Jp, qlim);
        const bool need = have && br != kBrInside && r.svd.s1 > 0;
        double pred[3] = {0, 0, 0};
        if (__ballot(need)) {
            for (int x = lane; x < 16 * mlpdev::kIn; x += 64) sc.x[x / mlpdev::kIn][x % mlpdev::kIn] = 0;
            mlpdev::wave_fence();
            if (need) {
                double f[5];
                map_features(r, Jp, br, f);
                for (int t = 0; t < 5; ++t)
                    sc.x[lane][t] = mlpdev::to_bf16((float)((f[t] - la.norm.in_mean[t]) / la.norm.in_scale[t]));
            }
            mlpdev::wave_fence();
            mlpdev::infer16(sc, wsh, la.pf);
            if (need)
                for (int t = 0; t < 3; ++t)
                    pred[t] = (double)sc.y[lane][t] * la.norm.out_scale[t] + la.norm.out_mean[t];
            mlpdev::wave_fence();
        }
        bool accepted = false;
        if (need) {
            const double s0 = r.svd.s0 * exp(pred[0]);   // log s0 + pred0, exponentiated
            const double s1 = r.svd.s1 * exp(pred[1]);
            // the shear branch leaves Jp_inv unchanged
            const double Jpn = (br == kBrTension) ? Jp * exp(pred[2]) : Jp;
            if (yield_residual(k, r, Jp, br, qlim, s0, s1, Jpn) <= la.tol) {
                usvt(r.svd, s0, s1, F00, F01, F10, F11);
                Jp = Jpn;
                accepted = true;
            }
        }
        if (have && !accepted) dp_return(k, r, F00, F01, F10, F11, Jp);
        const unsigned long long acc = __ballot(accepted), fb = __ballot(have && !accepted);
        const unsigned long long ten = __ballot(have && br == kBrTension);
        if (lane == 0) {
            if (acc) atomicAdd(&counts[0], (unsigned)__popcll(acc));
            if (fb) atomicAdd(&counts[1], (unsigned)__popcll(fb));
            if (acc & ten) atomicAdd(&counts[3], (unsigned)__popcll(acc & ten));
            if (fb & ten) atomicAdd(&counts[4], (unsigned)__popcll(fb & ten));
            if (acc & ~ten) atomicAdd(&counts[5], (unsigned)__popcll(acc & ~ten));
            if (fb & ~ten) atomicAdd(&counts[6], (unsigned)__popcll(fb & ~ten));
        }
        if (have) {
            const int pt = e.pt;
            if constexpr (F32) {
                fe_rec(R, pp)[pt] = fe4{(float)(F00 - fe0), (float)F01, (float)F10, (float)(F11 - fe0)};
            } else {
                R[pp * 2 + pt] = (V)(F00 - fe0);
                R[pp * 3 + pt] = (V)F01;
                R[pp * 4 + pt] = (V)F10;
                R[pp * 5 + pt] = (V)(F11 - fe0);
            }
            if (Jp != e.Jp) R[pp * 10 + pt] = (V)(Jp - fe0);
            if (gridOut) scatter_point<F32>(e, cp, k, F00, F01, F10, F11, gridOut, gpitch);
        }
    }
    __syncthreads();
    if (threadIdx.x < kMapStats && counts[threadIdx.x])
        atomicAdd(&la.stats[threadIdx.x], (unsigned long long)counts[threadIdx.x]);
}

__global__ void k_reset_bounds(int4 *bounds, int nCases) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c < nCases) bounds[c] = make_int4(INT_MAX, INT_MAX, -1, -1);
}

// Cell key of every point of the batch, offset by its case's first node so
// that a sort keeps the cases contiguous and in order; vals = slot index.
template <class PT>
__global__ void k_batch_keys(const PT *__restrict__ pos, size_t pitch, int nPts,
                             const CaseParams *__restrict__ cases, int nCases, int *__restrict__ keys,
                             int *__restrict__ vals) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nPts) return;
    int lo = 0, hi = nCases - 1;   // the last case with ptOffset <= i
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (cases[mid].ptOffset <= i) lo = mid; else hi = mid - 1;
    }
    const CaseParams &cp = cases[lo];
    double x, y;
    pos_load(pos, pitch, i, cp, x, y);
    int key = cp.gridTotal - 1;
    if (x == x && y == y) {
        const double bx = fmin(fmax(x * cp.h_inv - 0.5, 0.0), (double)(cp.gx - 1));
        const double by = fmin(fmax(y * cp.h_inv - 0.5, 0.0), (double)(cp.gy - 1));
        key = band_key((int)bx, (int)by, cp.gx, cp.gy);
    }
    keys[i] = cp.gridOffset + key;
    vals[i] = i;
}

// The case-local base cell of every slot (of slot order[i], when an order that
// keeps the cases apart is given), packed as column | row << 16
// (finalize keeps every grid within 65536 columns and rows): what the chunk
// table is built from, without the band key's divisions on the host.
template <class PT>
__global__ void k_batch_cells(const PT *__restrict__ pos, size_t pitch, int nPts,
                              const CaseParams *__restrict__ cases, int nCases, const int *__restrict__ order,
                              unsigned *__restrict__ cells) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nPts) return;
    int lo = 0, hi = nCases - 1;   // the last case with ptOffset <= i
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (cases[mid].ptOffset <= i) lo = mid; else hi = mid - 1;
    }
    const CaseParams &cp = cases[lo];
    double x, y;
    pos_load(pos, pitch, order ? order[i] : i, cp, x, y);
    // the cell k_batch_keys keys the slot by (a NaN position: the last cell)
    unsigned cx = (unsigned)(cp.gx - 1), cy = (unsigned)(cp.gy - 1);
    if (x == x && y == y) {
        cx = (unsigned)fmin(fmax(x * cp.h_inv - 0.5, 0.0), (double)(cp.gx - 1));
        cy = (unsigned)fmin(fmax(y * cp.h_inv - 0.5, 0.0), (double)(cp.gy - 1));
    }
    cells[i] = cx | cy << 16;
}

// An order of the points in band order, rearranged into the chunks' slot orders.
__global__ void k_chunk_order(const ChunkRec *__restrict__ recs, int nChunks, const int *__restrict__ in,
                              int *__restrict__ out) {
    const int ch = blockIdx.x;
    if (ch >= nChunks) return;
    const int beg = recs[ch].beg, n = chunk_count(recs[ch].shape);
    if ((int)threadIdx.x < n) out[beg + threadIdx.x] = in[beg + chunk_point((int)threadIdx.x, recs[ch].shape)];
}

// Points [first, first + pitch) of a case in the layout they came in: rows 0 and
// 3-15 of the point SoA (row r > 2 at out + (r - 2) pitch), every point at its
// index within the case less first.  bad: set when the slot map is not one.
template <bool F32>
__global__ __launch_bounds__(256) void k_read_points(Rows<F32> S, const int *__restrict__ orig, CaseParams cp, int first,
                                                     int pitch, double *__restrict__ out, int *__restrict__ bad) {
    const int k = blockIdx.x * 256 + threadIdx.x, n = cp.nPts, o = cp.ptOffset;
    if (k >= n) return;
    const int slot = o + k, i = orig[slot] - o - first;
    if (i < -first || i >= n - first) {
        *bad = 1;
        return;
    }
    if (i < 0 || i >= pitch) return;   // of another part
    const size_t pp = S.pitch;
    const auto *__restrict__ R = S.rest;
    double v[13];   // Jp, x, y, v, Fe, Bp
    unsigned char crushed;
    short grain = 0;
    if constexpr (F32) {
        const unsigned w = pos_load(S.pos, pp, slot, cp, v[1], v[2]);
        crushed = (unsigned char)(w & 0xFFu);
        grain = (short)(w >> 16);
        const fe4 f = fe_rec(R, pp)[slot];
        v[5] = (double)f.x + 1.0;
        v[6] = (double)f.y;
        v[7] = (double)f.z;
        v[8] = (double)f.w + 1.0;
        v[0] = (double)R[pp * 10 + slot] + 1.0;
    } else {
        pos_load(S.pos, pp, slot, cp, v[1], v[2]);
        crushed = S.crushed[slot];
        if (S.grain) grain = S.grain[slot];
        for (int r = 2; r < 6; ++r) v[3 + r] = R[pp * r + slot];
        v[0] = R[pp * 10 + slot];
    }
    v[3] = (double)R[slot];
    v[4] = (double)R[pp + slot];
    for (int r = 6; r < 10; ++r) v[3 + r] = (double)R[pp * r + slot];
    unsigned char *u8 = reinterpret_cast<unsigned char *>(out);
    u8[i] = crushed;
    *reinterpret_cast<short *>(u8 + pitch + 2 * (size_t)i) = grain;   // point.cpp:19-23
    for (int r = 0; r < 13; ++r) out[(size_t)(r + 1) * pitch + i] = v[r];
}

// Point state permuted: slot k of the destination <- slot perm[k] of the source.
template <bool F32>
__global__ void k_batch_permute(Rows<F32> src, Rows<F32> dst, const int *__restrict__ srcOrig,
                                int *__restrict__ dstOrig, const int *__restrict__ perm, int nPts) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nPts) return;
    const int j = perm[k];
    const size_t p = src.pitch;
    if constexpr (F32)
        reinterpret_cast<prec4 *>(dst.pos)[k] = reinterpret_cast<const prec4 *>(src.pos)[j];
    else
        for (int r = 0; r < Rows<F32>::kPosRows; ++r) dst.pos[r * p + k] = src.pos[r * p + j];
    if constexpr (F32) {
        for (int r = 0; r < 11; ++r)
            if (r < 2 || r > 5) dst.rest[r * p + k] = src.rest[r * p + j];
        fe_rec(dst.rest, p)[k] = fe_rec(static_cast<const float *>(src.rest), p)[j];
    } else {
        for (int r = 0; r < 11; ++r) dst.rest[r * p + k] = src.rest[r * p + j];
    }
    dst.crushed[k] = src.crushed[j];
    if (src.grain) dst.grain[k] = src.grain[j];
    dstOrig[k] = srcOrig[j];
}

}  // namespace batch
}  // namespace icempm

using namespace icempm;
using namespace icempm::batch;

constexpr int kReadGroups = 4;       // groups of rows of a readback
constexpr int kReadPart = 1 << 16;   // points of a case it brings down at a time (a multiple of 64)

struct icempm_batch {
    int precision = ICEMPM_BATCH_F64;
    hipStream_t stream = nullptr;
    // The cases in kChains groups of about equal point counts run their
    // substep loops as independent chains (group g > 0 on side[g - 1]), so
    // that one group's launches fill the gaps and the tail of the other's.
    // groupCase: each group's first case; grpChunk / grpBlock: the groups'
    // ranges of the chunk records and of the node blocks; chains: the
    // number of groups (1 when there is one case).
    static constexpr int kChains = ICEMPM_BATCH_CHAINS;
    hipStream_t side[kChains - 1] = {};
    hipEvent_t evFork = nullptr;
    hipEvent_t evJoin[kChains - 1] = {};
    int chains = 1;
    int groupCase[kChains + 1] = {};
    int grpChunk[kChains + 1] = {};
    int grpBlock[kChains + 1] = {};
    std::string lastError;
    bool finalized = false;

    struct HostCase {
        CaseParams cp;
        std::vector<double> pos;        // 2 x n
        std::vector<double> rest;       // 11 x n
        std::vector<unsigned char> crushed;
        std::vector<short> grain;
        std::vector<int> keys;
    };
    std::vector<HostCase> hc;

    // device
    void *pos = nullptr;          // Rows<F32>::kPosRows rows of Rows<F32>::P
    void *rest = nullptr;
    unsigned char *crushed = nullptr;
    short *grain = nullptr;       // per-point grain ids (when a case has GrainVariability != 0)
    double *bins = nullptr;       // indenter force bins of every case, summed over a run
    int binsTotal = 0;            // doubles
    size_t pitch = 0;
    int nPts = 0;
    double *grids = nullptr;   // three grids of 3 rows each, used in turn: read, scattered into, cleared
    int4 *bounds = nullptr;    // per case: the nodes touched since the run's fresh start
    size_t gpitch = 0;
    long nNodes = 0;
    CaseParams *cases = nullptr;
    ChunkRec *recs = nullptr;   // nChunks records
    int nChunks = 0;
    int waves = 4;              // wavefronts of a workgroup, for the largest of them
    bool inOrder = true;        // the points of a chunk are in band order (else in rows)
    size_t recCap = 0;
    int2 *nodeBlock = nullptr;
    int nNodeBlocks = 0;
    int *err = nullptr;
    double *tTab = nullptr;
    double *hist = nullptr;
    int cap = 0;               // substeps the buffers hold
    int lastRun = 0;

    double t = 0;
    int step = 0;

    // return map of crushed points
    int rmap = kMapExact;
    unsigned short *mlpW = nullptr;   // MLP parameters as BF16 bits
    float *mlpP = nullptr;            // and as FP32
    mlpdev::Norm norm{};
    double tol = 1e-4;
    float *hx = nullptr, *ht = nullptr;
    unsigned long long *hcount = nullptr;
    int hcap = 0;
    unsigned long long *stats = nullptr;   // kMapStats counters
    int mapBranches = kMapTension | kMapShear;   // branches the network proposes for
    double mapMinAccept = 0.5;         // autotune: a branch accepted less often is switched off
    unsigned long long tuneBranchStats[4] = {};   // the last autotune's per-branch accepted / fell back
    MapEntry *mapQ = nullptr;          // deferred points (learned map), nPts entries
    unsigned int *mapCount = nullptr;  // two counters, used alternately

    // executable graphs of the substep loop, two per start (of different
    // step counts, the least recently used replaced): fresh (row 0), or the
    // first substep's P2G already in grid 0, 1 or 2 (rows 1-3, and 4-6 where
    // the boxes are not renewed); each with the step count, time table and
    // history rows it was captured with, and the grid that holds the next P2G
    // after it
    struct GraphSlot {
        hipGraphExec_t exec = nullptr;
        int steps = 0;
        const double *T = nullptr;
        double *H = nullptr;
        int end = -1;
        unsigned long long used = 0;
    };
    GraphSlot graphs[7][2];
    unsigned long long graphTick = 0;
    // the grid (0, 1 or 2) that holds the P2G of the next substep, made
    // from the current points by the last pass of the previous run; -1 when
    // there is none, or the points have changed since (restore, re-sort)
    int pending = -1;
    int boxAge = 0;   // substeps of the last runs since one of them renewed the chunks' boxes
    hipEvent_t e0 = nullptr, e1 = nullptr;
    float lastMs = 0;

    // tuning: points per chunk (at most; = threads per workgroup of the substep
    // kernel) and the re-sort cadence in substeps (0: never)
    int chunkPoints = 256;
    int resortEvery = 0;
    std::vector<int> hcstart, hccase;       // the chunk table on the host
    bool hcdense = false;                   // of a dense cloud (kDensePoints)
    int *orig = nullptr;                    // batch index of the point in each slot
    // re-sort scratch
    int *sKeys = nullptr, *sVals = nullptr, *sKeys2 = nullptr, *sVals2 = nullptr, *sTmp = nullptr;
    // the slots' base cells for a new chunk table: on the device, and read
    // back into pinned host memory
    unsigned *dcells = nullptr, *hcells = nullptr;
    void *tpos = nullptr;
    void *trest = nullptr;
    unsigned char *tcrushed = nullptr;
    short *tgrain = nullptr;
    int *torig = nullptr;
    // checkpoint of the state
    bool haveCheckpoint = false;
    void *kpos = nullptr;
    void *krest = nullptr;
    unsigned char *kcrushed = nullptr;
    short *kgrain = nullptr;
    int *korig = nullptr;
    double kt = 0;
    int kstep = 0;
    std::vector<int> kcstart, kccase;
    bool kcdense = false;
    int kChunkPoints = 256;
    double runMs = 0;   // device time of the last run's segments + re-sorts

    // scratch of read_points, for up to rbPitch points at a time
    std::mutex rbLock;
    double *rbDev = nullptr, *rbHost = nullptr;
    size_t rbPitch = 0;
    hipEvent_t rbEvent[kReadGroups] = {};

    // device timing of the fused particle pass (stream launches only)
    int timingStride = 0;
    std::vector<hipEvent_t> tev;   // pairs
    hipEvent_t evAfter = nullptr;  // while set: recorded after the next particle kernel
    bool storeVB = false;          // while set: the next particle kernel stores v and Bp
    size_t tevNext = 0;
    double timedMs = 0;
    int timedLaunches = 0;
};

namespace {

// A case's constants from its parameters, but for the offsets of a batch.
void fill_case(CaseParams &c, const icy::SimParams &P) {
    c = CaseParams{};
    c.dt = P.InitialTimeStep; c.vol = P.ParticleVolume; c.mass = P.ParticleMass; c.h = P.cellsize;
    c.h_inv = P.cellsize_inv; c.Dinv = P.Dp_inv; c.mu = P.mu; c.kappa = P.kappa; c.gravity = P.Gravity;
    c.indRsq = P.IndRSq; c.indV = P.IndVelocity; c.ics = P.IceCompressiveStrength;
    c.its = P.IceTensileStrength; c.iss = P.IceShearStrength; c.tanPhi = P.DP_tan_phi;
    c.dpThr = P.DP_threshold_p; c.x0 = P.indenter_x_initial; c.y0 = P.indenter_y;
    {
        // NACC constants of grain 0 with no variability (gpu_implementation5.cu:97-141)
        const double pmax = P.IceCompressiveStrength, pmin = -P.IceTensileStrength, qmax = P.IceShearStrength;
        const double beta = -pmin / pmax;
        const double a = pmax * (1 + beta);
        c.pmax = pmax;
        c.msq = (4 * qmax * qmax * (1 + 2 * beta)) / (a * a);
        c.betaPmax = beta * pmax;
        c.onePlus2Beta = 1. + 2. * beta;
        c.slope = -(2 * std::sqrt(-pmax * pmin) * qmax / (pmax - pmin)) / -3e6;
    }
    c.gx = P.GridX; c.gy = P.GridY; c.gridTotal = P.GridTotal; c.nPts = P.nPts;
    c.gxInv = 1.0 / c.gx;
    c.grainVar = P.GrainVariability;
    c.nbins = P.n_indenter_subdivisions;
    c.scm = c.dt * c.vol * c.Dinv / c.mass;
    c.vmax = 0.5 * c.h / c.dt;
    c.dtCells = c.dt * c.h_inv;
    {
        // FP32 storage: 48 - ib fraction bits, ib the bits a cell index needs
        // (finalize refuses grids beyond 65536 nodes a side: ib <= 16)
        int ib = 0;
        while (ib < 16 && (1 << ib) < std::max(c.gx, c.gy)) ++ib;
        const int F = 48 - ib;
        c.cellQ = std::ldexp(1.0, -F);
        c.cellQ16 = std::ldexp(1.0, 16 - F);
        c.cellInvQ = std::ldexp(1.0, F);
        c.posQ = c.h * c.cellQ;
        c.posInvQ = c.cellInvQ / c.h;
    }
}

int bfail(icempm_batch *b, int code, const std::string &m) {
    if (b) b->lastError = m;
    return code;
}

#define BCHK(b, call, tag)                                                                   \
    do {                                                                                     \
        hipError_t _e = (call);                                                              \
        if (_e != hipSuccess) return bfail(b, ICEMPM_E_HIP, std::string(tag) + ": " + hipGetErrorString(_e)); \
    } while (0)

template <class T>
void dfree(T *&p) {
    if (p) (void)hipFree(p);
    p = nullptr;
}

// An array that is allocated once: an earlier call may have failed after some of
// those it needs.
template <class T>
hipError_t once(T *&p, size_t bytes) {
    return p ? hipSuccess : hipMalloc(&p, bytes);
}

constexpr int kMapBlocks = 256;
// batches of fewer chunks run as one chain
constexpr int kChainChunks = 2048;
// FP32 batches of fewer chunks add the wavefronts' windows up in the workgroup
// before they go to the grid, which saves a third of the atomics.  us a substep
// each wavefront for itself -> together: 81 thousand points 9.2 -> 8.2, 671
// thousand with the learned map 38.6 -> 36.2, 6.98 million 171.9 -> 172.0.  There
// the memory's rate is the limit, which the atomics of one line share.
constexpr int kJointChunks = 8192;

// One launch of the substep kernel: a range of the chunks (and of the
// node blocks) with the grids it reads, scatters into and clears.
struct Pass {
    hipStream_t stream;
    int in, out;              // grids
    int chunk0, chunks;
    int block0, blocks;       // node blocks
    const double *t;          // the substep's time
    double *hist;             // of this substep
    int step;                 // its place in the renewals of the boxes
    bool storeVB;
};

template <bool F32, bool G2P, int RMAP, int kWaves, bool kInOrder>
void launch_waves(icempm_batch *b, const Pass &p, const LearnArgs &la, const MapQueue &mq) {
    Rows<F32> S{static_cast<typename Rows<F32>::P *>(b->pos), reinterpret_cast<typename Rows<F32>::V *>(b->rest),
                b->crushed, b->grain, b->pitch};
    const size_t grid = 3 * b->gpitch;
    const int clear = 3 - p.in - p.out;   // the third grid (unused by a first P2G, where in = out)
    NodeWork nw{b->nodeBlock + p.block0, b->grids + (G2P ? clear * grid : 0), p.hist, b->bins};
    const int groups = ((p.chunks + 7) / 8) * 8;
    const int blocks = G2P ? p.blocks * (4 / kWaves) : 0;
    hipLaunchKernelGGL((k_batch_substep<F32, G2P, RMAP, kWaves, kInOrder>), dim3((unsigned)(groups + blocks)), dim3(64 * kWaves), 0,
                       p.stream, b->recs + p.chunk0, b->grids + p.in * grid, p.chunks, groups, S.pos, S.rest, b->gpitch,
                       b->cases, S.crushed, S.pitch, b->grids + p.out * grid, b->bounds, b->err, b->grain,
                       S.rest + 10 * S.pitch, p.t, 0.0, p.step, nw, la, mq, p.storeVB ? 1 : 0,
                       b->nChunks < kJointChunks ? 1 : 0);
    if (b->evAfter) (void)hipEventRecord(b->evAfter, p.stream);
    if (G2P && RMAP == kMapLearned && la.branches != 0) {
        // the deferred points: map, store, and their P2G into the pass's output grid
        hipLaunchKernelGGL((k_batch_map<F32>), dim3(kMapBlocks), dim3(256), 0, p.stream, S, b->cases, mq.q, mq.count,
                           mq.count == b->mapCount ? b->mapCount + 1 : b->mapCount, b->grids + p.out * grid, b->gpitch,
                           b->err, la);
    }
}

template <bool F32, bool G2P, int RMAP>
void launch_one(icempm_batch *b, const Pass &p, const LearnArgs &la, const MapQueue &mq) {
    if constexpr (!F32)
        if (!b->inOrder) return launch_waves<F32, G2P, RMAP, 4, false>(b, p, la, mq);
    if (b->waves == 4)
        launch_waves<F32, G2P, RMAP, 4, true>(b, p, la, mq);
    else if (b->waves == 2)
        launch_waves<F32, G2P, RMAP, 2, true>(b, p, la, mq);
    else
        launch_waves<F32, G2P, RMAP, 1, true>(b, p, la, mq);
}

template <bool F32>
void launch_prec(icempm_batch *b, bool g2p, const Pass &p, const LearnArgs &la, const MapQueue &mq) {
    // the learned map with every branch switched off is the exact map: its
    // pass, without the queue logic and the learned map's counters
    if (!g2p)
        launch_one<F32, false, kMapExact>(b, p, la, mq);
    else if (b->rmap == kMapHarvest)
        launch_one<F32, true, kMapHarvest>(b, p, la, mq);
    else if (b->rmap == kMapLearned && b->mapBranches != 0)
        launch_one<F32, true, kMapLearned>(b, p, la, mq);
    else
        launch_one<F32, true, kMapExact>(b, p, la, mq);
}

// One substep of a range of chunks, or (g2p false) the first P2G (and,
// with the learned map, the map kernel after it).
hipError_t launch_pass(icempm_batch *b, bool g2p, const Pass &p) {
    if (p.chunks <= 0) return hipSuccess;
    LearnArgs la{};
    la.wbf = b->mlpW;
    la.pf = b->mlpP;
    la.norm = b->norm;
    la.tol = b->tol;
    la.hx = b->hx;
    la.ht = b->ht;
    la.hcount = b->hcount;
    la.hcap = b->hcap;
    la.stats = b->stats;
    la.branches = b->mapBranches;
    // the steps use the two queue counters in turn
    MapQueue mq{b->mapQ, b->mapCount ? b->mapCount + (p.step & 1) : nullptr, b->nPts};
    if (b->precision == ICEMPM_BATCH_F32)
        launch_prec<true>(b, g2p, p, la, mq);
    else
        launch_prec<false>(b, g2p, p, la, mq);
    return hipGetLastError();
}

// Chunks of n consecutive points with the given base cells (column | row <<
// 16), the first of them slot o: <= cap points whose cells span at most two
// cell rows and cols (<= kChunkCols) columns, so that the workgroup's LDS holds all their
// stencils, cut greedily.  A chunk that is cut for its columns alone ends at a
// wavefront's last point if it can.  Points in band order give chunks of one
// band each, until they move.  Returns the cells that the chunks span.
long cut_chunks(const unsigned *cells, int n, int o, int cap, int cols, std::vector<int> &starts) {
    starts.reserve((size_t)n / (size_t)cap + 16);
    long spanned = 0;
    for (int cs = 0; cs < n;) {
        int c0 = INT_MAX, r0 = INT_MAX, c1 = -1, r1 = -1, i = cs;
        bool wide = false;
        long area = 0;
        for (; i < n && i - cs < cap; ++i) {
            const int cc = (int)(cells[i] & 0xFFFFu), r = (int)(cells[i] >> 16);
            r0 = std::min(r0, r);
            r1 = std::max(r1, r);
            c0 = std::min(c0, cc);
            c1 = std::max(c1, cc);
            wide = c1 - c0 > cols - 1;
            if (r1 - r0 > 1 || wide) break;
            area = (long)(c1 - c0 + 1) * (r1 - r0 + 1);
        }
        spanned += area;
        if (wide && r1 - r0 <= 1 && i - cs > 64) i = cs + (i - cs) / 64 * 64;
        starts.push_back(o + cs);
        cs = i;
    }
    return spanned;
}

// Every case's chunks, from the case-local base cells of the points in slot order;
// returns the cells they span.  The cases are independent, so they are cut on
// several host threads.
long cut_cases(const icempm_batch *b, const unsigned *cells, int cap, int cols, std::vector<std::vector<int>> &starts) {
    const size_t nc = b->hc.size();
    std::vector<long> spanned(nc, 0);
    auto cut = [&](size_t ci) {
        const CaseParams &cp = b->hc[ci].cp;
        starts[ci].clear();
        if (cp.nPts > 0) spanned[ci] = cut_chunks(cells + cp.ptOffset, cp.nPts, cp.ptOffset, cap, cols, starts[ci]);
    };
    const unsigned hw = std::thread::hardware_concurrency();
    const size_t nt = std::min<size_t>(nc, std::min(16u, std::max(1u, hw)));
    if (nt <= 1 || b->nPts < (1 << 16)) {
        for (size_t ci = 0; ci < nc; ++ci) cut(ci);
    } else {
        // the calling thread works too; a helper that cannot be started
        // leaves its share to the others, and an exception (allocation)
        // in any of them is rethrown here, as the serial loop would throw
        // (the entry point's host_guard turns it into ICEMPM_E_HOST)
        std::atomic<size_t> next{0};
        std::exception_ptr failure;
        std::mutex failureLock;
        auto work = [&] {
            try {
                for (size_t ci; (ci = next.fetch_add(1)) < nc;) cut(ci);
            } catch (...) {
                std::lock_guard<std::mutex> g(failureLock);
                if (!failure) failure = std::current_exception();
            }
        };
        std::vector<std::thread> pool;
        for (size_t t = 1; t < nt; ++t) {
            try {
                pool.emplace_back(work);
            } catch (const std::system_error &) {
                break;
            }
        }
        work();
        for (auto &t : pool) t.join();
        if (failure) std::rethrow_exception(failure);
    }
    long all = 0;
    for (long a : spanned) all += a;
    return all;
}

// The chunks as b's host table.  A cloud of about a point a cell (kSparsePoints)
// in FP32 storage has chunks of one wavefront, no wider than its window: of the
// wider ones half the wavefronts have no points, or points past their window.
// 960 thousand points at 1, 0.8 and 0.5 a cell: 60 -> 51, 84 -> 55 and 167 -> 74 us a
// substep (the grid update and pass before: 56, 62 and 148).
constexpr double kSparsePoints = 1.15;
void chunk_table(icempm_batch *b, const unsigned *cells) {
    std::vector<int> &cstart = b->hcstart, &ccase = b->hccase;
    std::vector<std::vector<int>> starts(b->hc.size());
    const long spanned = cut_cases(b, cells, b->chunkPoints, kChunkCols, starts);
    b->hcdense = (double)b->nPts > kDensePoints * (double)spanned;
    if (b->precision == ICEMPM_BATCH_F32 && (double)b->nPts < kSparsePoints * (double)spanned)
        cut_cases(b, cells, std::min(b->chunkPoints, 64), kWinCols - 2, starts);
    cstart.clear();
    ccase.clear();
    for (size_t ci = 0; ci < starts.size(); ++ci)
        for (int st : starts[ci]) {
            cstart.push_back(st);
            ccase.push_back((int)ci);
        }
    cstart.push_back(b->nPts);
}

void drop_graph(icempm_batch *b) {
    for (auto &row : b->graphs)
        for (auto &g : row) {
            if (g.exec) (void)hipGraphExecDestroy(g.exec);
            g = icempm_batch::GraphSlot{};
        }
}


// The boxes of the chunks from the points as they are.
hipError_t launch_boxes(icempm_batch *b) {
    const dim3 nb((unsigned)((b->nChunks + 3) / 4));
    if (b->precision == ICEMPM_BATCH_F32)
        hipLaunchKernelGGL(k_chunk_boxes<true>, nb, dim3(256), 0, b->stream, b->recs, b->nChunks,
                           static_cast<const unsigned int *>(b->pos), b->pitch, b->cases, b->bounds, nullptr,
                           b->waves, b->inOrder ? 1 : 0);
    else
        hipLaunchKernelGGL(k_chunk_boxes<false>, nb, dim3(256), 0, b->stream, b->recs, b->nChunks,
                           static_cast<const double *>(b->pos), b->pitch, b->cases, b->bounds, nullptr,
                           b->waves, b->inOrder ? 1 : 0);
    return hipGetLastError();
}

// Wavefronts of a workgroup for the host chunk table's chunks.
int chunk_waves(const icempm_batch *b) {
    int most = 0;
    for (size_t c = 0; c < b->hccase.size(); ++c) most = std::max(most, b->hcstart[c + 1] - b->hcstart[c]);
    return most <= 64 ? 1 : (most <= 128 ? 2 : 4);
}

// Whether its chunks' points are in band order.
bool chunk_in_order(const icempm_batch *b) {
    return b->precision == ICEMPM_BATCH_F32 || b->hcdense || chunk_waves(b) < 4;
}

// The host chunk table as records on the device (grown when needed).  Boxes
// are made when a run starts afresh; a table rebuilt between two runs gets
// them here.
int upload_chunks(icempm_batch *b) {
    const size_t n = b->hccase.size();
    std::vector<ChunkRec> t(n);
    const int waves = chunk_waves(b);
    const bool inOrder = chunk_in_order(b);
    for (size_t c = 0; c < n; ++c) {
        const CaseParams &cp = b->hc[(size_t)b->hccase[c]].cp;
        const int count = b->hcstart[c + 1] - b->hcstart[c];
        t[c] = ChunkRec{b->hcstart[c], inOrder ? (unsigned)count : chunk_shape(count),
                        b->hccase[c], cp.gridOffset, (unsigned)cp.gx | (unsigned)cp.gy << 16, 0, 0, 0, {}};
    }
    const ChunkRec *before = b->recs;
    const int nBefore = b->nChunks;
    if (n > b->recCap) {
        // (where it cannot be had, the former table stays: any cut into chunks is correct)
        ChunkRec *recs = nullptr;
        BCHK(b, hipMalloc(&recs, n * sizeof(ChunkRec)), "chunk table");
        dfree(b->recs);
        b->recs = recs;
        b->recCap = n;
    }
    BCHK(b, hipMemcpy(b->recs, t.data(), n * sizeof(ChunkRec), hipMemcpyHostToDevice), "chunk table");
    b->nChunks = (int)n;
    const bool kernelBefore = b->waves == waves && b->inOrder == inOrder;
    b->waves = waves;
    b->inOrder = inOrder;
    // each group's first chunk
    bool splitMoved = false;
    for (int g = 0; g <= b->chains; ++g) {
        const int c = g == b->chains ? (int)n
                                     : (int)(std::lower_bound(b->hccase.begin(), b->hccase.end(), b->groupCase[g]) -
                                             b->hccase.begin());
        splitMoved = splitMoved || c != b->grpChunk[g];
        b->grpChunk[g] = c;
    }
    // a captured loop holds the table's address, the chunk count, the kernel
    // for their size and the groups' ranges (the grid sizes of its launches);
    // the table's contents are read at run time
    if (b->recs != before || b->nChunks != nBefore || !kernelBefore || splitMoved) drop_graph(b);
    if (b->pending >= 0) BCHK(b, launch_boxes(b), "chunk table");
    return ICEMPM_OK;
}

// the sort keys (batch-wide band keys) and slot indices of the current
// slots in sKeys / sVals
int sort_keys(icempm_batch *b) {
    const int n = b->nPts;
    BCHK(b, once(b->sKeys, (size_t)n * sizeof(int)), "keys");
    BCHK(b, once(b->sVals, (size_t)n * sizeof(int)), "keys");
    if (b->precision == ICEMPM_BATCH_F32)
        hipLaunchKernelGGL(k_batch_keys<unsigned int>, dim3((n + 255) / 256), dim3(256), 0, b->stream,
                           static_cast<const unsigned int *>(b->pos), b->pitch, n, b->cases, (int)b->hc.size(),
                           b->sKeys, b->sVals);
    else
        hipLaunchKernelGGL(k_batch_keys<double>, dim3((n + 255) / 256), dim3(256), 0, b->stream,
                           static_cast<const double *>(b->pos), b->pitch, n, b->cases, (int)b->hc.size(), b->sKeys,
                           b->sVals);
    BCHK(b, hipGetLastError(), "keys");
    return ICEMPM_OK;
}

// the base cells of the current slots (or of the slots in the given order), in
// b->hcells on the host
int current_cells(icempm_batch *b, const int *order = nullptr) {
    const int n = b->nPts;
    BCHK(b, once(b->dcells, (size_t)n * sizeof(unsigned)), "cells");
    if (!b->hcells) BCHK(b, hipHostMalloc(&b->hcells, (size_t)n * sizeof(unsigned), hipHostMallocDefault), "cells");
    if (b->precision == ICEMPM_BATCH_F32)
        hipLaunchKernelGGL(k_batch_cells<unsigned int>, dim3((n + 255) / 256), dim3(256), 0, b->stream,
                           static_cast<const unsigned int *>(b->pos), b->pitch, n, b->cases, (int)b->hc.size(),
                           order, b->dcells);
    else
        hipLaunchKernelGGL(k_batch_cells<double>, dim3((n + 255) / 256), dim3(256), 0, b->stream,
                           static_cast<const double *>(b->pos), b->pitch, n, b->cases, (int)b->hc.size(), order,
                           b->dcells);
    BCHK(b, hipGetLastError(), "cells");
    BCHK(b, hipMemcpyAsync(b->hcells, b->dcells, (size_t)n * sizeof(unsigned), hipMemcpyDeviceToHost, b->stream),
         "cells");
    BCHK(b, hipStreamSynchronize(b->stream), "cells");
    return ICEMPM_OK;
}

size_t pos_bytes(const icempm_batch *b) {
    return b->precision == ICEMPM_BATCH_F32 ? Rows<true>::kPosRows * b->pitch * sizeof(unsigned int)
                                             : Rows<false>::kPosRows * b->pitch * sizeof(double);
}

size_t rest_bytes(const icempm_batch *b) {
    return 11 * b->pitch * (b->precision == ICEMPM_BATCH_F32 ? sizeof(float) : sizeof(double));
}

// Element of rest value r (v0, v1, Fe00, Fe01, Fe10, Fe11, Bp00..Bp11, Jp_inv)
// of a slot: a row each, except FP32 storage's Fe, one 4-float record per
// slot in the space of rows 2-5.
size_t rest_elem(const icempm_batch *b, int r, size_t slot) {
    if (b->precision == ICEMPM_BATCH_F32 && r >= 2 && r <= 5) return 2 * b->pitch + 4 * slot + (size_t)(r - 2);
    return (size_t)r * b->pitch + slot;
}

// What a re-sort needs.
int resort_scratch(icempm_batch *b) {
    const size_t n = (size_t)b->nPts;
    BCHK(b, once(b->sKeys2, n * sizeof(int)), "re-sort");
    BCHK(b, once(b->sVals2, n * sizeof(int)), "re-sort");
    BCHK(b, once(b->sTmp, radix_tmp_ints(n) * sizeof(int)), "re-sort");
    BCHK(b, once(b->tpos, pos_bytes(b)), "re-sort");
    BCHK(b, once(b->trest, rest_bytes(b)), "re-sort");
    BCHK(b, once(b->tcrushed, b->pitch), "re-sort");
    BCHK(b, once(b->torig, b->pitch * sizeof(int)), "re-sort");
    if (b->grain) BCHK(b, once(b->tgrain, b->pitch * sizeof(short)), "re-sort");
    return ICEMPM_OK;
}

// Stable re-sort of every case's points by their current cell, then a new
// chunk table.  The slot -> batch-index map (orig) follows the points, so
// reads return them in their original order.
int resort(icempm_batch *b) {
    const int n = b->nPts;
    if (n <= 1) return ICEMPM_OK;
    int rc = sort_keys(b);
    if (rc) return rc;
    if ((rc = resort_scratch(b))) return rc;
    BCHK(b, radix_sort_pairs(b->sKeys, b->sVals, b->sKeys2, b->sVals2, (size_t)n, b->sTmp, b->stream), "re-sort");
    // the cells in sorted order give the new chunk table, whose chunks then
    // (FP64 storage) arrange their points
    if ((rc = current_cells(b, b->sVals))) return rc;
    chunk_table(b, b->hcells);
    if ((rc = upload_chunks(b))) return rc;
    const int *from = b->sVals;
    if (!b->inOrder) {
        hipLaunchKernelGGL(k_chunk_order, dim3((unsigned)b->nChunks), dim3(256), 0, b->stream, b->recs, b->nChunks,
                           b->sVals, b->sVals2);
        BCHK(b, hipGetLastError(), "re-sort");
        from = b->sVals2;
    }
    const unsigned nb = (unsigned)((n + 255) / 256);
    if (b->precision == ICEMPM_BATCH_F32) {
        Rows<true> a{static_cast<unsigned int *>(b->pos), reinterpret_cast<float *>(b->rest), b->crushed, b->grain,
                     b->pitch};
        Rows<true> t{static_cast<unsigned int *>(b->tpos), reinterpret_cast<float *>(b->trest), b->tcrushed,
                     b->tgrain, b->pitch};
        hipLaunchKernelGGL(k_batch_permute<true>, dim3(nb), dim3(256), 0, b->stream, a, t, b->orig, b->torig, from, n);
    } else {
        Rows<false> a{static_cast<double *>(b->pos), reinterpret_cast<double *>(b->rest), b->crushed, b->grain,
                      b->pitch};
        Rows<false> t{static_cast<double *>(b->tpos), reinterpret_cast<double *>(b->trest), b->tcrushed,
                      b->tgrain, b->pitch};
        hipLaunchKernelGGL(k_batch_permute<false>, dim3(nb), dim3(256), 0, b->stream, a, t, b->orig, b->torig, from, n);
    }
    BCHK(b, hipGetLastError(), "re-sort");
    BCHK(b, hipStreamSynchronize(b->stream), "re-sort");
    std::swap(b->pos, b->tpos);
    std::swap(b->rest, b->trest);
    std::swap(b->crushed, b->tcrushed);
    std::swap(b->grain, b->tgrain);
    std::swap(b->orig, b->torig);
    drop_graph(b);   // the captured launches hold the old row addresses
    b->pending = -1;   // a P2G in a grid scattered the points from their old slots
    return ICEMPM_OK;
}

// Scratch of read_points, for the largest case or kReadPart of its points: the
// device rows, the pinned rows they come down to and an event per group of rows.
int read_scratch(icempm_batch *b) {
    size_t pitch = 0;
    for (const auto &h : b->hc) pitch = std::max(pitch, ((size_t)h.cp.nPts + 63) / 64 * 64);
    pitch = std::min(pitch, (size_t)kReadPart);
    for (hipEvent_t &e : b->rbEvent)
        if (!e) BCHK(b, hipEventCreateWithFlags(&e, hipEventDisableTiming), "read_points");
    if (b->rbPitch >= pitch) return ICEMPM_OK;
    b->rbPitch = 0;
    dfree(b->rbDev);
    if (b->rbHost) (void)hipHostFree(b->rbHost);
    b->rbHost = nullptr;
    BCHK(b, hipMalloc(&b->rbDev, 14 * pitch * sizeof(double) + 64), "read_points");
    BCHK(b, hipHostMalloc(&b->rbHost, 14 * pitch * sizeof(double) + 64, hipHostMallocDefault), "read_points");
    b->rbPitch = pitch;
    return ICEMPM_OK;
}

// A case's points to the host: put in order on the device, brought down in
// groups of rows to pinned memory and copied to the caller's from there, a group
// while the next comes down.  What it takes is the caller's pages: 7 million
// points (32 cases, 0.9 GB) in 73 ms, where a copy per row and the ordering
// on the host took 192.  (Helper threads copy no faster: 84 ms with eight.)  A
// case of more than kReadPart points goes by parts of that many, which bounds the
// scratch (112 bytes a point on either side); the kernel looks at all slots for
// each, 4 bytes a slot.  The part is as small as costs later reads nothing, for
// pinning takes a first read longer than the copies: 1.4 million points, first and
// later read, 57 and 13 ms in parts of 2^20, 25 and 13 of 2^18, 20 and 14 of 2^17,
// 17 and 14 of 2^16, 16 and 15 of 2^15; 282 thousand 14 and 1.9, 14 and 1.9, 8.8
// and 1.9, 6.1 and 2.1, 4.7 and 2.4 (a copy per row: 51 and 50, 9 and 10).
int read_points(icempm_batch *b, int c, double *soa, size_t pitch) {
    const CaseParams &cp = b->hc[c].cp;
    std::lock_guard<std::mutex> lock(b->rbLock);
    int rc = read_scratch(b);
    if (rc) return rc;
    constexpr int kGroups = kReadGroups, kRows = 14;
    const auto group = [](int g) { return g * kRows / kGroups; };   // first row
    const size_t n = (size_t)cp.nPts;
    unsigned char *out = reinterpret_cast<unsigned char *>(soa);
    for (size_t first = 0; first < n; first += kReadPart) {
        const size_t count = std::min(n - first, (size_t)kReadPart), dp = (count + 63) / 64 * 64;   // points, pitch on the device
        int *bad = reinterpret_cast<int *>(b->rbDev + kRows * dp);
        BCHK(b, launch_fill_f64(b->rbDev, dp, 0.0, b->stream), "read_points");
        BCHK(b, launch_fill_i32(bad, 1, 0, b->stream), "read_points");
        const dim3 nb((unsigned)((n + 255) / 256));
        if (b->precision == ICEMPM_BATCH_F32) {
            Rows<true> S{static_cast<unsigned int *>(b->pos), reinterpret_cast<float *>(b->rest), b->crushed, b->grain, b->pitch};
            hipLaunchKernelGGL(k_read_points<true>, nb, dim3(256), 0, b->stream, S, b->orig, cp, (int)first, (int)dp, b->rbDev,
                               bad);
        } else {
            Rows<false> S{static_cast<double *>(b->pos), reinterpret_cast<double *>(b->rest), b->crushed, b->grain, b->pitch};
            hipLaunchKernelGGL(k_read_points<false>, nb, dim3(256), 0, b->stream, S, b->orig, cp, (int)first, (int)dp, b->rbDev,
                               bad);
        }
        BCHK(b, hipGetLastError(), "read_points");
        int *hostBad = reinterpret_cast<int *>(b->rbHost + kRows * dp);
        BCHK(b, hipMemcpyAsync(hostBad, bad, sizeof(int), hipMemcpyDeviceToHost, b->stream), "read_points");
        for (int g = 0; g < kGroups; ++g) {
            BCHK(b, hipMemcpyAsync(b->rbHost + group(g) * dp, b->rbDev + group(g) * dp,
                                   (size_t)(group(g + 1) - group(g)) * dp * sizeof(double), hipMemcpyDeviceToHost, b->stream),
                 "read_points");
            BCHK(b, hipEventRecord(b->rbEvent[g], b->stream), "read_points");
        }
        const bool end = first + count == n;   // the rows' padding with the last points
        const size_t pad = end ? (pitch - n) * sizeof(double) : 0;
        for (int g = 0; g < kGroups; ++g) {
            if (g == 1 && first == 0) std::memset(soa + pitch, 0, 2 * pitch * sizeof(double));   // P and Q: a batch keeps none
            BCHK(b, hipEventSynchronize(b->rbEvent[g]), "read_points");
            for (int d = group(g); d < group(g + 1); ++d) {
                const double *src = b->rbHost + (size_t)d * dp;
                if (d > 0) {
                    double *dst = soa + (size_t)(d + 2) * pitch + first;
                    std::memcpy(dst, src, count * sizeof(double));
                    std::memset(dst + count, 0, pad);
                } else {   // the flags, and the grain ids at byte pitch + 2 i
                    const unsigned char *u8 = reinterpret_cast<const unsigned char *>(src);
                    if (first == 0) std::memset(out, 0, pitch * sizeof(double));
                    std::memcpy(out + first, u8, count);
                    std::memcpy(out + pitch + 2 * first, u8 + dp, 2 * count);
                }
            }
        }
        BCHK(b, hipStreamSynchronize(b->stream), "read_points");
        if (*hostBad) return bfail(b, ICEMPM_E_STATE, "read_points: slot map corrupt");
    }
    return ICEMPM_OK;
}

// The chunk table for chunkPoints.  From rows, and where they may be wanted, the
// points are put in order anew, if there is memory for it: another cut of the same
// slots has chunks as wide as the former ones.
int rebuild_chunks(icempm_batch *b) {
    if (b->nPts > 1 && (!b->inOrder || (b->precision != ICEMPM_BATCH_F32 && b->chunkPoints == 256))) {
        if (resort_scratch(b) == ICEMPM_OK) return resort(b);
        (void)hipGetLastError();
    }
    int rc = current_cells(b);
    if (rc) return rc;
    chunk_table(b, b->hcells);
    return upload_chunks(b);
}

// The substep loop: n launches of the substep kernel (per group of cases).  A
// fresh start (start < 0) clears the grids and scatters the points into grid 0
// first; start = 0, 1 or 2 takes the P2G that the previous run's last pass
// left in that grid.  Substep i reads grid start + i, scatters into the next
// and clears the one after (mod 3).  renew: the boxes are renewed by the first
// substep and every kBoxEvery-th after it; else n is less than kBoxEvery and none
// does.  *end receives the grid that then holds the next substep's P2G.
hipError_t enqueue_loop(icempm_batch *b, int n, const double *tTab, double *hist, int start, bool renew, int *end) {
    hipError_t e;
    const size_t nc = b->hc.size();
    if ((e = launch_fill_f64(hist, 2 * (size_t)n * nc, 0.0, b->stream)) != hipSuccess) return e;
    if (b->mapCount &&
        (e = launch_fill_i32(reinterpret_cast<int *>(b->mapCount), 2, 0, b->stream)) != hipSuccess)
        return e;
    Pass p{};
    p.stream = b->stream;
    if (start < 0) {
        // what the grids hold, and where, is unknown at a fresh start
        start = 0;
        if ((e = launch_fill_f64(b->grids, 9 * b->gpitch, 0.0, b->stream)) != hipSuccess) return e;
        hipLaunchKernelGGL(k_reset_bounds, dim3((unsigned)((nc + 255) / 256)), dim3(256), 0, b->stream, b->bounds, (int)nc);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        if ((e = launch_boxes(b)) != hipSuccess) return e;
        p.chunks = b->nChunks;
        if ((e = launch_pass(b, false, p)) != hipSuccess) return e;
    }
    // The groups of cases as independent chains, when there are several,
    // the map kernel (one queue for all cases) is not in the loop and no
    // pass is being timed: the side chains start after everything above,
    // and the main stream waits for them at the end.
    const bool mapKernel = b->rmap == kMapLearned && b->mapBranches != 0;
    const int groups = (!mapKernel && b->timingStride <= 0 && b->nChunks >= kChainChunks) ? b->chains : 1;
    if (groups > 1) {
        if ((e = hipEventRecord(b->evFork, b->stream)) != hipSuccess) return e;
        for (int g = 1; g < groups; ++g)
            if ((e = hipStreamWaitEvent(b->side[g - 1], b->evFork, 0)) != hipSuccess) return e;
    }
    for (int g = 0; g < groups; ++g) {
        hipStream_t st = p.stream = g == 0 ? b->stream : b->side[g - 1];
        p.chunk0 = groups > 1 ? b->grpChunk[g] : 0;
        p.chunks = (groups > 1 ? b->grpChunk[g + 1] : b->nChunks) - p.chunk0;
        p.block0 = groups > 1 ? b->grpBlock[g] : 0;
        p.blocks = (groups > 1 ? b->grpBlock[g + 1] : b->nNodeBlocks) - p.block0;
        for (int i = 0; i < n; ++i) {
            p.in = (start + i) % 3;
            p.out = (start + i + 1) % 3;
            p.t = tTab + i;
            p.hist = hist + 2 * nc * (size_t)i;
            p.step = renew ? i : i + 1;
            const bool timeIt = b->timingStride > 0 && i % b->timingStride == 0;
            hipEvent_t t0 = nullptr, t1 = nullptr;
            if (timeIt) {
                if (b->tevNext + 2 > b->tev.size()) {
                    for (int q = 0; q < 2; ++q) {
                        hipEvent_t ev;
                        if ((e = hipEventCreate(&ev)) != hipSuccess) return e;
                        b->tev.push_back(ev);
                    }
                }
                t0 = b->tev[b->tevNext];
                t1 = b->tev[b->tevNext + 1];
                b->tevNext += 2;
                if ((e = hipEventRecord(t0, st)) != hipSuccess) return e;
            }
            b->evAfter = timeIt ? t1 : nullptr;   // recorded right after the particle kernel
            p.storeVB = (i == n - 1);
            e = launch_pass(b, true, p);
            b->evAfter = nullptr;
            if (e != hipSuccess) return e;
        }
    }
    for (int g = 1; g < groups; ++g) {
        if ((e = hipEventRecord(b->evJoin[g - 1], b->side[g - 1])) != hipSuccess) return e;
        if ((e = hipStreamWaitEvent(b->stream, b->evJoin[g - 1], 0)) != hipSuccess) return e;
    }
    *end = (start + n) % 3;
    return hipSuccess;
}

}  // namespace

// ---- one case on its context's own arrays -----------------------------------
namespace icempm {
namespace single {

static_assert(sizeof(ChunkRec) == kRecBytes && sizeof(CaseParams) <= kCaseBytes, "sizes of internal.h");

bool case_constants(const icy::SimParams &P, double x0, double y0, void *out) {
    // the substep kernel's premises: 16-bit cell indices, 32-bit byte offsets,
    // consistent cell sizes, numbers for the strengths
    if (P.nPts <= 0 || P.nPts >= 1 << 28 || P.GridX > 32767 || P.GridY > 32767 || P.GridTotal >= 1 << 28) return false;
    if (!(P.cellsize_inv == 1. / P.cellsize) || !(P.Dp_inv == 4. / (P.cellsize * P.cellsize))) return false;
    if (!(P.GrainVariability == P.GrainVariability)) return false;
    CaseParams c;
    fill_case(c, P);
    if (c.slope < 0) return false;   // its tension line is compared by squares
    c.x0 = x0;
    c.y0 = y0;
    std::memset(out, 0, kCaseBytes);
    std::memcpy(out, &c, sizeof(c));
    return true;
}

hipError_t plan(Run &r, int *keys, int *vals, int *keys2, int *vals2, int *tmp, std::vector<int> &starts) {
    const int n = r.n;
    hipLaunchKernelGGL(k_batch_keys<double>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, r.stream, r.pts + kRowPosX * r.pp,
                       r.pp, n, static_cast<const CaseParams *>(r.cp), 1, keys, vals);
    hipError_t e = radix_sort_pairs(keys, vals, keys2, vals2, (size_t)n, tmp, r.stream);
    if (e != hipSuccess) return e;
    const std::unique_ptr<int[]> hk(new int[(size_t)n]);
    if ((e = hipMemcpyAsync(hk.get(), keys, (size_t)n * sizeof(int), hipMemcpyDeviceToHost, r.stream)) != hipSuccess) return e;
    if ((e = hipStreamSynchronize(r.stream)) != hipSuccess) return e;
    // cut_chunks' cuts, for points that are in band order: a chunk's points lie
    // in one band, their columns ascending, so only its ends are looked at
    starts.clear();
    const auto fits = [&](int a, int b) {
        int xa, ya, xb, yb;
        band_cell(hk[(size_t)a], r.gx, r.gy, xa, ya);
        band_cell(hk[(size_t)b], r.gx, r.gy, xb, yb);
        return ya >> 1 == yb >> 1 && xb - xa <= kChunkCols - 1;
    };
    long spanned = 0;   // cells, of the keys from a chunk's first to its last
    for (int cs = 0; cs < n;) {
        starts.push_back(cs);
        int lo = cs + 1, hi = std::min(cs + 256, n);   // the chunk's end lies in [lo, hi]
        if (!fits(cs, hi - 1)) {
            while (lo < hi) {
                const int mid = (lo + hi) / 2;
                if (fits(cs, mid))
                    lo = mid + 1;
                else
                    hi = mid;
            }
        }
        spanned += hk[(size_t)hi - 1] - hk[(size_t)cs] + 1;
        cs = hi;
    }
    starts.push_back(n);
    r.inOrder = (double)n > kDensePoints * (double)spanned;
    return hipSuccess;
}

__global__ __launch_bounds__(256) void k_slots(const int *__restrict__ starts, const int *__restrict__ sorted,
                                               int *__restrict__ perm, int inOrder) {
    const int beg = starts[blockIdx.x], n = starts[blockIdx.x + 1] - beg, l = threadIdx.x;
    if (l < n) perm[beg + l] = sorted[beg + (inOrder ? l : chunk_point(l, chunk_shape(n)))];
}

hipError_t slots(const Run &r, const int *sorted, int *perm) {
    hipLaunchKernelGGL(k_slots, dim3((unsigned)r.nChunks), dim3(256), 0, r.stream, r.starts, sorted, perm,
                       r.inOrder ? 1 : 0);
    return hipGetLastError();
}

// The rows a substep reads and writes, from the points' own order to band
// order and back; v and Bp are not among them, since every substep makes its
// own, and P and Q are not touched.
__global__ __launch_bounds__(256) void k_pack(const double *__restrict__ pts, size_t pp, int n, const int *__restrict__ perm,
                                              double *__restrict__ rows) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    const int j = perm[k];
    rows[k] = pts[kRowPosX * pp + j];
    rows[pp + k] = pts[(kRowPosX + 1) * pp + j];
#pragma unroll
    for (int r = 0; r < 4; ++r) rows[(2 + r) * pp + k] = pts[(kRowFe00 + r) * pp + j];
    rows[6 * pp + k] = pts[kRowJp * pp + j];
    const unsigned char *u = reinterpret_cast<const unsigned char *>(pts + kRowUtil * pp);
    unsigned char *v = reinterpret_cast<unsigned char *>(rows + 7 * pp);
    v[k] = u[j];
    reinterpret_cast<short *>(v + pp)[k] = reinterpret_cast<const short *>(u + pp)[j];
}
__global__ __launch_bounds__(256) void k_unpack(const double *__restrict__ rows, size_t pp, int n,
                                                const int *__restrict__ perm, double *__restrict__ pts) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    const int j = perm[k];
    pts[kRowPosX * pp + j] = rows[k];
    pts[(kRowPosX + 1) * pp + j] = rows[pp + k];
#pragma unroll
    for (int r = 0; r < 4; ++r) pts[(kRowFe00 + r) * pp + j] = rows[(2 + r) * pp + k];
    pts[kRowJp * pp + j] = rows[6 * pp + k];
    reinterpret_cast<unsigned char *>(pts + kRowUtil * pp)[j] = reinterpret_cast<const unsigned char *>(rows + 7 * pp)[k];
}

hipError_t enter(const Run &r) {
    int4 *bounds = static_cast<int4 *>(r.bounds);
    hipLaunchKernelGGL(k_pack, dim3((unsigned)((r.n + 255) / 256)), dim3(256), 0, r.stream, r.pts, r.pp, r.n, r.perm, r.rows);
    hipLaunchKernelGGL(k_reset_bounds, dim3(1), dim3(64), 0, r.stream, bounds, 1);
    hipLaunchKernelGGL(k_chunk_boxes<false>, dim3((unsigned)((r.nChunks + 3) / 4)), dim3(256), 0, r.stream,
                       static_cast<ChunkRec *>(r.recs), r.nChunks, r.rows, r.pp, static_cast<const CaseParams *>(r.cp), bounds,
                       r.starts, 4, r.inOrder ? 1 : 0);
    return hipGetLastError();
}

hipError_t leave(const Run &r) {
    hipLaunchKernelGGL(k_unpack, dim3((unsigned)((r.n + 255) / 256)), dim3(256), 0, r.stream, r.rows, r.pp, r.n, r.perm, r.pts);
    return hipGetLastError();
}

hipError_t substep(const Run &r, const double *in, double *out, double *clear, double *hist2, double t, int step) {
    const int groups = ((r.nChunks + 7) / 8) * 8, blocks = (r.gx * r.gy + kNodeBlk - 1) / kNodeBlk;
    const NodeWork nw{nullptr, clear, hist2, r.bins};
    unsigned char *util = reinterpret_cast<unsigned char *>(r.rows + 7 * r.pp);
    // rows 2-5 of the kernel's 11 are Fe; without storeVB it takes no other
    const auto kernel = r.inOrder ? k_batch_substep<false, true, kMapSingle, 4, true>
                                  : k_batch_substep<false, true, kMapSingle, 4, false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(groups + blocks)), dim3(256), 0, r.stream,
                       static_cast<ChunkRec *>(r.recs), in, r.nChunks, groups, r.rows, r.rows, r.gp,
                       static_cast<const CaseParams *>(r.cp), util, r.pp, out, static_cast<int4 *>(r.bounds), r.err,
                       reinterpret_cast<const short *>(util + r.pp), r.rows + 6 * r.pp, nullptr, t, step, nw, LearnArgs{},
                       MapQueue{}, 0, 1);
    return hipGetLastError();
}

}  // namespace single
}  // namespace icempm

extern "C" {

int icempm_batch_create(icempm_batch **out, int precision) {
    return host_guard(nullptr, [&]() -> int {
        if (!out || (precision != ICEMPM_BATCH_F64 && precision != ICEMPM_BATCH_F32)) return ICEMPM_E_ARG;
        *out = nullptr;
        icempm_batch *b = new icempm_batch();
        b->precision = precision;
        hipError_t e = hipSetDevice(0);
        if (e == hipSuccess) e = hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&b->evFork, hipEventDisableTiming);
        for (int g = 0; g + 1 < icempm_batch::kChains && e == hipSuccess; ++g) {
            e = hipStreamCreateWithFlags(&b->side[g], hipStreamNonBlocking);
            if (e == hipSuccess) e = hipEventCreateWithFlags(&b->evJoin[g], hipEventDisableTiming);
        }
        if (e == hipSuccess) e = hipEventCreate(&b->e0);
        if (e == hipSuccess) e = hipEventCreate(&b->e1);
        if (e != hipSuccess) {
            icempm_batch_destroy(b);
            return ICEMPM_E_HIP;
        }
        *out = b;
        return ICEMPM_OK;
    });
}

void icempm_batch_destroy(icempm_batch *b) {
    if (!b) return;
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    for (hipStream_t st : b->side)
        if (st) (void)hipStreamSynchronize(st);
    drop_graph(b);
    dfree(b->pos); dfree(b->rest); dfree(b->crushed); dfree(b->grids); dfree(b->bounds);
    dfree(b->cases); dfree(b->recs); dfree(b->nodeBlock);
    dfree(b->err); dfree(b->tTab); dfree(b->hist);
    dfree(b->mlpW); dfree(b->mlpP); dfree(b->hx); dfree(b->ht); dfree(b->hcount); dfree(b->stats);
    dfree(b->mapQ); dfree(b->mapCount);
    dfree(b->dcells);
    if (b->hcells) (void)hipHostFree(b->hcells);
    dfree(b->rbDev);
    if (b->rbHost) (void)hipHostFree(b->rbHost);
    for (hipEvent_t ev : b->rbEvent)
        if (ev) (void)hipEventDestroy(ev);
    b->hcells = nullptr;
    dfree(b->orig); dfree(b->sKeys); dfree(b->sVals); dfree(b->sKeys2); dfree(b->sVals2); dfree(b->sTmp);
    dfree(b->tpos); dfree(b->trest); dfree(b->tcrushed); dfree(b->torig);
    dfree(b->kpos); dfree(b->krest); dfree(b->kcrushed); dfree(b->korig);
    dfree(b->grain); dfree(b->tgrain); dfree(b->kgrain); dfree(b->bins);
    for (hipEvent_t ev : b->tev) (void)hipEventDestroy(ev);
    if (b->e0) (void)hipEventDestroy(b->e0);
    if (b->e1) (void)hipEventDestroy(b->e1);
    if (b->evFork) (void)hipEventDestroy(b->evFork);
    for (hipEvent_t ev : b->evJoin)
        if (ev) (void)hipEventDestroy(ev);
    for (hipStream_t st : b->side)
        if (st) (void)hipStreamDestroy(st);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    delete b;
}

const char *icempm_batch_last_error(const icempm_batch *b) { return b ? b->lastError.c_str() : ""; }

int icempm_batch_add_case(icempm_batch *b, const void *simparams, size_t nbytes, const double *soa,
                          size_t pitch) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b || !simparams || !soa || nbytes != sizeof(icy::SimParams)) return -ICEMPM_E_ARG;
        if (b->finalized) return -bfail(b, ICEMPM_E_STATE, "add_case: batch already finalized");
        icy::SimParams P;
        std::memcpy(&P, simparams, sizeof(P));
        if (P.nPts <= 0 || (size_t)P.nPts > pitch || P.GridX <= 0 || P.GridY <= 0)
            return -bfail(b, ICEMPM_E_ARG, "add_case: bad sizes");
        if (P.GridX > 32767 || P.GridY > 32767)   // cell indices travel as 16-bit halves in the particle pass
            return -bfail(b, ICEMPM_E_ARG, "add_case: grid wider or taller than 32767 cells");
        // the case's grid slice, its node blocks and every node index the kernels
        // form (X + Y * GridX) are sized from GridTotal: it must be the product
        if ((long)P.GridTotal != (long)P.GridX * (long)P.GridY)
            return -bfail(b, ICEMPM_E_ARG, "add_case: GridTotal is not GridX * GridY");
        // the stencils use cellsize_inv, the weights and stresses cellsize and dt
        // (derived as in ComputeHelperVariables, parameters_sim.cpp:131-133)
        if (!(P.cellsize > 0) || !(P.InitialTimeStep > 0) || !(P.cellsize_inv == 1. / P.cellsize) ||
            !(P.Dp_inv == 4. / (P.cellsize * P.cellsize)))
            return -bfail(b, ICEMPM_E_ARG, "add_case: cellsize, cellsize_inv, Dp_inv and dt must be positive and consistent");
        if (!(P.GrainVariability == P.GrainVariability))
            return -bfail(b, ICEMPM_E_ARG, "add_case: GrainVariability is NaN");
        if (P.n_indenter_subdivisions <= 0 || P.n_indenter_subdivisions > 1 << 16)
            return -bfail(b, ICEMPM_E_ARG, "add_case: n_indenter_subdivisions out of range");
        if (!b->hc.empty() && P.InitialTimeStep != b->hc[0].cp.dt)
            return -bfail(b, ICEMPM_E_ARG, "add_case: all cases of a batch share one time step");
        icempm_batch::HostCase h{};
        CaseParams &c = h.cp;
        fill_case(c, P);
        const int n = P.nPts;
        h.pos.resize(2 * (size_t)n);
        h.rest.resize(11 * (size_t)n);
        h.crushed.resize(n);
        h.grain.resize(n);
        h.keys.resize(n);
        const unsigned char *u8 = reinterpret_cast<const unsigned char *>(soa);
        for (int i = 0; i < n; ++i) {
            h.pos[i] = soa[pitch * 4 + i];
            h.pos[n + i] = soa[pitch * 5 + i];
            for (int r = 0; r < 10; ++r) h.rest[(size_t)r * n + i] = soa[pitch * (6 + r) + i];
            h.rest[10 * (size_t)n + i] = soa[pitch * 3 + i];
            h.crushed[i] = u8[i];
            std::memcpy(&h.grain[i], u8 + pitch + 2 * (size_t)i, sizeof(short));   // point.cpp:19-23
            // the base cell's band key, clamped into the grid as on the device
            const double x = h.pos[i], y = h.pos[n + i];
            int key = c.gridTotal - 1;
            if (x == x && y == y) {
                const double bx = std::fmin(std::fmax(x * c.h_inv - 0.5, 0.0), (double)(c.gx - 1));
                const double by = std::fmin(std::fmax(y * c.h_inv - 0.5, 0.0), (double)(c.gy - 1));
                key = band_key((int)bx, (int)by, c.gx, c.gy);
            }
            h.keys[i] = key;
        }
        b->hc.push_back(std::move(h));
        return (int)b->hc.size() - 1;
    });
}

int icempm_batch_finalize(icempm_batch *b) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b || b->hc.empty()) return ICEMPM_E_ARG;
        if (b->finalized) return bfail(b, ICEMPM_E_STATE, "finalize: already finalized");
        // point and node offsets, node-block table, keys of the points in slot order
        std::vector<int2> nblk;
        std::vector<int> keys;
        long pofs = 0, gofs = 0, bofs = 0;
        bool anyGrains = false;
        // every case's points in band order (stable): slot o + k holds point
        // order[k] of the case, and orig maps it back
        std::vector<std::vector<int>> order(b->hc.size());
        for (size_t ci = 0; ci < b->hc.size(); ++ci) {
            auto &h = b->hc[ci];
            h.cp.ptOffset = (int)pofs;
            h.cp.gridOffset = (int)gofs;
            h.cp.binOffset = (int)bofs;
            bofs += 2 * (long)h.cp.nbins;
            anyGrains = anyGrains || h.cp.grainVar != 0;
            auto &ord = order[ci];
            ord.resize((size_t)h.cp.nPts);
            for (int i = 0; i < h.cp.nPts; ++i) ord[(size_t)i] = i;
            std::stable_sort(ord.begin(), ord.end(), [&h](int a, int c) { return h.keys[(size_t)a] < h.keys[(size_t)c]; });
            for (int k = 0; k < h.cp.nPts; ++k) keys.push_back(h.keys[(size_t)ord[(size_t)k]]);
            for (int nd = 0; nd < h.cp.gridTotal; nd += kNodeBlk) nblk.push_back(make_int2((int)ci, nd));
            pofs += h.cp.nPts;
            gofs += h.cp.gridTotal;
        }
        // the particle pass addresses rows through 32-bit byte offsets
        if (pofs >= (1L << 29) || gofs >= (1L << 29) || bofs > INT_MAX / 2)
            return bfail(b, ICEMPM_E_ARG, "finalize: batch too large (2^29 points or grid nodes at most)");
        // a base cell packs its column and row into 16 bits each
        for (const auto &h : b->hc)
            if (h.cp.gx > 65536 || h.cp.gy > 65536)
                return bfail(b, ICEMPM_E_ARG, "finalize: a case's grid is wider or taller than 65536 nodes");
        b->binsTotal = (int)bofs;
        b->nPts = (int)pofs;
        b->nNodes = gofs;
        b->nNodeBlocks = (int)nblk.size();
        // the groups of cases: group g starts at the case boundary nearest to
        // g / chains of all points (each group non-empty)
        {
            const int nc = (int)b->hc.size();
            b->chains = std::max(1, std::min(icempm_batch::kChains, nc));
            b->groupCase[0] = 0;
            long acc = 0;   // points of the cases before case k
            int k = 0;
            for (int g = 1; g < b->chains; ++g) {
                const long target = (long)g * pofs;   // in units of 1 / chains points
                if (k <= b->groupCase[g - 1]) {
                    acc += b->hc[k].cp.nPts;
                    ++k;
                }
                while (k < nc - (b->chains - g) &&
                       std::labs((acc + b->hc[k].cp.nPts) * b->chains - target) <= std::labs(acc * b->chains - target)) {
                    acc += b->hc[k].cp.nPts;
                    ++k;
                }
                b->groupCase[g] = k;
            }
            b->groupCase[b->chains] = nc;
            for (int g = 0; g <= b->chains; ++g) {
                int kb = (int)nblk.size();
                for (size_t q = 0; q < nblk.size(); ++q)
                    if (nblk[q].x >= b->groupCase[g]) {
                        kb = (int)q;
                        break;
                    }
                b->grpBlock[g] = kb;
            }
        }
        b->pitch = (pofs + 63) / 64 * 64;
        b->gpitch = ((size_t)gofs + 63) / 64 * 64;
        {
            // the cells of the band keys, case-local (the key of a cell is
            // band_key of its column and row)
            std::vector<unsigned> cells(keys.size());
            for (size_t ci = 0; ci < b->hc.size(); ++ci) {
                const CaseParams &cp = b->hc[ci].cp;
                for (int k = 0; k < cp.nPts; ++k) {
                    int cx, cy;
                    band_cell(keys[(size_t)cp.ptOffset + k], cp.gx, cp.gy, cx, cy);
                    cells[(size_t)cp.ptOffset + k] = (unsigned)cx | (unsigned)cy << 16;
                }
            }
            chunk_table(b, cells.data());
            // every chunk's points in its slot order, where that is not band order
            const bool inOrder = chunk_in_order(b);
            std::vector<int> sorted;
            for (size_t c = 0; c < b->hccase.size() && !inOrder; ++c) {
                std::vector<int> &ord = order[(size_t)b->hccase[c]];
                const int o = b->hc[(size_t)b->hccase[c]].cp.ptOffset;
                const int p = b->hcstart[c] - o, n = b->hcstart[c + 1] - b->hcstart[c];
                sorted.assign(ord.begin() + p, ord.begin() + p + n);
                for (int l = 0; l < n; ++l) ord[(size_t)(p + l)] = sorted[(size_t)chunk_point(l, chunk_shape(n))];
            }
        }
        const size_t vs = b->precision == ICEMPM_BATCH_F32 ? sizeof(float) : sizeof(double);
        BCHK(b, hipMalloc(&b->pos, pos_bytes(b)), "batch finalize");
        BCHK(b, hipMalloc(&b->rest, 11 * b->pitch * vs), "batch finalize");
        BCHK(b, hipMalloc(&b->crushed, b->pitch), "batch finalize");
        if (anyGrains) BCHK(b, hipMalloc(&b->grain, b->pitch * sizeof(short)), "batch finalize");
        BCHK(b, hipMalloc(&b->bins, (size_t)b->binsTotal * sizeof(double)), "batch finalize");
        BCHK(b, hipMalloc(&b->orig, b->pitch * sizeof(int)), "batch finalize");
        BCHK(b, hipMalloc(&b->grids, 9 * b->gpitch * sizeof(double)), "batch finalize");
        BCHK(b, hipMalloc(&b->bounds, b->hc.size() * sizeof(int4)), "batch finalize");
        BCHK(b, hipMalloc(&b->cases, b->hc.size() * sizeof(CaseParams)), "batch finalize");
        BCHK(b, hipMalloc(&b->nodeBlock, nblk.size() * sizeof(int2)), "batch finalize");
        BCHK(b, hipMalloc(&b->err, sizeof(int)), "batch finalize");
        BCHK(b, hipMalloc(&b->hcount, sizeof(unsigned long long)), "batch finalize");
        BCHK(b, hipMalloc(&b->stats, kMapStats * sizeof(unsigned long long)), "batch finalize");
        // host staging in the device layout
        std::vector<double> hpos(2 * b->pitch, 0.0);
        std::vector<unsigned char> hrest(11 * b->pitch * vs, 0), hcr(b->pitch, 0);
        std::vector<short> hgr(b->pitch, 0);
        std::vector<int> horig(b->pitch, 0);
        std::vector<CaseParams> hcp;
        for (size_t ci = 0; ci < b->hc.size(); ++ci) {
            const auto &h = b->hc[ci];
            const int n = h.cp.nPts, o = h.cp.ptOffset;
            for (int k = 0; k < n; ++k) {
                const int i = order[ci][(size_t)k];
                hpos[o + k] = h.pos[i];
                hpos[b->pitch + o + k] = h.pos[n + i];
                hcr[o + k] = h.crushed[i];
                hgr[o + k] = h.grain[i];
                horig[o + k] = o + i;
                for (int r = 0; r < 11; ++r) {
                    double v = h.rest[(size_t)r * n + i];
                    if (b->precision == ICEMPM_BATCH_F32) {
                        if (r == 2 || r == 5 || r == 10) v -= 1.0;    // Fe00, Fe11, Jp_inv stored less 1
                        float f = (float)v;
                        std::memcpy(&hrest[rest_elem(b, r, (size_t)(o + k)) * vs], &f, vs);
                    } else {
                        std::memcpy(&hrest[rest_elem(b, r, (size_t)(o + k)) * vs], &v, vs);
                    }
                }
            }
            hcp.push_back(h.cp);
        }
        if (b->precision == ICEMPM_BATCH_F32) {
            // one record per slot: 48-bit fixed point (high words of x and y,
            // both low halves) and the crushed flag
            std::vector<unsigned int> q(4 * b->pitch, 0u);
            for (size_t ci = 0; ci < hcp.size(); ++ci) {
                const CaseParams &cp = hcp[ci];
                for (int k = 0; k < cp.nPts; ++k) {
                    const size_t i = (size_t)cp.ptOffset + k;
                    unsigned int hx, lx, hy, ly;
                    fix48_put(hpos[i], cp, hx, lx);
                    fix48_put(hpos[b->pitch + i], cp, hy, ly);
                    q[4 * i] = hx;
                    q[4 * i + 1] = hy;
                    q[4 * i + 2] = lx | (ly << 16);
                    q[4 * i + 3] = hcr[i] | ((unsigned int)(unsigned short)hgr[i] << 16);
                }
            }
            BCHK(b, hipMemcpy(b->pos, q.data(), q.size() * sizeof(unsigned int), hipMemcpyHostToDevice), "batch upload");
        } else {
            BCHK(b, hipMemcpy(b->pos, hpos.data(), hpos.size() * sizeof(double), hipMemcpyHostToDevice), "batch upload");
        }
        BCHK(b, hipMemcpy(b->rest, hrest.data(), hrest.size(), hipMemcpyHostToDevice), "batch upload");
        BCHK(b, hipMemcpy(b->crushed, hcr.data(), hcr.size(), hipMemcpyHostToDevice), "batch upload");
        if (b->grain)
            BCHK(b, hipMemcpy(b->grain, hgr.data(), hgr.size() * sizeof(short), hipMemcpyHostToDevice), "batch upload");
        {
            const std::vector<double> zb((size_t)b->binsTotal, 0.0);
            BCHK(b, hipMemcpy(b->bins, zb.data(), zb.size() * sizeof(double), hipMemcpyHostToDevice), "batch upload");
        }
        BCHK(b, hipMemcpy(b->orig, horig.data(), horig.size() * sizeof(int), hipMemcpyHostToDevice), "batch upload");
        BCHK(b, hipMemcpy(b->cases, hcp.data(), hcp.size() * sizeof(CaseParams), hipMemcpyHostToDevice), "batch upload");
        BCHK(b, hipMemcpy(b->nodeBlock, nblk.data(), nblk.size() * sizeof(int2), hipMemcpyHostToDevice), "batch upload");
        int zero = 0;
        BCHK(b, hipMemcpy(b->err, &zero, sizeof(int), hipMemcpyHostToDevice), "batch upload");
        const unsigned long long z7[kMapStats] = {};
        BCHK(b, hipMemcpy(b->hcount, z7, sizeof(unsigned long long), hipMemcpyHostToDevice), "batch upload");
        BCHK(b, hipMemcpy(b->stats, z7, sizeof(z7), hipMemcpyHostToDevice), "batch upload");
        int rc = upload_chunks(b);
        if (rc) return rc;
        b->finalized = true;
        return ICEMPM_OK;
    });
}

}  // extern "C"

namespace {

// n substeps with the given time table and force-history rows, from the
// P2G the previous run left (b->pending) or from a fresh P2G, as one graph
// launch (captured when the start, the step count or the pointers change)
// or as stream launches; returns the device time in ms.
// The executable graph of n substeps from the given start (-1 fresh, 0, 1 or
// 2: the P2G in that grid, the boxes renewed or not) with these time-table and
// history rows, captured, instantiated and put on the device unless its slot
// already holds it.
int ensure_graph(icempm_batch *b, int n, const double *tTab, double *hist, int start,
                 bool renew, const icempm_batch::GraphSlot **out) {
    icempm_batch::GraphSlot *row = b->graphs[renew ? start + 1 : start + 4];
    for (int w = 0; w < 2; ++w)
        if (row[w].exec && row[w].steps == n && row[w].T == tTab && row[w].H == hist) {
            row[w].used = ++b->graphTick;
            if (out) *out = &row[w];
            return ICEMPM_OK;
        }
    icempm_batch::GraphSlot &g = row[row[0].used <= row[1].used ? 0 : 1];
    if (g.exec) (void)hipGraphExecDestroy(g.exec);
    g = icempm_batch::GraphSlot{};
    hipGraph_t graph = nullptr;
    int end = -1;
    BCHK(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal), "batch capture");
    hipError_t e = enqueue_loop(b, n, tTab, hist, start, renew, &end);
    hipError_t e2 = hipStreamEndCapture(b->stream, &graph);
    if (e != hipSuccess) {
        if (graph) (void)hipGraphDestroy(graph);
        return bfail(b, ICEMPM_E_HIP, std::string("batch capture: ") + hipGetErrorString(e));
    }
    BCHK(b, e2, "batch capture");
    e = hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    BCHK(b, e, "batch graph instantiate");
    g.steps = n;
    g.T = tTab;
    g.H = hist;
    g.end = end;
    g.used = ++b->graphTick;
    if (out) *out = &g;
    // put the executable graph on the device now, so that its first launch
    // costs what a replay costs
    BCHK(b, hipGraphUpload(g.exec, b->stream), "batch graph upload");
    BCHK(b, hipStreamSynchronize(b->stream), "batch graph upload");
    return ICEMPM_OK;
}

// the time-table and history buffers for runs of up to n substeps
int ensure_capacity(icempm_batch *b, int n) {
    if (n <= b->cap) return ICEMPM_OK;
    drop_graph(b);
    dfree(b->tTab);
    dfree(b->hist);
    b->cap = 0;
    BCHK(b, hipMalloc(&b->tTab, (size_t)n * sizeof(double)), "batch run");
    BCHK(b, hipMalloc(&b->hist, 2 * b->hc.size() * (size_t)n * sizeof(double)), "batch run");
    b->cap = n;
    return ICEMPM_OK;
}

// Runs this short may leave the boxes to a later one: renewing them costs a
// substep of 6.4M points 25 us, each time for runs of one substep.  A longer run
// gains less than the second set of graphs costs it.
constexpr int kShortRun = kBoxEvery / 2;

int run_segment(icempm_batch *b, int n, int use_graph, const double *tTab, double *hist, float *ms) {
    b->tevNext = 0;
    const int start = b->pending;
    const bool renew = start < 0 || n > kShortRun || b->boxAge + n > kBoxEvery;
    b->pending = -1;   // until the loop below is enqueued whole
    int end = -1;
    if (use_graph) {
        const icempm_batch::GraphSlot *g = nullptr;
        const int rc = ensure_graph(b, n, tTab, hist, start, renew, &g);
        if (rc) return rc;
        end = g->end;
        // timed from here: capture and instantiation are host work before it
        BCHK(b, hipEventRecord(b->e0, b->stream), "batch run");
        BCHK(b, hipGraphLaunch(g->exec, b->stream), "batch graph launch");
    } else {
        BCHK(b, hipEventRecord(b->e0, b->stream), "batch run");
        BCHK(b, enqueue_loop(b, n, tTab, hist, start, renew, &end), "batch run");
    }
    BCHK(b, hipEventRecord(b->e1, b->stream), "batch run");
    BCHK(b, hipEventSynchronize(b->e1), "batch run");
    b->pending = end;
    b->boxAge = renew ? (n - 1) % kBoxEvery + 1 : b->boxAge + n;
    BCHK(b, hipEventElapsedTime(ms, b->e0, b->e1), "batch run");
    for (size_t q = 0; q + 1 < b->tevNext; q += 2) {
        float kms = 0;
        BCHK(b, hipEventElapsedTime(&kms, b->tev[q], b->tev[q + 1]), "batch timing");
        b->timedMs += kms;
        b->timedLaunches += 1;
    }
    b->tevNext = 0;
    return ICEMPM_OK;
}

}  // namespace

extern "C" {

int icempm_batch_run(icempm_batch *b, int n, int use_graph) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b || n <= 0) return ICEMPM_E_ARG;
        if (!b->finalized) return bfail(b, ICEMPM_E_STATE, "run: batch not finalized");
        if (use_graph && b->timingStride > 0)
            return bfail(b, ICEMPM_E_STATE, "run: kernel timing needs stream launches (use_graph = 0)");
        const size_t nc = b->hc.size();
        int rc0 = ensure_capacity(b, n);
        if (rc0) return rc0;
        // the time of each substep by repeated addition (model.cpp:23)
        std::vector<double> tt((size_t)n);
        double t = b->t;
        for (int i = 0; i < n; ++i) {
            t += b->hc[0].cp.dt;
            tt[i] = t;
        }
        BCHK(b, hipMemcpyAsync(b->tTab, tt.data(), n * sizeof(double), hipMemcpyHostToDevice, b->stream), "batch run");
        // the force bins sum over the run (Model::Step sums them over a cycle, model.cpp:18)
        BCHK(b, launch_fill_f64(b->bins, (size_t)b->binsTotal, 0.0, b->stream), "batch run");
        BCHK(b, hipStreamSynchronize(b->stream), "batch run");
        // segments of resortEvery substeps, the points re-sorted between them
        const int seg = b->resortEvery > 0 ? b->resortEvery : n;
        double total = 0;
        for (int s0 = 0; s0 < n; s0 += seg) {
            if (s0 > 0) {
                const auto h0 = std::chrono::steady_clock::now();
                int rc = resort(b);
                if (rc) return rc;
                total += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - h0).count();
            }
            const int len = std::min(seg, n - s0);
            float ms = 0;
            const auto h0 = std::chrono::steady_clock::now();
            int rc = run_segment(b, len, use_graph, b->tTab + s0, b->hist + 2 * nc * (size_t)s0, &ms);
            if (rc) return rc;
            // with re-sorting, each segment is captured anew: count the host time
            total += b->resortEvery > 0 ? std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - h0).count()
                                        : (double)ms;
        }
        b->lastMs = (float)total;
        b->t = t;
        b->step += n;
        b->lastRun = n;
        return ICEMPM_OK;
    });
}

int icempm_batch_prepare(icempm_batch *b, int n) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b || n <= 0) return ICEMPM_E_ARG;
        if (!b->finalized) return bfail(b, ICEMPM_E_STATE, "prepare: batch not finalized");
        BCHK(b, hipStreamSynchronize(b->stream), "prepare");
        int rc = ensure_capacity(b, n);
        if (rc) return rc;
        // the first segment of such a run, from each of the four starts
        const int len = b->resortEvery > 0 ? std::min(b->resortEvery, n) : n;
        for (int start = -1; start <= 2; ++start) {
            if ((rc = ensure_graph(b, len, b->tTab, b->hist, start, true, nullptr))) return rc;
            if (start >= 0 && len <= kShortRun && (rc = ensure_graph(b, len, b->tTab, b->hist, start, false, nullptr))) return rc;
        }
        return ICEMPM_OK;
    });
}

int icempm_batch_last_ms(const icempm_batch *b, float *ms) {
    if (!b || !ms) return ICEMPM_E_ARG;
    *ms = b->lastMs;
    return ICEMPM_OK;
}

int icempm_batch_num_points(const icempm_batch *b) { return b ? b->nPts : 0; }

long icempm_batch_num_nodes(const icempm_batch *b) { return b ? b->nNodes : 0; }

int icempm_batch_kernel_timing(icempm_batch *b, int stride) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b || stride < 0) return ICEMPM_E_ARG;
        b->timingStride = stride;
        b->timedMs = 0;
        b->timedLaunches = 0;
        return ICEMPM_OK;
    });
}

int icempm_batch_kernel_timing_read(icempm_batch *b, double *total_ms, int *launches) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b || !total_ms || !launches) return ICEMPM_E_ARG;
        *total_ms = b->timedMs;
        *launches = b->timedLaunches;
        return ICEMPM_OK;
    });
}

int icempm_batch_force_history(icempm_batch *b, int c, double *out, int n) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b || !out || c < 0 || (size_t)c >= b->hc.size() || n < 0 || n > b->lastRun) return ICEMPM_E_ARG;
        const size_t nc = b->hc.size();
        std::vector<double> all(2 * nc * (size_t)n);
        if (n == 0) return ICEMPM_OK;
        BCHK(b, hipMemcpy(all.data(), b->hist, all.size() * sizeof(double), hipMemcpyDeviceToHost), "force history");
        for (int i = 0; i < n; ++i) {
            out[2 * i] = all[(size_t)i * 2 * nc + 2 * c];
            out[2 * i + 1] = all[(size_t)i * 2 * nc + 2 * c + 1];
        }
        return ICEMPM_OK;
    });
}

int icempm_batch_force_bins(icempm_batch *b, int c, double *out, int nbins) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b || !out || c < 0 || (size_t)c >= b->hc.size()) return ICEMPM_E_ARG;
        if (!b->finalized) return bfail(b, ICEMPM_E_STATE, "force_bins: batch not finalized");
        const CaseParams &cp = b->hc[c].cp;
        if (nbins != cp.nbins) return bfail(b, ICEMPM_E_ARG, "force_bins: nbins is not the case's n_indenter_subdivisions");
        BCHK(b, hipStreamSynchronize(b->stream), "force_bins");
        BCHK(b, hipMemcpy(out, b->bins + cp.binOffset, 2 * (size_t)nbins * sizeof(double), hipMemcpyDeviceToHost),
             "force_bins");
        return ICEMPM_OK;
    });
}

int icempm_batch_read_points(icempm_batch *b, int c, double *soa, size_t pitch) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b || !soa || c < 0 || (size_t)c >= b->hc.size()) return ICEMPM_E_ARG;
        if (!b->finalized) return bfail(b, ICEMPM_E_STATE, "read_points: batch not finalized");
        if ((size_t)b->hc[c].cp.nPts > pitch) return bfail(b, ICEMPM_E_ARG, "read_points: pitch too small");
        return read_points(b, c, soa, pitch);
    });
}

int icempm_batch_error_flag(icempm_batch *b, int *flag) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b || !flag) return ICEMPM_E_ARG;
        BCHK(b, hipMemcpy(flag, b->err, sizeof(int), hipMemcpyDeviceToHost), "error flag");
        return ICEMPM_OK;
    });
}

int icempm_batch_set_return_map(icempm_batch *b, int mode, const float *params, const float *norm,
                                double tol, int harvest_capacity) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b) return ICEMPM_E_ARG;
        if (!b->finalized) return bfail(b, ICEMPM_E_STATE, "set_return_map: batch not finalized");
        if (mode != kMapExact && mode != kMapHarvest && mode != kMapLearned)
            return bfail(b, ICEMPM_E_ARG, "set_return_map: unknown mode");
        if (mode == kMapHarvest && harvest_capacity <= 0)
            return bfail(b, ICEMPM_E_ARG, "set_return_map: harvest needs a positive capacity");
        if (mode == kMapLearned && (!params || !norm))
            return bfail(b, ICEMPM_E_ARG, "set_return_map: the learned map needs parameters and a normalisation");
        if (mode == kMapLearned && !(tol == tol))
            return bfail(b, ICEMPM_E_ARG, "set_return_map: tolerance is NaN");
        BCHK(b, hipStreamSynchronize(b->stream), "set_return_map");
        // a captured loop holds the previous kernel arguments
        drop_graph(b);
        if (mode == kMapHarvest) {
            if (harvest_capacity != b->hcap) {
                dfree(b->hx);
                dfree(b->ht);
                b->hcap = 0;
                BCHK(b, hipMalloc(&b->hx, (size_t)harvest_capacity * 5 * sizeof(float)), "set_return_map");
                BCHK(b, hipMalloc(&b->ht, (size_t)harvest_capacity * 3 * sizeof(float)), "set_return_map");
                b->hcap = harvest_capacity;
            }
            const unsigned long long zero = 0;
            BCHK(b, hipMemcpy(b->hcount, &zero, sizeof(zero), hipMemcpyHostToDevice), "set_return_map");
        }
        if (mode == kMapLearned) {
            const int np = mlpdev::kParams;
            std::vector<unsigned short> wb(np);
            for (int i = 0; i < np; ++i) wb[i] = mlpdev::to_bf16(params[i]);
            if (!b->mlpW) BCHK(b, hipMalloc(&b->mlpW, np * sizeof(unsigned short)), "set_return_map");
            if (!b->mlpP) BCHK(b, hipMalloc(&b->mlpP, np * sizeof(float)), "set_return_map");
            BCHK(b, hipMemcpy(b->mlpW, wb.data(), np * sizeof(unsigned short), hipMemcpyHostToDevice), "set_return_map");
            BCHK(b, hipMemcpy(b->mlpP, params, np * sizeof(float), hipMemcpyHostToDevice), "set_return_map");
            std::memcpy(b->norm.in_mean, norm, 5 * sizeof(float));
            std::memcpy(b->norm.in_scale, norm + 5, 5 * sizeof(float));
            std::memcpy(b->norm.out_mean, norm + 10, 3 * sizeof(float));
            std::memcpy(b->norm.out_scale, norm + 13, 3 * sizeof(float));
            for (int q = 0; q < 5; ++q)
                if (!(b->norm.in_scale[q] > 0)) return bfail(b, ICEMPM_E_ARG, "set_return_map: input scale must be > 0");
            b->tol = tol;
            if (!b->mapQ) BCHK(b, hipMalloc(&b->mapQ, (size_t)b->nPts * sizeof(MapEntry)), "set_return_map");
            if (!b->mapCount) BCHK(b, hipMalloc(&b->mapCount, 2 * sizeof(unsigned int)), "set_return_map");
        }
        b->rmap = mode;
        return ICEMPM_OK;
    });
}

int icempm_batch_read_harvest(icempm_batch *b, float *X, float *T, int cap, unsigned long long *total) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b || !total || cap < 0 || (cap > 0 && (!X || !T))) return ICEMPM_E_ARG;
        if (!b->finalized) return bfail(b, ICEMPM_E_STATE, "read_harvest: batch not finalized");
        BCHK(b, hipStreamSynchronize(b->stream), "read_harvest");
        unsigned long long n = 0;
        BCHK(b, hipMemcpy(&n, b->hcount, sizeof(n), hipMemcpyDeviceToHost), "read_harvest");
        *total = n;
        const int m = (int)std::min<unsigned long long>(std::min<unsigned long long>(n, (unsigned long long)b->hcap),
                                                        (unsigned long long)cap);
        if (m > 0) {
            BCHK(b, hipMemcpy(X, b->hx, (size_t)m * 5 * sizeof(float), hipMemcpyDeviceToHost), "read_harvest");
            BCHK(b, hipMemcpy(T, b->ht, (size_t)m * 3 * sizeof(float), hipMemcpyDeviceToHost), "read_harvest");
        }
        return ICEMPM_OK;
    });
}

int icempm_batch_set_tuning(icempm_batch *b, int knob, int value) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b) return ICEMPM_E_ARG;
        switch (knob) {
        case ICEMPM_BATCH_TUNE_CHUNK:
            if (value != 64 && value != 128 && value != 256)
                return bfail(b, ICEMPM_E_ARG, "set_tuning: points per chunk is 64, 128 or 256");
            if (value != b->chunkPoints) {
                const int before = b->chunkPoints;
                b->chunkPoints = value;
                if (b->finalized) {
                    BCHK(b, hipStreamSynchronize(b->stream), "set_tuning");
                    const int rc = rebuild_chunks(b);
                    if (rc) b->chunkPoints = before;
                    return rc;
                }
            }
            return ICEMPM_OK;
        case ICEMPM_BATCH_TUNE_RESORT:
            if (value < 0) return bfail(b, ICEMPM_E_ARG, "set_tuning: the re-sort cadence is >= 0");
            b->resortEvery = value;
            return ICEMPM_OK;
        case ICEMPM_BATCH_TUNE_MAP_MIN_ACCEPT:
            if (value < 0 || value > 100) return bfail(b, ICEMPM_E_ARG, "set_tuning: acceptance threshold is 0..100 percent");
            b->mapMinAccept = value / 100.0;
            return ICEMPM_OK;
        default:
            return bfail(b, ICEMPM_E_ARG, "set_tuning: unknown knob");
        }
    });
}

int icempm_batch_get_tuning(const icempm_batch *b, int knob) {
    if (!b) return -1;
    switch (knob) {
    case ICEMPM_BATCH_TUNE_CHUNK: return b->chunkPoints;
    case ICEMPM_BATCH_TUNE_RESORT: return b->resortEvery;
    case ICEMPM_BATCH_TUNE_MAP_MIN_ACCEPT: return (int)std::lround(b->mapMinAccept * 100.0);
    default: return -1;
    }
}

int icempm_batch_resort(icempm_batch *b) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b) return ICEMPM_E_ARG;
        if (!b->finalized) return bfail(b, ICEMPM_E_STATE, "resort: batch not finalized");
        BCHK(b, hipStreamSynchronize(b->stream), "resort");
        return resort(b);
    });
}

int icempm_batch_checkpoint(icempm_batch *b) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b) return ICEMPM_E_ARG;
        if (!b->finalized) return bfail(b, ICEMPM_E_STATE, "checkpoint: batch not finalized");
        BCHK(b, once(b->kpos, pos_bytes(b)), "checkpoint");
        BCHK(b, once(b->krest, rest_bytes(b)), "checkpoint");
        BCHK(b, once(b->kcrushed, b->pitch), "checkpoint");
        BCHK(b, once(b->korig, b->pitch * sizeof(int)), "checkpoint");
        if (b->grain) BCHK(b, once(b->kgrain, b->pitch * sizeof(short)), "checkpoint");
        BCHK(b, hipMemcpyAsync(b->kpos, b->pos, pos_bytes(b), hipMemcpyDeviceToDevice, b->stream), "checkpoint");
        BCHK(b, hipMemcpyAsync(b->krest, b->rest, rest_bytes(b), hipMemcpyDeviceToDevice, b->stream), "checkpoint");
        BCHK(b, hipMemcpyAsync(b->kcrushed, b->crushed, b->pitch, hipMemcpyDeviceToDevice, b->stream), "checkpoint");
        BCHK(b, hipMemcpyAsync(b->korig, b->orig, b->pitch * sizeof(int), hipMemcpyDeviceToDevice, b->stream), "checkpoint");
        if (b->grain)   // re-sorts permute the grain row with the points
            BCHK(b, hipMemcpyAsync(b->kgrain, b->grain, b->pitch * sizeof(short), hipMemcpyDeviceToDevice, b->stream),
                 "checkpoint");
        BCHK(b, hipStreamSynchronize(b->stream), "checkpoint");
        b->kt = b->t;
        b->kstep = b->step;
        b->kcstart = b->hcstart;
        b->kccase = b->hccase;
        b->kcdense = b->hcdense;
        b->kChunkPoints = b->chunkPoints;
        b->haveCheckpoint = true;
        return ICEMPM_OK;
    });
}

int icempm_batch_restore(icempm_batch *b) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b) return ICEMPM_E_ARG;
        if (!b->haveCheckpoint) return bfail(b, ICEMPM_E_STATE, "restore: no checkpoint");
        BCHK(b, hipStreamSynchronize(b->stream), "restore");
        BCHK(b, hipMemcpyAsync(b->pos, b->kpos, pos_bytes(b), hipMemcpyDeviceToDevice, b->stream), "restore");
        BCHK(b, hipMemcpyAsync(b->rest, b->krest, rest_bytes(b), hipMemcpyDeviceToDevice, b->stream), "restore");
        BCHK(b, hipMemcpyAsync(b->crushed, b->kcrushed, b->pitch, hipMemcpyDeviceToDevice, b->stream), "restore");
        BCHK(b, hipMemcpyAsync(b->orig, b->korig, b->pitch * sizeof(int), hipMemcpyDeviceToDevice, b->stream), "restore");
        if (b->grain)
            BCHK(b, hipMemcpyAsync(b->grain, b->kgrain, b->pitch * sizeof(short), hipMemcpyDeviceToDevice, b->stream),
                 "restore");
        BCHK(b, hipStreamSynchronize(b->stream), "restore");
        b->pending = -1;   // the grids hold the P2G of the state before the restore
        b->t = b->kt;
        b->step = b->kstep;
        b->hcstart = b->kcstart;
        b->hccase = b->kccase;
        b->hcdense = b->kcdense;
        b->chunkPoints = b->kChunkPoints;
        return upload_chunks(b);
    });
}

int icempm_batch_autotune(icempm_batch *b, int probe_steps, double *report, int cap, int *rows) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b || probe_steps < 16 || cap < 0 || (cap > 0 && !report) || !rows) return ICEMPM_E_ARG;
        if (!b->finalized) return bfail(b, ICEMPM_E_STATE, "autotune: batch not finalized");
        if (b->timingStride > 0) return bfail(b, ICEMPM_E_STATE, "autotune: switch kernel timing off first");
        // the probes would append their pairs to the harvest buffer
        if (b->rmap == kMapHarvest) return bfail(b, ICEMPM_E_STATE, "autotune: not in harvest mode");
        int rc = icempm_batch_checkpoint(b);
        if (rc) return rc;
        // what the probes change besides the point state: the map statistics
        // and the error flag (restored below), the force history and lastRun
        // (the probes' own; a caller reads them after its next run)
        unsigned long long stats0[kMapStats] = {};
        int err0 = 0;
        BCHK(b, hipMemcpy(stats0, b->stats, sizeof(stats0), hipMemcpyDeviceToHost), "autotune");
        BCHK(b, hipMemcpy(&err0, b->err, sizeof(int), hipMemcpyDeviceToHost), "autotune");
        const int chunks[3] = {256, 128, 64};
        const int resorts[3] = {0, probe_steps / 2, probe_steps / 4};
        double best = 1e300;
        int bestChunk = b->chunkPoints, bestResort = b->resortEvery, nrow = 0;
        for (int ci = 0; ci < 3; ++ci)
            for (int ri = 0; ri < 3; ++ri) {
                // one clock for every candidate: the host time of the whole
                // probe (re-sorts and graph captures included), measured on a
                // second run so that the no-re-sort candidates replay a graph
                // captured by the first
                b->chunkPoints = chunks[ci];
                b->resortEvery = resorts[ri];
                double per = 0;
                for (int pass = 0; pass < 2; ++pass) {
                    if ((rc = icempm_batch_restore(b))) return rc;
                    b->chunkPoints = chunks[ci];
                    if ((rc = rebuild_chunks(b))) return rc;
                    const auto h0 = std::chrono::steady_clock::now();
                    if ((rc = icempm_batch_run(b, probe_steps, 1))) return rc;
                    per = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - h0).count() /
                          probe_steps;
                }
                if (nrow < cap) {
                    report[3 * nrow] = chunks[ci];
                    report[3 * nrow + 1] = resorts[ri];
                    report[3 * nrow + 2] = per;
                }
                ++nrow;
                if (per < best) {
                    best = per;
                    bestChunk = chunks[ci];
                    bestResort = resorts[ri];
                }
            }
        *rows = nrow;
        // With the learned map: a branch whose network proposals the yield gate
        // passed less often than mapMinAccept over the probes is switched off
        // (its projections take the exact map in the particle pass, with no
        // queue and no map kernel)
        if (b->rmap == kMapLearned) {
            unsigned long long st[kMapStats];
            BCHK(b, hipMemcpy(st, b->stats, sizeof(st), hipMemcpyDeviceToHost), "autotune");
            int mask = 0;
            const unsigned long long tA = st[3] - stats0[3], tF = st[4] - stats0[4];
            const unsigned long long sA = st[5] - stats0[5], sF = st[6] - stats0[6];
            if ((b->mapBranches & kMapTension) && tA + tF > 0 && (double)tA >= b->mapMinAccept * (double)(tA + tF))
                mask |= kMapTension;
            if ((b->mapBranches & kMapShear) && sA + sF > 0 && (double)sA >= b->mapMinAccept * (double)(sA + sF))
                mask |= kMapShear;
            b->tuneBranchStats[0] = tA; b->tuneBranchStats[1] = tF;
            b->tuneBranchStats[2] = sA; b->tuneBranchStats[3] = sF;
            if ((rc = icempm_batch_set_map_branches(b, mask))) return rc;
        }
        // back to the checkpointed state, with the fastest setting
        if ((rc = icempm_batch_restore(b))) return rc;
        BCHK(b, hipMemcpy(b->stats, stats0, sizeof(stats0), hipMemcpyHostToDevice), "autotune");
        BCHK(b, hipMemcpy(b->err, &err0, sizeof(int), hipMemcpyHostToDevice), "autotune");
        b->resortEvery = bestResort;
        if (bestChunk == b->chunkPoints) return ICEMPM_OK;   // the restored table is the one
        b->chunkPoints = bestChunk;
        return rebuild_chunks(b);
    });
}

int icempm_batch_map_stats(icempm_batch *b, unsigned long long *out, int reset) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b || !out) return ICEMPM_E_ARG;
        if (!b->finalized) return bfail(b, ICEMPM_E_STATE, "map_stats: batch not finalized");
        BCHK(b, hipStreamSynchronize(b->stream), "map_stats");
        unsigned long long all[kMapStats];
        BCHK(b, hipMemcpy(all, b->stats, sizeof(all), hipMemcpyDeviceToHost), "map_stats");
        std::memcpy(out, all, 3 * sizeof(unsigned long long));
        if (reset) {
            const unsigned long long z[kMapStats] = {};
            BCHK(b, hipMemcpy(b->stats, z, sizeof(z), hipMemcpyHostToDevice), "map_stats");
        }
        return ICEMPM_OK;
    });
}

int icempm_batch_map_branch_stats(icempm_batch *b, unsigned long long *out, int reset) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b || !out) return ICEMPM_E_ARG;
        if (!b->finalized) return bfail(b, ICEMPM_E_STATE, "map_branch_stats: batch not finalized");
        BCHK(b, hipStreamSynchronize(b->stream), "map_branch_stats");
        unsigned long long all[kMapStats];
        BCHK(b, hipMemcpy(all, b->stats, sizeof(all), hipMemcpyDeviceToHost), "map_branch_stats");
        std::memcpy(out, all + 3, 4 * sizeof(unsigned long long));
        if (reset) {
            const unsigned long long z[kMapStats] = {};
            BCHK(b, hipMemcpy(b->stats, z, sizeof(z), hipMemcpyHostToDevice), "map_branch_stats");
        }
        return ICEMPM_OK;
    });
}

int icempm_batch_set_map_branches(icempm_batch *b, int mask) {
    return host_guard(b ? &b->lastError : nullptr, [&]() -> int {
        if (!b || mask < 0 || mask > (kMapTension | kMapShear)) return ICEMPM_E_ARG;
        if (mask != b->mapBranches) {
            BCHK(b, hipStreamSynchronize(b->stream), "set_map_branches");
            drop_graph(b);   // the captured launches hold the mask (and the map kernel or not)
            b->mapBranches = mask;
        }
        return ICEMPM_OK;
    });
}

int icempm_batch_get_map_branches(const icempm_batch *b) { return b ? b->mapBranches : -1; }

int icempm_batch_autotune_branch_stats(const icempm_batch *b, unsigned long long *out) {
    if (!b || !out) return ICEMPM_E_ARG;
    std::memcpy(out, b->tuneBranchStats, sizeof(b->tuneBranchStats));
    return ICEMPM_OK;
}

}  // extern "C"
