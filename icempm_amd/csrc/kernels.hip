// kernels.hip -- grid kernels of the MLS-MPM substep for gfx950 (CDNA4),
// FP64, built without FMA contraction.  (The particle pass is in
// particles.inc, built twice: particles_exact.hip and particles_fast.hip.)
//
//   k_update<false>  grid update (FAST mode) with the indenter force reduced
//       per workgroup in shared memory; also clears the next substep's grid.
// ORDERED path (bit-reproducible):
//   k_point_records / k_node_fold  every node sums its contributions in
//       increasing particle index (and, in a run, is updated at once);
//   k_update<true>, k_bins_fold  the indenter force is summed in increasing
//       node index.
#include <climits>

#include "internal.h"
#include "ordered_device.h"

namespace icempm {

__global__ void k_fill_f64(double *__restrict__ p, size_t n, double v) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x)
        p[i] = v;
}

__global__ void k_fill_i32(int *__restrict__ p, size_t n, int v) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x)
        p[i] = v;
}

static unsigned fill_blocks(size_t n) {
    size_t b = (n + 255) / 256;
    return (unsigned)(b < 4096 ? (b == 0 ? 1 : b) : 4096);
}

hipError_t launch_fill_f64(double *p, size_t n, double v, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_f64, dim3(fill_blocks(n)), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}

hipError_t launch_fill_i32(int *p, size_t n, int v, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_i32, dim3(fill_blocks(n)), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}

// Plain streaming copy: the reference point for the achievable HBM bandwidth
// and for scaling the HBM traffic counters.  Each thread moves four
// independent 16-byte vectors per iteration so that enough loads are in
// flight per wavefront.
__global__ __launch_bounds__(256) void k_copy(const double2 *__restrict__ src,
                                              double2 *__restrict__ dst, size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    for (; i + 3 * stride < n; i += 4 * stride) {
        const double2 a = src[i], b = src[i + stride], c = src[i + 2 * stride],
                      d = src[i + 3 * stride];
        dst[i] = a;
        dst[i + stride] = b;
        dst[i + 2 * stride] = c;
        dst[i + 3 * stride] = d;
    }
    for (; i < n; i += stride) dst[i] = src[i];
}

hipError_t launch_copy(const double *src, double *dst, size_t n_doubles, hipStream_t s) {
    const size_t n2 = n_doubles / 2;
    if (n2 == 0) return hipSuccess;
    hipLaunchKernelGGL(k_copy, dim3(4096), dim3(256), 0, s,
                       reinterpret_cast<const double2 *>(src), reinterpret_cast<double2 *>(dst), n2);
    return hipGetLastError();
}

__global__ void k_hello(int *flag) {
    if (threadIdx.x == 0 && blockIdx.x == 0) flag[0] = 1;
}

hipError_t launch_hello(int *flag, hipStream_t s) {
    hipLaunchKernelGGL(k_hello, dim3(1), dim3(64), 0, s, flag);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Grid update: v2_kernel_update_nodes (gpu_implementation5.cu:215-290).
constexpr int kUpdBlock = 256;
constexpr int kMaxLdsBins = 256;

// A node of the given mass (not zero): v is its momentum, then its velocity; bin
// and f are set where the indenter touches it.
static __device__ __forceinline__ void node_update(const KParams &k, int idx, double mass, double ind_x, double ind_y,
                                                   double &v0, double &v1, int &bin, double &f0, double &f1) {
    const int nb = k.nbins;
    const double dt = k.dt, h = k.h, V = k.indV;
    const int gx = k.gridX, gy = k.gridY;
    v0 = v0 / mass;
    v1 = v1 / mass;
    v1 = v1 - dt * k.gravity;
    const double vmax = 0.5 * h / dt;
    const double vn = sqrt(v0 * v0 + v1 * v1);
    if (vn > vmax) {
        v0 = v0 / vn * vmax;
        v1 = v1 / vn * vmax;
    }
    const int ix = idx % gx;
    const int iy = idx / gx;
    double n0 = ix * h - ind_x;
    double n1 = iy * h - ind_y;
    if (n0 * n0 + n1 * n1 < k.indRsq) {
        const double r0 = v0 - V;
        const double r1 = v1 - 0.0;
        const double z = n0 * n0 + n1 * n1;
        if (z > 0) {
            const double nz = sqrt(z);
            n0 = n0 / nz;
            n1 = n1 / nz;
        }
        const double vnr = r0 * n0 + r1 * n1;
        if (vnr < 0) {
            const double t0 = r0 - n0 * vnr;
            const double t1 = r1 - n1 * vnr;
            const double p0 = v0, p1 = v1;
            v0 = V + t0;
            v1 = 0.0 + t1;
            f0 = (p0 - v0) * mass / dt;
            f1 = (p1 - v1) * mass / dt;
            double angle = atan2(n0, n1);
            angle += kPi;
            angle *= nb / (2 * kPi);
            int index = (int)angle;
            index = max(index, 0);
            index = min(index, nb - 1);
            bin = index;
        }
    }
    if (iy <= 2) {
        v0 = 0;
        v1 = 0;
    } else if (iy >= gy - 3 && v1 > 0) {
        v1 = 0;
    }
    if (ix <= 2 && v0 < 0)
        v0 = 0;
    else if (ix >= gx - 3 && v0 > 0)
        v0 = 0;
}

template <bool ORDERED>
__global__ __launch_bounds__(kUpdBlock) void k_update(KParams k, double *__restrict__ grid,
                                                      double ind_x, double ind_y,
                                                      double *__restrict__ hist2,
                                                      double *__restrict__ zeroGrid,
                                                      int *__restrict__ nodeBin,
                                                      double *__restrict__ nodeF) {
    __shared__ double sb[2 * kMaxLdsBins + 2];
    __shared__ int any;
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    const bool in = idx < k.gridTotal;
    const size_t gp = k.gp;
    const int nb = k.nbins;
    const bool ldsBins = nb <= kMaxLdsBins;
    if constexpr (!ORDERED) {
        if (ldsBins)
            for (int e = threadIdx.x; e < 2 * nb + 2; e += blockDim.x) sb[e] = 0;
        if (threadIdx.x == 0) any = 0;
        __syncthreads();
    }
    int bin = -1;
    double f0 = 0, f1 = 0;
    if (in) {
        if (zeroGrid) {
            zeroGrid[idx] = 0;
            zeroGrid[gp + idx] = 0;
            zeroGrid[2 * gp + idx] = 0;
        }
        const double mass = grid[idx];
        if (mass != 0) {
            double v0 = grid[gp + idx], v1 = grid[2 * gp + idx];
            node_update(k, idx, mass, ind_x, ind_y, v0, v1, bin, f0, f1);
            grid[gp + idx] = v0;
            grid[2 * gp + idx] = v1;
        }
    }
    if constexpr (ORDERED) {
        if (in) {
            nodeBin[idx] = bin;
            nodeF[2 * (size_t)idx] = f0;
            nodeF[2 * (size_t)idx + 1] = f1;
        }
    } else {
        if (bin >= 0) {
            if (ldsBins) {
                atomicAdd(&sb[2 * bin], f0);
                atomicAdd(&sb[2 * bin + 1], f1);
                atomicAdd(&sb[2 * nb], f0);
                atomicAdd(&sb[2 * nb + 1], f1);
                any = 1;
            } else {
                unsafeAtomicAdd(&k.bins[2 * bin], f0);
                unsafeAtomicAdd(&k.bins[2 * bin + 1], f1);
                if (hist2) {
                    unsafeAtomicAdd(&hist2[0], f0);
                    unsafeAtomicAdd(&hist2[1], f1);
                }
            }
        }
        __syncthreads();
        if (ldsBins && any) {
            for (int e = threadIdx.x; e < 2 * nb + 2; e += blockDim.x) {
                const double v = sb[e];
                if (v != 0) {
                    if (e < 2 * nb)
                        unsafeAtomicAdd(&k.bins[e], v);
                    else if (hist2)
                        unsafeAtomicAdd(&hist2[e - 2 * nb], v);
                }
            }
        }
    }
}

hipError_t launch_update(const KParams &k, double *grid, double ix, double iy, double *hist2,
                         double *zeroGrid, bool ordered, int *nodeBin, double *nodeF,
                         hipStream_t s) {
    if (k.gridTotal <= 0) return hipSuccess;
    const unsigned nb = (unsigned)((k.gridTotal + kUpdBlock - 1) / kUpdBlock);
    if (ordered)
        hipLaunchKernelGGL(k_update<true>, dim3(nb), dim3(kUpdBlock), 0, s, k, grid, ix, iy,
                           hist2, zeroGrid, nodeBin, nodeF);
    else
        hipLaunchKernelGGL(k_update<false>, dim3(nb), dim3(kUpdBlock), 0, s, k, grid, ix, iy,
                           hist2, zeroGrid, nodeBin, nodeF);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// ORDERED P2G, in two kernels: every point makes the record its contributions
// follow from and enters its base cell's list; every node then collects the
// points of its nine cells, puts them in order and sums.  What bounds it is
// latency: few workgroups, each a chain of loads and LDS passes.  A substep of
// 60,000 points takes 31 us, of which the fold 16 (found, ranked, listed and
// summed in about equal parts) and the G2P with the records 14; through memory, with a
// counting sort and an insertion sort per node, it took 249 (contributions 20,
// sort 60, fold 165).  An insertion sort of each node's list in LDS took up to 20
// us (the points of one row of the load's order lie in two rows of cells), a rank
// by comparing all points of a tile 6.
struct Terms {   // a point's part of its contributions: weights, distances, affine momentum, momentum
    double wx[3], wy[3], dx[3], dy[3], A00, A01, A10, A11, mv0, mv1;
};
static __device__ __forceinline__ void axis_terms(double fx, double h, double *w, double *d) {
    // as stencil
    const double v0 = 1.5 - fx, v1 = fx - 1.0, v2 = fx - 0.5;
    w[0] = 0.5 * v0 * v0;
    w[1] = 0.75 - v1 * v1;
    w[2] = 0.5 * v2 * v2;
#pragma unroll
    for (int i = 0; i < 3; ++i) d[i] = (i - fx) * h;
}
static __device__ __forceinline__ Terms terms_of(const PointRec &r, double h) {
    Terms t;
    axis_terms(r.f.x, h, t.wx, t.dx);
    axis_terms(r.f.y, h, t.wy, t.dy);
    t.A00 = r.a.x; t.A01 = r.a.y; t.A10 = r.b.x; t.A11 = r.b.y;
    t.mv0 = r.mv.x; t.mv1 = r.mv.y;
    return t;
}
// The contribution to node (i, j) of the stencil: mass (part 0) or momentum (1, 2).
static __device__ __forceinline__ double term(const Terms &t, int i, int j, int part, double mass) {
    const double W = t.wx[i] * t.wy[j];
    if (part == 0) return W * mass;
    const double d0 = t.dx[i], d1 = t.dy[j];
    return part == 1 ? W * (t.mv0 + (t.A00 * d0 + t.A01 * d1)) : W * (t.mv1 + (t.A10 * d0 + t.A11 * d1));
}

__global__ __launch_bounds__(kFoldBlock) void k_bins_fold(BinsFold B) {
    __shared__ BinsLds L;
    fold_bins(B, L);
}

BinsFold ordered_force(const KParams &k, const OrderedScratch &o, double *hist2, double ix, double iy) {
    // the nodes in contact lie within the disc; two nodes of margin for the rounding
    const double R = sqrt(k.indRsq);
    const auto range = [&](double c, int g, int &lo, int &n) {
        // (by h, which places the nodes; h_inv places the points)
        const double a = floor((c - R) / k.h) - 2, b = ceil((c + R) / k.h) + 2;
        lo = 0;
        n = g;
        if (!(a <= b)) return;   // not a number: all
        lo = (int)fmin(fmax(a, 0.0), (double)(g - 1));
        n = (int)fmin(fmax(b, 0.0), (double)(g - 1)) - lo + 1;
    };
    BinsFold B{k.bins, o.nodeBin, o.nodeF, hist2, k.nbins, k.gridX, 0, 0, 0, 0};
    range(ix, k.gridX, B.x0, B.w);
    range(iy, k.gridY, B.y0, B.h);
    return B;
}

hipError_t ordered_fold_forces(const KParams &k, OrderedScratch &o, double *hist2, double ix, double iy,
                               hipStream_t s) {
    if (k.nbins + 1 > kFoldBinsMax) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_bins_fold, dim3(1), dim3(kFoldBlock), 0, s, ordered_force(k, o, hist2, ix, iy));
    return hipGetLastError();
}

// padGrid (may be null): the padding of its rows is cleared.
__global__ __launch_bounds__(256) void k_point_records(KParams k, PointLists lists, double *__restrict__ padGrid) {
    const int pt = blockIdx.x * blockDim.x + threadIdx.x;
    if (padGrid && (size_t)k.gridTotal + pt < k.gp)
        for (int r = 0; r < kGridRows; ++r) padGrid[r * k.gp + k.gridTotal + pt] = 0;
    if (pt >= k.nPts) return;
    const double *P = k.pts + pt;
    const size_t pp = k.pp;
    point_record(k, lists, pt, P[pp * kRowPosX], P[pp * (kRowPosX + 1)], P[pp * kRowVelX], P[pp * (kRowVelX + 1)],
                 P[pp * (kRowFe00 + 0)], P[pp * (kRowFe00 + 1)], P[pp * (kRowFe00 + 2)], P[pp * (kRowFe00 + 3)],
                 P[pp * (kRowBp00 + 0)], P[pp * (kRowBp00 + 1)], P[pp * (kRowBp00 + 2)], P[pp * (kRowBp00 + 3)]);
}

// A workgroup takes a tile of 8 x 8 nodes: the points of its 10 x 10 cells, put in
// order by counting the smaller ones, a bit mask of them per cell, a node's list
// from the bits of its nine cells, and a wavefront per component that adds up.
// Tiles of more points than kFoldPts, about 4.4 a cell, go by quarters, and
// where those or a cell's bucket overflow, a quarter's points in batches of
// ascending indices.
constexpr int kTileN = 8, kTileNodes = kTileN * kTileN, kTileCells = (kTileN + 2) * (kTileN + 2);
constexpr int kBuckets = 1024;   // of the ranking
constexpr int kFoldPts = 440, kFoldWords = (kFoldPts + 63) / 64, kFoldList = 4096;
struct FoldLds {
    union {
        struct {
            unsigned long long mask[kTileCells][kFoldWords];   // a cell's points, by their places in order
            unsigned long long node[kFoldWords][kTileNodes];   // a node's
            unsigned short before[kFoldWords][kTileNodes];     // how many of them are in the words before
            __attribute__((aligned(16))) int count[kBuckets];  // points per bucket of the ranking, then its first place
            int sorted[kFoldPts];                              // the points, bucket by bucket
        };
        struct {
            Terms t;
            double pad;   // 19 doubles: the places of a wavefront spread over the banks
        } terms[kFoldPts];
    };
    int idx[kFoldPts];                // the points as found
    unsigned char cell[kFoldPts];     // their cells: column | row << 4
    unsigned short list[kFoldList];   // entry e of node t at e nodes + t: its cell among the nine << 9 | place
    int wave[4], low[4], high[4], over, crowded, found;
    double res[3][kTileNodes];
};
static_assert(kFoldPts < 512 && kTileCells <= 128, "list entries hold a place in 9 bits; two wavefronts hold the cells");

// Adds the contributions of the points found (L.idx, L.cell; total of them) to the
// sums of T x T nodes: wavefront part, lane node, in the points' order.  False,
// with nothing added, if the nodes' lists do not fit.  L.mask and L.count are
// zero.
static __device__ bool fold_found(const KParams &k, FoldLds &L, const PointRec *__restrict__ rec, int total, int T,
                                  double &sum) {
    const int t = threadIdx.x, lane = t & 63, E = T + 2;
    // the records of the points found at t and t + 256 are on their way while
    // the lists are made
    PointRec r[2];
    int v[2], place[2] = {0, 0};
    int low = INT_MAX, high = 0;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int e = t + 256 * q;
        v[q] = e < total ? L.idx[e] : -1;
        r[q] = rec[e < total ? v[q] : 0];
        if (e < total) {
            low = min(low, v[q]);
            high = max(high, v[q]);
        }
    }
    // their places in order: buckets over the range of the indices, and within
    // a bucket the smaller ones counted
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        low = min(low, __shfl_xor(low, d, 64));
        high = max(high, __shfl_xor(high, d, 64));
    }
    if (lane == 0) {
        L.low[t >> 6] = low;
        L.high[t >> 6] = high;
    }
    __syncthreads();
    low = min(min(L.low[0], L.low[1]), min(L.low[2], L.low[3]));
    high = max(max(L.high[0], L.high[1]), max(L.high[2], L.high[3]));
    const float scale = (float)kBuckets / ((float)(high - low) + 1.f);
    int bin[2], pos[2];
#pragma unroll
    for (int q = 0; q < 2; ++q)
        if (t + 256 * q < total) {
            bin[q] = min((int)((float)(v[q] - low) * scale), kBuckets - 1);
            pos[q] = atomicAdd(&L.count[bin[q]], 1);
        }
    __syncthreads();
    {
        const int4 c = *reinterpret_cast<const int4 *>(&L.count[4 * t]);
        const int sum = c.x + c.y + c.z + c.w;
        int run = sum;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(run, d, 64);
            if (lane >= d) run += o;
        }
        if (lane == 63) L.wave[t >> 6] = run;
        __syncthreads();
        for (int w = 0; w < t >> 6; ++w) run += L.wave[w];
        run -= sum;
        *reinterpret_cast<int4 *>(&L.count[4 * t]) = make_int4(run, run + c.x, run + c.x + c.y, run + c.x + c.y + c.z);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 2; ++q)
        if (t + 256 * q < total) L.sorted[L.count[bin[q]] + pos[q]] = v[q];
    __syncthreads();
    const int nodes = T * T, words = (total + 63) >> 6;
    int cx[2], cy[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int e = t + 256 * q;
        if (e >= total) continue;
        const int from = L.count[bin[q]], to = bin[q] + 1 < kBuckets ? L.count[bin[q] + 1] : total;
        int p = from;
        for (int o = from; o < to; ++o) p += L.sorted[o] < v[q];
        place[q] = p;
        cx[q] = L.cell[e] & 15;
        cy[q] = L.cell[e] >> 4;
        atomicOr(&L.mask[cy[q] * E + cx[q]][p >> 6], 1ull << (p & 63));
    }
    __syncthreads();
    for (int e = t; e < nodes * words; e += 256) {
        const int node = e % nodes, w = e / nodes, c = node / T * E + node % T;
        unsigned long long m = 0;
#pragma unroll
        for (int c9 = 0; c9 < 9; ++c9) m |= L.mask[c + c9 / 3 * E + c9 % 3][w];
        L.node[w][node] = m;
    }
    __syncthreads();
    int len = 0;   // of the node lane's list
    if (lane < nodes)
        for (int w = 0; w < words; ++w) {
            if (t < 64) L.before[w][lane] = (unsigned short)len;
            len += __popcll(L.node[w][lane]);
        }
    if (len * nodes > kFoldList) L.crowded = 1;
    __syncthreads();
    if (L.crowded) return false;
    // every point enters the lists of the nodes around it, at the place its
    // place in order gives
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        if (t + 256 * q >= total) continue;
        const int p = place[q], w = p >> 6;
        const unsigned long long smaller = (1ull << (p & 63)) - 1ull;
#pragma unroll
        for (int c9 = 0; c9 < 9; ++c9) {
            const int x = cx[q] - c9 % 3, y = cy[q] - c9 / 3;
            if (x < 0 || x >= T || y < 0 || y >= T) continue;
            const int node = y * T + x, at = L.before[w][node] + __popcll(L.node[w][node] & smaller);
            L.list[at * nodes + node] = (unsigned short)(c9 << 9 | p);
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 2; ++q)
        if (t + 256 * q < total) L.terms[place[q]].t = terms_of(r[q], k.h);
    __syncthreads();
    if (lane < nodes && t < 3 * 64) {
        const unsigned short *list = L.list + lane;
        const int part = t >> 6;
#pragma unroll 4
        for (int e = 0; e < len; ++e) {
            const int o = list[e * nodes], c9 = o >> 9;
            sum += term(L.terms[o & 511].t, 2 - c9 % 3, 2 - c9 / 3, part, k.mass);
        }
    }
    return true;
}

// The T x T nodes from (X0, Y0) of the tile at (TX, TY); false if they do not fit.
static __device__ bool fold_tile(const KParams &k, FoldLds &L, const PointRec *__restrict__ rec,
                                 const int *__restrict__ bucket, const int2 *__restrict__ cells, int T, int X0, int Y0,
                                 int TX, int TY) {
    const int t = threadIdx.x, lane = t & 63, E = T + 2, gx = k.gridX, gy = k.gridY;
    // a cell a thread: its count, and the first of its points at the same time
    int n = 0;
    int4 head = make_int4(0, 0, 0, 0);
    const int4 *b = nullptr;
    if (t < E * E) {
        const int X = X0 - 2 + t % E, Y = Y0 - 2 + t / E;
        if (X >= 0 && X < gx && Y >= 0 && Y < gy) {
            const size_t c = (size_t)X + (size_t)Y * gx;
            b = reinterpret_cast<const int4 *>(bucket) + kCellCap / 4 * c;
            n = cells[c].x;
            head = b[0];
        }
    }
    int inc = n;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int v = __shfl_up(inc, d, 64);
        if (lane >= d) inc += v;
    }
    __syncthreads();   // the tile before has been used
    if (t < 128 && lane == 63) L.wave[t >> 6] = inc;
    if (t == 0) L.over = L.crowded = 0;
    for (int e = t; e < kTileCells * kFoldWords; e += 256) L.mask[0][e] = 0;
    *reinterpret_cast<int4 *>(&L.count[4 * t]) = make_int4(0, 0, 0, 0);
    __syncthreads();
    const int total = L.wave[0] + L.wave[1];
    if (n > kCellCap) L.over = 1;
    __syncthreads();
    if (L.over || total > kFoldPts) return false;
    const int at = inc - n + (t >= 64 ? L.wave[0] : 0);
    for (int e = 0; e < n; ++e) {
        if (e > 0 && (e & 3) == 0) head = b[e >> 2];
        L.idx[at + e] = (e & 3) == 0 ? head.x : ((e & 3) == 1 ? head.y : ((e & 3) == 2 ? head.z : head.w));
        L.cell[at + e] = (unsigned char)(t % E | t / E << 4);
    }
    __syncthreads();
    double sum = 0.0;
    if (!fold_found(k, L, rec, total, T, sum)) return false;
    if (lane < T * T && t < 3 * 64) L.res[t >> 6][(Y0 - TY + lane / T) * kTileN + X0 - TX + lane % T] = sum;
    return true;
}

// The same for crowded cells: a quarter's points in batches of ascending indices
// that fit, each as fold_found adds it.  A batch is cut by a histogram of the
// indices not yet taken, and the histogram drawn again over its first bucket
// where that alone holds too many.  Every batch goes through the cells' buckets
// and chains again.  A substep of 60,000 points at 16, 25 and 49 a cell takes 0.36,
// 0.60 and 1.4 ms; with the points looked up node by node, the least index above
// the last, it took 10.8, 25 and 89 ms, and with a counting sort and an insertion
// sort per node in memory 2.3, 4.8 and 16 ms.
constexpr int kPartPts = 256;
static_assert(kPartPts * (kTileN / 2) * (kTileN / 2) <= kFoldList && kPartPts <= kFoldPts, "a batch always fits");
static __device__ void fold_crowded(const KParams &k, FoldLds &L, const PointRec *__restrict__ rec,
                                    const int *__restrict__ bucket, const int2 *__restrict__ cells,
                                    const int *__restrict__ next, int X0, int Y0, int TX, int TY) {
    constexpr int T = kTileN / 2, E = T + 2;
    const int t = threadIdx.x, lane = t & 63, X = X0 - 2 + t % E, Y = Y0 - 2 + t / E;
    const bool in = t < E * E && X >= 0 && X < k.gridX && Y >= 0 && Y < k.gridY;
    const size_t c = in ? (size_t)X + (size_t)Y * k.gridX : 0;
    const int2 head = in ? cells[c] : make_int2(0, 0);
    const auto each = [&](auto &&see) {   // the points of the thread's cell
        for (int e = 0; e < min(head.x, kCellCap); ++e) see(bucket[kCellCap * c + e]);
        for (int e = kCellCap, p = head.y; e < head.x && p > 0; ++e, p = next[p - 1]) see(p - 1);
    };
    double sum = 0.0;
    for (int lo = 0; lo < k.nPts;) {
        // the batch: the points with indices in [lo, hi)
        int hi = k.nPts;
        for (;;) {
            int sh = 0;
            while ((hi - lo - 1) >> sh >= kBuckets) ++sh;
            __syncthreads();   // what is in the LDS has been used
            *reinterpret_cast<int4 *>(&L.count[4 * t]) = make_int4(0, 0, 0, 0);
            __syncthreads();
            each([&](int v) {
                if (v >= lo && v < hi) atomicAdd(&L.count[(v - lo) >> sh], 1);
            });
            __syncthreads();
            // how many of the leading buckets fit
            const int4 n = *reinterpret_cast<const int4 *>(&L.count[4 * t]);
            int run = n.x + n.y + n.z + n.w;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int o = __shfl_up(run, d, 64);
                if (lane >= d) run += o;
            }
            if (lane == 63) L.wave[t >> 6] = run;
            __syncthreads();
            for (int w = 0; w < t >> 6; ++w) run += L.wave[w];
            int fit = (run <= kPartPts) + (run - n.w <= kPartPts) + (run - n.w - n.z <= kPartPts) +
                      (run - n.w - n.z - n.y <= kPartPts);
#pragma unroll
            for (int d = 32; d > 0; d >>= 1) fit += __shfl_xor(fit, d, 64);
            if (lane == 0) L.low[t >> 6] = fit;
            __syncthreads();
            fit = L.low[0] + L.low[1] + L.low[2] + L.low[3];
            if (fit == kBuckets) break;
            if (fit > 0) {
                hi = lo + (fit << sh);
                break;
            }
            hi = lo + (1 << sh);   // more than one index: a point each
        }
        __syncthreads();
        if (t == 0) L.found = L.crowded = 0;
        for (int e = t; e < E * E * kFoldWords; e += 256) L.mask[0][e] = 0;
        *reinterpret_cast<int4 *>(&L.count[4 * t]) = make_int4(0, 0, 0, 0);
        __syncthreads();
        each([&](int v) {
            if (v >= lo && v < hi) {
                const int at = atomicAdd(&L.found, 1);
                L.idx[at] = v;
                L.cell[at] = (unsigned char)(t % E | t / E << 4);
            }
        });
        __syncthreads();
        const int total = L.found;
        if (total > 0) (void)fold_found(k, L, rec, total, T, sum);
        lo = hi;
    }
    if (lane < T * T && t < 3 * 64) L.res[t >> 6][(Y0 - TY + lane / T) * kTileN + X0 - TX + lane % T] = sum;
}

// UPDATE: the grid update of the node as well.  Clears the other list of cells
// for the next P2G.
template <bool UPDATE>
__global__ __launch_bounds__(256) void k_node_fold(KParams k, double *__restrict__ grid, const PointRec *__restrict__ rec,
                                                  const int *__restrict__ bucket, const int2 *__restrict__ cells,
                                                  int2 *__restrict__ cellsNext, const int *__restrict__ next,
                                                  double ind_x, double ind_y, int *__restrict__ nodeBin,
                                                  double *__restrict__ nodeF) {
    __shared__ FoldLds L;
    const int TX = (int)blockIdx.x * kTileN, TY = (int)blockIdx.y * kTileN;
    if (!fold_tile(k, L, rec, bucket, cells, kTileN, TX, TY, TX, TY)) {
        constexpr int T = kTileN / 2;
        for (int q = 0; q < 4; ++q) {
            const int X0 = TX + (q & 1) * T, Y0 = TY + (q >> 1) * T;
            if (!fold_tile(k, L, rec, bucket, cells, T, X0, Y0, TX, TY))
                fold_crowded(k, L, rec, bucket, cells, next, X0, Y0, TX, TY);
        }
    }
    __syncthreads();
    const int lane = threadIdx.x, X = TX + lane % kTileN, Y = TY + lane / kTileN;
    if (lane >= kTileNodes || X >= k.gridX || Y >= k.gridY) return;
    const int idx = X + Y * k.gridX;
    const double mass = L.res[0][lane];
    double v0 = L.res[1][lane], v1 = L.res[2][lane];
    if constexpr (UPDATE) {
        int bin = -1;
        double f0 = 0, f1 = 0;
        if (mass != 0) node_update(k, idx, mass, ind_x, ind_y, v0, v1, bin, f0, f1);
        nodeBin[idx] = bin;
        nodeF[2 * (size_t)idx] = f0;
        nodeF[2 * (size_t)idx + 1] = f1;
    }
    grid[idx] = mass;
    grid[k.gp + idx] = v0;
    grid[2 * k.gp + idx] = v1;
    cellsNext[idx] = make_int2(0, 0);
}

PointLists ordered_lists(const OrderedScratch &o) {
    return PointLists{reinterpret_cast<PointRec *>(o.rec), o.bucket, o.cells[o.flip], o.next};
}

hipError_t ordered_records(const KParams &k, const OrderedScratch &o, double *padGrid, hipStream_t s) {
    const int threads = k.nPts > 64 ? k.nPts : 64;   // 64: the rows' padding
    hipLaunchKernelGGL(k_point_records, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, k, ordered_lists(o),
                       padGrid);
    return hipGetLastError();
}

hipError_t ordered_fold(const KParams &k, double *grid, OrderedScratch &o, bool update, double ix, double iy,
                        hipStream_t s) {
    const PointLists l = ordered_lists(o);
    int2 *other = o.cells[o.flip ^ 1];
    const dim3 tiles((unsigned)((k.gridX + kTileN - 1) / kTileN), (unsigned)((k.gridY + kTileN - 1) / kTileN));
    if (update)
        hipLaunchKernelGGL(k_node_fold<true>, tiles, dim3(256), 0, s, k, grid, l.rec, l.bucket, l.cells, other, l.next, ix, iy,
                           o.nodeBin, o.nodeF);
    else
        hipLaunchKernelGGL(k_node_fold<false>, tiles, dim3(256), 0, s, k, grid, l.rec, l.bucket, l.cells, other, l.next, ix, iy,
                           o.nodeBin, o.nodeF);
    const hipError_t e = hipGetLastError();
    if (e == hipSuccess) o.flip ^= 1;
    return e;
}

}  // namespace icempm
