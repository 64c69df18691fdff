// MI355X (gfx950) kernels of the SPHERA v10 particle-interaction hot path.
//
// Layout in HBM (one context = one solve, capacity N particles), all arrays in
// cell-sorted order (cells ascending, particle id ascending inside a cell):
//   xm   double4 (x, y, z, mass)          x2 buffers (trajectory writes the other)
//   vel  double4 (vx, vy, vz, id)         x3 buffers (momentum -> smoothing -> sort)
//   rp   double2 (rho, p)                 x3 buffers (sort -> continuity -> smoothing)
//   lam  int32 laminar flag               x2 buffers
//   acc  double4, dden, vpres             outputs of the passes
//   xq int4 (x, y, z in units of P.lsb modulo 2^32, mass): separations of
//   the search and of the FP32-mixed pair sums
//   FP32-mixed: vf float4 (vx, vy, vz, rho - den0) x2 buffers, dr float rho - den0
//   Neighbour list, in groups of 8 entries per particle, a group rank
//   contiguous over the particles; count in nnb[i].  Tiles (below) that fit
//   the pair passes' LDS: 16-bit entries, the neighbour's slot of the
//   particle's tile times 16 (nb16_index), filled up to whole eights with the
//   particle itself.
//   Elsewhere: entry k of particle i at nb_index(N, i, k), the sorted index of
//   the k-th neighbour in bits 0..26 and its stencil cell code
//   (dx+1)+3(dy+1)+9(dz+1) in bits 27..31.
//
// FP64 kernels are compiled with -ffp-contract=off and evaluate every
// expression in the order of the cited reference line, so sums over a list in
// the reference's order reproduce the reference's values.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "sph_device.h"

namespace sph {

// ----------------------------------------------------------------------------
// grid helpers: CellNumber.f90:53-59, ParticleCellNumber.f90:52-62,
// CellIndices.f90:51-63 (1-based cell ids, 0 = outside)
// ----------------------------------------------------------------------------
__device__ __forceinline__ int d_cell_number(DPC& P, int i, int j, int k) {
    if (i < 1 || i > P.ncd[0] || j < 1 || j > P.ncd[1] || k < 1 || k > P.ncd[2]) return 0;
    return ((k - 1) * P.ncd[1] + (j - 1)) * P.ncd[0] + i;
}
__device__ __forceinline__ int d_particle_cell(DPC& P, double x, double y, double z) {
    const double xp = x - P.extr_lo[0];
    const double yp = y - P.extr_lo[1];
    const double zp = z - P.extr_lo[2];
    const int i = (int)ceil(xp / P.dcd[0]);
    const int k = (int)ceil(zp / P.dcd[2]);
    const int j = P.dim == 2 ? 1 : (int)ceil(yp / P.dcd[1]);  // :59-61 (2D: j = 1)
    return d_cell_number(P, i, j, k);
}
// x / d for 0 <= x < 2^30 from inv = 1.0 / d: (x + 1/2) / d is at least 1/(2 d)
// away from an integer, far above the product's rounding
__device__ __forceinline__ int div_inv(int x, double inv) { return (int)(((double)x + 0.5) * inv); }
__device__ __forceinline__ void d_cell_indices(DPC& P, int nc, int& i, int& j, int& k) {
    const int nij = P.ncd[0] * P.ncd[1];
    k = div_inv(nc - 1, P.inv_nij) + 1;
    const int ncij = nc - nij * (k - 1);
    j = div_inv(ncij - 1, P.inv_ni) + 1;
    i = ncij - P.ncd[0] * (j - 1);
}

// 8 XCDs each with their own L2: consecutive workgroups are dispatched round
// robin over the XCDs, so remap them to give every XCD one contiguous range
// of cell-sorted particles (their neighbour data then share that XCD's L2).
__device__ __forceinline__ int xcd_block(int nblocks) {
    const int b = blockIdx.x;
    const int per = (nblocks + 7) >> 3;
    const int xcd = b & 7;
    const int r = b >> 3;
    const int full = nblocks - (per - 1) * 8;  // XCDs that get `per` blocks
    int base;
    if (xcd < full) base = xcd * per;
    else base = full * per + (xcd - full) * (per - 1);
    return base + r;
}

// ----------------------------------------------------------------------------
// kernel function values: CalcVarLength.f90:243-265
// ----------------------------------------------------------------------------
struct K64 { double K1, K2, K3, W; };

__device__ __forceinline__ void kvals64(DPC& P, double rij, bool need12, bool need3,
                                        bool needW, K64& K) {
    const double rij2 = rij;
    const double r = sqrt(rij);
    const double q = r / P.h;
    const double q2 = rij2 / P.squareh;
    const int iq = (int)q;
    K.K1 = K.K2 = K.K3 = K.W = 0.0;
    if (iq >= 2) return;
    const double denom = 1.0 / (r + P.eta);
    if (need12) {
        double gm = -2.0 * q + 1.5 * q2;
        if (iq > 0) gm = -gm + q2 - 2.0;
        gm = gm * P.ke_coef;
        K.K1 = gm * denom;
        K.K2 = K.K1 / (rij2 + P.eta2);
    }
    if (need3) {
        double gw = -12.0 - 3.0 * q2 + 12.0 * q;
        gw = gw * P.kacl_coef;
        K.K3 = gw * denom;
    }
    if (needW) {
        double wu = 0.666666667 + q2 * (q * 0.5 - 1.0);
        if (iq > 0) wu = (2.0 - q) * (2.0 - q) * (2.0 - q) * 0.166666666667;
        K.W = wu * P.coefke;
    }
}

// The pair loops form the terms of two list entries side by side: an FP64
// operation's result is ready after several issue slots, and two wavefronts a
// SIMD (what the registers and the LDS leave) do not fill them.
using d2 = double __attribute__((ext_vector_type(2)));
__device__ __forceinline__ d2 fma2(d2 a, d2 b, d2 c) { return __builtin_elementwise_fma(a, b, c); }

// FP64 quotients and roots of the pair loops, correctly rounded as `/` and
// sqrt() are, without the scaling steps those take for operands near the ends
// of the exponent range: Newton's iteration for the reciprocal and Markstein's
// final correction, q + (a - d q) y with y = 1/d (P. Markstein, "Computation of
// elementary functions on the IBM RISC System/6000 processor", 1990); for the
// root Goldschmidt's iteration (R. E. Goldschmidt, "Applications of division by
// convergence", 1964) and the residual's correction.  A divisor that several
// quotients share is inverted once.
__device__ __forceinline__ d2 newton64(d2 d, d2 y) { return fma2(fma2(-d, y, d2(1.0)), y, y); }
__device__ __forceinline__ d2 inv64(d2 d) {
    return newton64(d, newton64(d, d2{__builtin_amdgcn_rcp(d.x), __builtin_amdgcn_rcp(d.y)}));
}
__device__ __forceinline__ d2 quot64(d2 a, d2 d, d2 y) {
    const d2 q = a * y;
    return fma2(fma2(-d, q, a), y, q);
}
// with zeros, infinities and NaN as `/` gives them
__device__ __forceinline__ d2 div64(d2 a, d2 d, d2 y) {
    const d2 q = quot64(a, d, y);
    return d2{__builtin_amdgcn_div_fixup(q.x, d.x, a.x), __builtin_amdgcn_div_fixup(q.y, d.y, a.y)};
}
__device__ __forceinline__ d2 sqrt64(d2 x) {
    const d2 y = {__builtin_amdgcn_rsq(x.x), __builtin_amdgcn_rsq(x.y)};
    d2 g = x * y, h = 0.5 * y;
    const d2 e = fma2(-h, g, d2(0.5));
    g = fma2(g, e, g);
    h = fma2(h, e, h);
    g = fma2(fma2(-g, g, x), h, g);
    g = fma2(fma2(-g, g, x), h, g);
    auto ends = [](double a, double r) { return a > 0.0 && a < __builtin_inf() ? r : a; };
    return d2{ends(x.x, g.x), ends(x.y, g.y)};
}

// lane U's value for lane 0 of each group of up to 16 lanes (the other lanes: any)
template <int U>
__device__ __forceinline__ double group_lane(double v) {
    if constexpr (U == 0) return v;
    else  // row_shl: lane l of a row of 16 takes lane l + U
        return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), 0x100 + U, 0xF, 0xF, true),
                                __builtin_amdgcn_mov_dpp(__double2loint(v), 0x100 + U, 0xF, 0xF, true));
}
// adds lane 0's, 1's, .. lane G-1's terms (each lane's t, then its more) to
// lane 0's sums, in that order
template <int G, int U = 0, int NS, class... More>
__device__ __forceinline__ void add_lanes(double (&sum)[NS], const double (&t)[NS], const More&... more) {
#pragma unroll
    for (int c = 0; c < NS; ++c) {
        sum[c] = sum[c] + group_lane<U>(t[c]);
        ((sum[c] = sum[c] + group_lane<U>(more[c])), ...);
    }
    if constexpr (U + 1 < G) add_lanes<G, U + 1>(sum, t, more...);
}

// LDS written by one lane of a wavefront is read by another: the barrier alone
// orders the lanes but not the compiler's LDS accesses
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// kvals64 of two pairs without branches (a wavefront's lanes differ), its
// quotients by the reciprocals of the constants
struct K64x2 { d2 K1, K2, K3, W; };
__device__ __forceinline__ K64x2 kvals64x2(DPC& P, d2 rij2, bool need12, bool need3, bool needW) {
    const d2 r = sqrt64(rij2);
    const d2 q = quot64(r, d2(P.h), d2(P.inv_h));
    const d2 q2 = quot64(rij2, d2(P.squareh), d2(P.inv_squareh));
    auto near = [&](double k) { return d2{q.x >= 2.0 ? 0.0 : k, q.y >= 2.0 ? 0.0 : k}; };
    auto part = [&](d2 outer, d2 inner) { return d2{q.x >= 1.0 ? outer.x : inner.x, q.y >= 1.0 ? outer.y : inner.y}; };
    K64x2 K;
    K.K1 = K.K2 = K.K3 = K.W = d2(0.0);
    d2 denom = d2(0.0);
    if (need12 || need3) {
        const d2 d = r + P.eta;
        denom = quot64(d2(1.0), d, inv64(d));
    }
    if (need12) {
        d2 gm = -2.0 * q + 1.5 * q2;
        gm = part(-gm + q2 - 2.0, gm);
        gm = gm * near(P.ke_coef);
        K.K1 = gm * denom;
        const d2 d = rij2 + P.eta2;
        K.K2 = quot64(K.K1, d, inv64(d));
    }
    if (need3) {
        d2 gw = -12.0 - 3.0 * q2 + 12.0 * q;
        gw = gw * near(P.kacl_coef);
        K.K3 = gw * denom;
    }
    if (needW) {
        const d2 a = 0.666666667 + q2 * (q * 0.5 - 1.0), b = (2.0 - q) * (2.0 - q) * (2.0 - q) * 0.166666666667;
        K.W = part(b, a) * near(P.coefke);
    }
    return K;
}

// ----------------------------------------------------------------------------
// SA-SPH geometry: LocalNormalCoordinates.f90:55-87 + IsPointInternal.f90
// ----------------------------------------------------------------------------
// IsPointInternal.f90 on the face's precomputed constants (kept in registers
// by the callers that test many points of one face)
struct PIC {
    double pu, a0, b0, c0, a1, b1, c1;
    int fkod;
};
__device__ __forceinline__ PIC pic_of(const DFace& F) {
    return PIC{F.pu, F.pA[0], F.pB[0], F.pC[0], F.pA[1], F.pB[1], F.pC[1], F.nodes - 2};
}
__device__ __forceinline__ bool d_point_internal(const PIC& c, double px0, double px1) {
    const double csi0 = (c.a0 + c.b0 * px0 + c.c0 * px1) * c.pu;
    const double csi1 = (c.a1 + c.b1 * px0 + c.c1 * px1) * c.pu;
    const double csi2 = 1.0 - (csi0 + csi1);
    const bool in01 = !(csi0 < 0.0 || csi0 > 1.0) && !(csi1 < 0.0 || csi1 > 1.0);
    if (c.fkod == 1) return in01 && !(csi2 < 0.0 || csi2 > 1.0);
    if (c.fkod == 2) return in01;
    return false;
}
__device__ __forceinline__ bool d_point_internal(const DFace& F, double px0, double px1) {
    return d_point_internal(pic_of(F), px0, px1);
}

// ----------------------------------------------------------------------------
// Tiles: the grid is cut into boxes of P.tdim cells.  The particles of a tile
// (home) and those of the cells around it (halo) are, row by row (fixed j, k;
// consecutive cells of a row are consecutive in memory), the tile's slots: a
// particle's neighbours all have a slot of its tile.  Where the slots fit the
// LDS of the pair passes (P.tcap), the neighbour lists hold 16-bit slot
// offsets; elsewhere 32-bit sorted indices with the stencil code.
// ----------------------------------------------------------------------------
// slots: 2, 3 and 4 workgroups a CU of 32 bytes a slot, 1, 1 and 2 of 64
constexpr int TILE_CAP_L = 2496, TILE_CAP_M = 1632, TILE_CAP_S = 1216, TILE_CAP_0 = 16;
constexpr int TILE_WG = 512;   // most threads of a pair pass
constexpr int TILE_U = 5;      // slots a thread stages at a time (FP64: 3)
constexpr int TILE_G2 = 40000;  // capacity below which two lanes take a particle
// FP64 passes that gather: capacity below which eight lanes take a particle,
// else four (DB-SPH steps, us: 2,000 particles eight 265, four 292, two 357;
// 70,000 eight 611, four 582, two 623; the four passes: 9,000 eight 81, four 88,
// two 133; 54,000 of twice water's density 331, 317, 327; 576,000 1834, 1375, 1442)
constexpr int TILE_G8 = 20000;
// tiles of water a solve is cut into (choose_tile); FP64
constexpr int TILE_MIN = 300, TILE_MIN2 = 200, TILE_MIN_L = 500;
constexpr int TILE_MIN64 = 130, TILE_MIN64_2 = 150;
struct TileS {
    int g[64];      // row r: sorted index of its first particle
    int l[65];      // its first slot; l[rows] the number of slots
    int h0[64];     // home part: sorted index of its first particle
    int hp[65];     // and home particles before the row; hp[rows] their number
};

// rows of a tile with its halo, at most 64 (choose_tile)
__device__ __forceinline__ int tile_rows(DPC& P) { return (P.tdim[1] + 2) * (P.tdim[2] + 2); }

// row `lane` of the tile (ti, tj, tk): its slot range and home range
__device__ __forceinline__ void tile_row(DPC& P, const int* __restrict__ start, int ti, int tj, int tk,
                                         int lane, int& g0, int& g1, int& h0, int& h1) {
    g0 = g1 = h0 = h1 = 0;
    const int ry = P.tdim[1] + 2;
    if (lane >= ry * (P.tdim[2] + 2)) return;
    const int rk = div_inv(lane, P.inv_ry), rj = lane - rk * ry;
    const int ni = P.ncd[0], nj = P.ncd[1], nk = P.ncd[2];
    const int i0 = ti * P.tdim[0] + 1, i1 = min(i0 + P.tdim[0] - 1, ni);
    const int j = tj * P.tdim[1] + rj, k = tk * P.tdim[2] + rk;
    if (j < 1 || j > nj || k < 1 || k > nk) return;
    const int rb = P.koff + ((k - 1) * nj + (j - 1)) * ni - 1;
    g0 = start[rb + max(i0 - 1, 1)];
    g1 = start[rb + min(i1 + 1, ni) + 1];
    if (rj >= 1 && rj <= P.tdim[1] && rk >= 1 && rk <= P.tdim[2]) {
        h0 = start[rb + i0];
        h1 = start[rb + i1 + 1];
    }
}

// the tile of a context's list entry: coordinates in its segment's tile grid
__device__ __forceinline__ void tile_coords(DPC& P, int id, int& ti, int& tj, int& tk) {
    const int t = id - P.toff;
    tk = div_inv(t, P.inv_ntij);
    const int r = t - tk * P.ntile[0] * P.ntile[1];
    tj = div_inv(r, P.inv_nti);
    ti = r - tj * P.ntile[0];
}

// ----------------------------------------------------------------------------
// sort: OrdGrid1.f90:58-105 as a device counting sort.  The particles arrive
// almost in cell order (they moved less than a cell since the last sort), so
// a workgroup's 256 particles fall in a narrow window of cells: it counts
// them in an LDS histogram and issues one global atomic per occupied cell.
// Inside the window a particle's rank among the workgroup's particles of its
// cell follows the thread order, so particles that stay in their cell keep
// their previous (ascending-id) order, in which k_gather compares few ids.
// ----------------------------------------------------------------------------
constexpr int HIST_W = 512;
constexpr int SCAN_B = 4096;  // keys per scan block (HIST_W < SCAN_B)

// Segmented contexts (SG): the workgroup's segment comes from the slot-block
// map; slots, keys, ids and the removal list are the segment's.
template <bool SG>
__global__ __launch_bounds__(256) void k_cell_count(Seg S, const double4* __restrict__ xm,
                                                    const double4* __restrict__ vel,
                                                    int* __restrict__ key, int* __restrict__ slot,
                                                    int* __restrict__ cnt, int* __restrict__ idslot,
                                                    int* __restrict__ rmids, int* iscal,
                                                    int* __restrict__ gone, int* ntile, int* __restrict__ bsum, int nrep, int nsb) {
    __shared__ int base[HIST_W];
    __shared__ int part[2];  // particles in the two scan blocks that the window can touch
    __shared__ int wcnt[4][HIST_W];  // particles of each window cell per wave
    __shared__ int cmin;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int sg = SG ? __builtin_amdgcn_readfirstlane(S.pblk[(blockIdx.x * blockDim.x) >> 8]) : 0;
    DPC& P = S.P[sg];
    iscal += sg * IS_COUNT;
    rmids += sg * RM_CAP;
    const int n = iscal[IS_N];
    if (i == 0) ntile[0] = ntile[1] = 0;  // k_scatter counts the tiles
    bsum += (blockIdx.x % nrep) * nsb;
    for (int b = threadIdx.x; b < HIST_W; b += blockDim.x)
        for (int w = 0; w < 4; ++w) wcnt[w][b] = 0;
    if (threadIdx.x == 0) cmin = 0x7fffffff;
    if (threadIdx.x < 2) part[threadIdx.x] = 0;
    __syncthreads();
    int k = -1;
    if (i - P.base < n) {
        const double4 x = xm[i];
        const int c = d_particle_cell(P, x.x, x.y, x.z);
        const int id = (int)vel[i].w;
        idslot[P.base + id] = i;
        // the last trajectory step left through an open face: cella = -1 (read once)
        const bool out = gone[i] != 0;
        if (out) gone[i] = 0;
        if (c <= 0 || out) {  // out of the grid or cella <= 0: removed (OrdGrid1.f90:66-82)
            k = P.koff + P.nmax;
            atomicAdd(&iscal[IS_REMOVED], 1);
            const int q = atomicAdd(&iscal[IS_NRM], 1);
            if (q < RM_CAP) rmids[q] = id;
        } else {
            k = P.koff + c - 1;
            atomicMin(&cmin, k);
        }
        key[i] = k;
    }
    __syncthreads();
    const int c0 = cmin;
    int loc = -1, rank = 0;
    if (k >= 0) {
        const int d = k - c0;
        if (k < P.koff + P.nmax && d < HIST_W) {
            loc = d;
        } else {
            slot[i] = atomicAdd(&cnt[k], 1);
            atomicAdd(&bsum[k / SCAN_B], 1);
        }
    }
    // rank within the wave among the lanes of the same window cell, one
    // ballot per distinct cell of the wave
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const unsigned long long below = (1ull << lane) - 1ull;
    unsigned long long todo = __ballot(loc >= 0);
    while (todo) {
        const int lead = __ffsll((long long)todo) - 1;
        const int dk = __shfl(loc, lead, 64);
        const unsigned long long m = __ballot(loc == dk);
        if (loc == dk) rank = __popcll(m & below);
        if (lane == lead) wcnt[wid][dk] = __popcll(m);
        todo &= ~m;
    }
    __syncthreads();
    if (loc >= 0)
        for (int w = 0; w < wid; ++w) rank += wcnt[w][loc];
    for (int b = threadIdx.x; b < HIST_W; b += blockDim.x) {
        const int tot = wcnt[0][b] + wcnt[1][b] + wcnt[2][b] + wcnt[3][b];
        if (tot > 0) {
            base[b] = atomicAdd(&cnt[c0 + b], tot);
            atomicAdd(&part[(c0 + b) / SCAN_B - c0 / SCAN_B], tot);
        }
    }
    __syncthreads();
    if (loc >= 0) slot[i] = base[loc] + rank;
    if (threadIdx.x < 2 && part[threadIdx.x]) atomicAdd(&bsum[c0 / SCAN_B + threadIdx.x], part[threadIdx.x]);
}

// wave64 inclusive scan
__device__ __forceinline__ int wave_incl_scan(int v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}

// Ids after the removals of this sort, as OrdGrid1.f90:62-83 leaves pg: the
// first loop walks npi upwards; a particle out of the grid is overwritten by
// pg(nag), nag decreases and the same npi is tested again.  So, for the removed
// ids r in ascending order while r < nag: the last particle moves to r unless
// it is itself removed (then it is dropped and the next last is tried).  One
// lane; removals are rare (particles leaving a closed tank).
// Segmented contexts: one lane per segment.
__device__ void renumber(const Seg& S, int sg, int* __restrict__ rmids, const int* __restrict__ idslot,
                         double4* __restrict__ vel, int* iscal) {
    const int pbase = S.P[sg].base;
    iscal += sg * IS_COUNT;
    rmids += sg * RM_CAP;
    const int m = iscal[IS_NRM];
    if (m == 0) return;
    if (m > RM_CAP) {
        iscal[IS_RM_OVERFLOW] = 1;
        return;
    }
    for (int a = 1; a < m; ++a) {  // insertion sort, ascending
        const int v = rmids[a];
        int b = a - 1;
        while (b >= 0 && rmids[b] > v) {
            rmids[b + 1] = rmids[b];
            --b;
        }
        rmids[b + 1] = v;
    }
    int nag = iscal[IS_N];
    for (int q = 0; q < m; ++q) {
        const int r = rmids[q];
        if (r >= nag) break;
        for (;;) {
            const int last = --nag;
            if (last == r) break;
            int lo = 0, hi = m;  // is `last` removed too?
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (rmids[mid] < last) lo = mid + 1;
                else hi = mid;
            }
            if (lo < m && rmids[lo] == last) continue;
            vel[idslot[pbase + last]].w = (double)r;
            break;
        }
    }
}

// Cell starts: exclusive scan of the counts, a block of SCAN_B keys per
// workgroup.  k_cell_count has summed the counts by block (in nrep copies:
// its workgroups run through the keys together, and on one copy their atomics
// queued, 45 against 18 us at 576,000 particles), so a workgroup adds up the
// blocks before its own and scans its keys: one launch for what took
// three (local scan, scan of the totals, their addition; a launch costs 4.5 us
// in a step whatever it does, and the sort had ten: now four).  Segmented contexts: a
// segment's slots begin at its base, and the particles before its keys are
// the earlier segments' particles.  The last workgroup renumbers the ids
// after removals.
template <bool SG>
__global__ __launch_bounds__(256) void k_cell_scan(Seg S, const int* __restrict__ cnt, int* __restrict__ start,
                                                   const int* __restrict__ bsum, int nrep, int nsb, int m, int* __restrict__ rmids,
                                                   const int* __restrict__ idslot, double4* __restrict__ vel,
                                                   int* iscal) {
    if (blockIdx.x == gridDim.x - 1) {
        for (int sg = threadIdx.x; sg < (SG ? S.nseg : 1); sg += blockDim.x) renumber(S, sg, rmids, idslot, vel, iscal);
        return;
    }
    __shared__ int wsum[4], wtot[4];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    int before = 0;
    // nrep is a power of two up to 16: copy t % nrep, blocks t / nrep + 256 / nrep * ...
    for (int b = threadIdx.x / nrep; b < (int)blockIdx.x; b += 256 / nrep)
        before += bsum[(threadIdx.x & (nrep - 1)) * nsb + b];
    constexpr int U = SCAN_B / 256;
    const int k0 = blockIdx.x * SCAN_B + threadIdx.x * U;
    // the particles of the segments before the workgroup's first are taken off again
    const int sg0 = SG ? S.kblk[(blockIdx.x * SCAN_B) >> 8] : 0;
    for (int q = threadIdx.x; q < sg0; q += 256) before -= iscal[q * IS_COUNT + IS_N];
    int v[U], tsum = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        v[u] = k0 + u < m ? cnt[k0 + u] : 0;
        tsum += v[u];
    }
    for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o, 64);
    const int incl = wave_incl_scan(tsum);
    if (lane == 63) wsum[wid] = incl;
    if (lane == 0) wtot[wid] = before;
    __syncthreads();
    int run = wtot[0] + wtot[1] + wtot[2] + wtot[3] + incl - tsum;
    for (int w = 0; w < wid; ++w) run += wsum[w];
    if (SG && k0 < m) {  // a thread's keys lie in one 256-block, hence in one segment
        const int sg = S.kblk[k0 >> 8];
        int earlier = 0;
        for (int q = sg0; q < sg; ++q) earlier += iscal[q * IS_COUNT + IS_N];
        run += S.P[sg].base - earlier;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (k0 + u < m) start[k0 + u] = run;
        run += v[u];
    }
}

// Workgroups past the first nsb list the tiles that hold particles (a tile per
// lane, ids in ascending order within a workgroup) instead.
template <bool SG>
__global__ __launch_bounds__(256) void k_scatter(Seg S, const int* __restrict__ key,
                                                 const int* __restrict__ slot, const int* __restrict__ start,
                                                 const double4* __restrict__ vel, int* __restrict__ perm,
                                                 int* __restrict__ pid, const int* iscal, int nsb,
                                                 int* __restrict__ tlist, int* ntile) {
    if ((int)blockIdx.x >= nsb) {
        __shared__ int wn[4], first;
        const int b = blockIdx.x - nsb, id = b * 256 + threadIdx.x;
        DPC& P = S.P[SG ? __builtin_amdgcn_readfirstlane(S.tblk[b]) : 0];
        int n = 0;
        if (id - P.toff < P.ntile[0] * P.ntile[1] * P.ntile[2]) {
            int ti, tj, tk;
            tile_coords(P, id, ti, tj, tk);
            const int i0 = ti * P.tdim[0], i1 = min(i0 + P.tdim[0], P.ncd[0]);
            const int j1 = min((tj + 1) * P.tdim[1], P.ncd[1]), k1 = min((tk + 1) * P.tdim[2], P.ncd[2]);
            for (int k = tk * P.tdim[2]; k < k1; ++k)
                for (int j = tj * P.tdim[1]; j < j1; ++j) {
                    const int rb = P.koff + (k * P.ncd[1] + j) * P.ncd[0];
                    n += start[rb + i1] - start[rb + i0];
                }
        }
        const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
        const unsigned long long m = __ballot(n > 0);
        if (lane == 0) wn[wid] = __popcll(m);
        __syncthreads();
        // (no atomic for 256 empty tiles: of a large grid most are, and the atomics queue)
        const int some = wn[0] + wn[1] + wn[2] + wn[3];
        if (some == 0) return;
        if (threadIdx.x == 0) first = atomicAdd(ntile, some);
        __syncthreads();
        int at = first + __popcll(m & ((1ull << lane) - 1ull));
        for (int w = 0; w < wid; ++w) at += wn[w];
        if (n > 0) tlist[at] = id;
        return;
    }
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int sg = SG ? __builtin_amdgcn_readfirstlane(S.pblk[(blockIdx.x * blockDim.x) >> 8]) : 0;
    const int pbase = S.P[sg].base;
    if (i - pbase >= iscal[sg * IS_COUNT + IS_N]) return;
    const int d = start[key[i]] + slot[i];
    perm[d] = i;
    pid[d] = (int)vel[i].w;
}

// A coordinate relative to the grid's corner in units of lsb, modulo 2^32:
// lsb_diff of two particles' values is their separation wherever that is below
// 2^31 lsb (eight cells).
__device__ __forceinline__ int lsb_units(double x, double inv) {
    const double t = rint(x * inv);
    return (int)(uint32_t)(t - floor(t * 0x1p-32) * 0x1p32);
}

// Permutes the state into the new order and writes the integer positions (the
// neighbour test's in both precisions).  Inside a cell the order is by
// ascending particle id, which OrdGrid1's 4th loop produces (NPartOrd), hence
// the reference's neighbour-list order: a particle's place is the number of
// smaller ids among the cell's (18) particles, whose ids are a few cache lines
// for a wavefront.  (A kernel that sorted each cell's run by insertion before
// this one took 33 us at 576,000 particles and 17 at 1,440.)
// Also clears the counters that the next sort counts in: m keys, their
// scan blocks, the removed ids, the boundary table's work counter.
template <bool SG>
__global__ void k_gather(Seg S, const int* __restrict__ perm, const int* __restrict__ pid,
                         const int* __restrict__ key,
                         const double4* __restrict__ xm_s, const double4* __restrict__ vel_s,
                         const double2* __restrict__ rp_s, const int* __restrict__ lam_s,
                         const double4* __restrict__ acc_s, double4* __restrict__ xm_d,
                         double4* __restrict__ vel_d, double2* __restrict__ rp_d,
                         int* __restrict__ lam_d, double4* __restrict__ acc_d,
                         int* __restrict__ cell_d, int4* __restrict__ xq, float4* __restrict__ vf,
                         const int* __restrict__ start, int* iscal,
                         const double* __restrict__ dd_s, double* __restrict__ dd_d,
                         const double* __restrict__ vp_s, double* __restrict__ vp_d,
                         const double* __restrict__ g_s, double* __restrict__ g_d,
                         const double* __restrict__ h_s, double* __restrict__ h_d,
                         int* __restrict__ cnt, int m, int* __restrict__ bsum, int nbsum, int* nwork) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    const int sg = SG ? __builtin_amdgcn_readfirstlane(S.pblk[(blockIdx.x * blockDim.x) >> 8]) : 0;
    DPC& P = S.P[sg];
    iscal += sg * IS_COUNT;
    for (int k = q; k < m; k += gridDim.x * blockDim.x) cnt[k] = 0;
    for (int k = q; k < nbsum; k += gridDim.x * blockDim.x) bsum[k] = 0;
    if (q == 0) *nwork = 0;
    const int nin = start[P.koff + P.nmax] - P.base;  // particles still inside the grid
    if (q == P.base) {
        iscal[IS_NPREV] = iscal[IS_N];
        iscal[IS_N] = nin;
        iscal[IS_NRM] = 0;
    }
    if (q - P.base >= nin) return;
    const int s = perm[q], id = pid[q];
    const int b = start[key[s]], e = start[key[s] + 1];
    int p = b;
    for (int t = b; t < e; ++t) p += pid[t] < id;
    const double4 x = xm_s[s];
    const double4 v = vel_s[s];
    const double2 r = rp_s[s];
    xm_d[p] = x;
    vel_d[p] = v;
    rp_d[p] = r;
    lam_d[p] = lam_s[s];
    acc_d[p] = acc_s[s];
    if (dd_s) {  // explicit RK1: dden and vpres of the step end in the new order
        dd_d[p] = dd_s[s];
        vp_d[p] = vp_s[s];
    }
    if (g_s) {  // DB-SPH: Gamma and dShep travel with the particle
        g_d[p] = g_s[s];
        h_d[p] = h_s[s];
    }
    const int c = key[s] - P.koff + 1;
    cell_d[p] = c;
    xq[p] = make_int4(lsb_units(x.x - P.extr_lo[0], P.inv_lsb), lsb_units(x.y - P.extr_lo[1], P.inv_lsb),
                      lsb_units(x.z - P.extr_lo[2], P.inv_lsb), __float_as_int((float)x.w));
    if (P.f32) vf[p] = make_float4((float)v.x, (float)v.y, (float)v.z, (float)(r.x - P.den0));
}

// ----------------------------------------------------------------------------
// neighbour lists: CalcVarLength.f90:133-242 — stencil y -> x -> z, ascending
// particle id in a cell, r^2 <= (2h)^2 in FP64, self included, truncation past
// NMAXPARTJ.  Candidates are tested in FP32 on separations of the integer
// positions; a candidate whose FP32 r^2 lies within a relative 4e-5 of (2h)^2
// is decided by the reference's FP64 expression on the FP64 positions, so the
// lists are exactly the reference's.
// ----------------------------------------------------------------------------
// One lane per particle, candidates from global memory, every one that FP32
// finds near decided in FP64 (P.far_y).  aux: per stencil cell in list order
// what turns a sorted index into its list entry.  Every accepted candidate is
// counted; the first NMAXPARTJ are stored, as in the reference.  Returns the count.
__device__ int nb_particle_global(DPC& P, int p, const double4* __restrict__ xm,
                                  const int4* __restrict__ xq, const int* __restrict__ cell,
                                  const int* __restrict__ start, uint32_t* __restrict__ nbr,
                                  const int* aux, bool fits, float hi) {
    const int ni = P.ncd[0], nj = P.ncd[1], nk = P.ncd[2];
    const int mj = P.nmaxpartj;
    const size_t N = P.cap;
    uint16_t* nbr16 = reinterpret_cast<uint16_t*>(nbr);
    int ic, jc, kc;
    d_cell_indices(P, cell[p], ic, jc, kc);
    const int4 xi = xq[p];
    const double4 xi64 = xm[p];
    int k = 0;
    for (int t = 0; t < 27; ++t) {
        const int jj = jc + t / 9 - 1, ii = ic + (t / 3) % 3 - 1, kk = kc + t % 3 - 1;
        if (ii < 1 || ii > ni || jj < 1 || jj > nj || kk < 1 || kk > nk) continue;
        const int key = P.koff + ((kk - 1) * nj + (jj - 1)) * ni + ii - 1;
        for (int m = start[key]; m < start[key + 1]; ++m) {
            const int4 xj = xq[m];
            const float r0 = (float)lsb_diff(xi.x, xj.x), r1 = (float)lsb_diff(xi.y, xj.y),
                        r2 = (float)lsb_diff(xi.z, xj.z);
            const float rr = __builtin_fmaf(r0, r0, __builtin_fmaf(r1, r1, r2 * r2));
            if (rr > hi) continue;
            const double4 xj64 = xm[m];
            const double d0 = xi64.x - xj64.x;
            const double d1 = xi64.y - xj64.y;
            const double d2 = xi64.z - xj64.z;
            if (d0 * d0 + d1 * d1 + d2 * d2 > P.square_doubleh) continue;
            if (k < mj) {
                if (fits) nbr16[nb16_index(N, p, k)] = (uint16_t)((m + aux[t]) << 4);
                else nbr[nb_index(N, p, k)] = (uint32_t)m | (uint32_t)aux[t];
            }
            ++k;
        }
    }
    if (fits)
        for (int q = min(k, mj); q & 7; ++q) nbr16[nb16_index(N, p, q)] = (uint16_t)((p + aux[13]) << 4);
    return k;
}

// One wavefront per cell.  All particles of a cell share the candidates of its
// 27 stencil cells (475 at 17.6 particles per cell), in the same order: the
// lanes hold them in registers (candidate 64 q + lane in chunk q), relative
// to the cell's first particle, and the particles of the cell are taken one
// after the other.  With c = |xj|^2 kept per candidate, the test
// c - 2 xi.xj <= (2h)^2 - |xi|^2 is three fused multiply-adds and a compare
// for 64 candidates; the hits of a chunk are a lane mask, so a hit's place in
// the list is the count of mask bits below it, and the list is built in LDS
// and stored in 16-byte pieces.  VALU issue bounds it: 9 instructions per 64
// candidates, against 19 per candidate and lane (with the append in the
// divergent branch of every test) for one lane per particle.
// 576,000 particles: 219 -> 163 us; a batch of eight solves, 536,000: 334 ->
// 152; 1,440 particles (one lane's 475 serial tests were the time): 71 -> 18 us.
//
// The FP32 test: a candidate's coordinates are within 2 dcd of the first
// particle, so with the rounding of the sums r^2 is within 3.5e-6 dcd^2; the
// guard band 4e-5 (2h)^2 (wider for cells larger than 2h) goes to the FP64 test.
// A wavefront takes the cells whose first particle lies in its NBC_SLOTS
// sorted slots: about one cell, so small solves spread over the chip.
// More candidates than the registers hold (27 cells of lattice water at h/dx of
// 1.4 and more, clusters) are taken in equal parts, one after the other, for 64
// particles of the cell at a time: a particle's count and the entries that do
// not fill a store yet wait in a register and in LDS for the next part.
// (One lane per particle over global memory before: 576,000 particles at h/dx of
// 1.4 831 -> 262 us, at 1.5 1550 -> 350; 72,000 189 -> 67, 216 -> 78; a cluster
// of twice the density 260 -> 91.)  A part has five to eight chunks: forms of
// nine and ten beside these spilled and took 163 -> 173 us from the common one.
// 2D solves whose particles differ in y take one lane per particle from global
// memory: two of them may lie whole wraps of the integer positions apart, so
// every candidate the FP32 test takes goes to the FP64 test.
constexpr int NBC_CH = 9;              // chunks of 64 candidates in registers
constexpr int NBC_MAX = 64 * NBC_CH;
// sorted slots per wavefront: small contexts, those of NBC_LARGE particles and more
// (us, 16 slots, 64: 72,000 particles 40, 59; 117,000 52, 61; 171,000 66, 72; 262,000
// 90, 87; 576,000 181, 162)
constexpr int NBC_SLOTS = 16, NBC_SLOTS_L = 64;
constexpr int NBC_LARGE = 200000;
constexpr int NBC_PAIRS = 64;          // pair counters, one 128-byte line each
constexpr int NBC_PSTRIDE = 16;

__device__ __forceinline__ float readlane_f(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// The cell's particles hb .. hb+hc-1 against its `total` candidates, NCH chunks
// of 64 (total <= 64 NCH).  A lane without a hit writes to the
// slot past the list, so a chunk's append has no branch.  FIT: 16-bit entries
// (the tile fits LDS).  Returns the sum of the list lengths without the
// particles themselves; over counts truncated lists.
// PART: one part of the candidates against the particles from h0 on, 64 at
// most: mine holds the lengths so far (lane u: particle h0 + u), tail the last
// length % 8 entries of each; last: the last part.
constexpr int NBC_VOID = NBC_MAX + 16;  // the slot of a lane without a hit, past the list and what fills it up
template <int NCH, bool FIT, bool PART = false>
__device__ __forceinline__ int nb_cell_lists(DPC& P, const double4* __restrict__ xm,
                                             const int4* __restrict__ xq, const uint32_t* cand, const int* aux,
                                             uint32_t* list32, int total, int hb, int hc, float lo, float hi,
                                             uint32_t* __restrict__ nbr, int* __restrict__ nnb, int& over,
                                             int h0 = 0, bool last = true, uint32_t* tail32 = nullptr,
                                             int* lengths = nullptr) {
    using E = typename std::conditional<FIT, uint16_t, uint32_t>::type;
    E* list = reinterpret_cast<E*>(list32);
    E* tail = reinterpret_cast<E*>(tail32);
    const int lane = threadIdx.x & 63;
    const int mj = P.nmaxpartj;
    const size_t N = P.cap;
    const int4 x0 = xq[hb];
    float cx[NCH], cy[NCH], cz[NCH], cq[NCH];
    uint32_t ce[NCH];
#pragma unroll
    for (int q = 0; q < NCH; ++q) {
        const int f = 64 * q + lane;
        ce[q] = f < total ? cand[f] : (uint32_t)hb;
    }
#pragma unroll
    for (int q = 0; q < NCH; ++q) {
        const int4 x = xq[ce[q] & NB_MASK];
        const int a = aux[ce[q] >> NB_SHIFT];
        ce[q] = FIT ? (uint32_t)((int)(ce[q] & NB_MASK) + a) << 4 : (ce[q] & NB_MASK) | (uint32_t)a;
        cx[q] = (float)lsb_diff(x.x, x0.x);
        cy[q] = (float)lsb_diff(x.y, x0.y);
        cz[q] = (float)lsb_diff(x.z, x0.z);
        const float r2 = __builtin_fmaf(cx[q], cx[q], __builtin_fmaf(cy[q], cy[q], cz[q] * cz[q]));
        cq[q] = 64 * q + lane < total ? r2 : 3.0e38f;
    }
    const int self = FIT ? aux[13] : 0;
    int pairs = 0;
    for (; h0 < hc; h0 += 64) {
        // the lane's own particle of the cell, as it enters the test
        float mx = 0.f, my = 0.f, mz = 0.f, tl = 0.f, th = 0.f;
        if (h0 + lane < hc) {
            const int4 x = xq[hb + h0 + lane];
            const float fx = (float)lsb_diff(x.x, x0.x), fy = (float)lsb_diff(x.y, x0.y),
                        fz = (float)lsb_diff(x.z, x0.z);
            const float r2 = __builtin_fmaf(fx, fx, __builtin_fmaf(fy, fy, fz * fz));
            mx = -2.0f * fx;
            my = -2.0f * fy;
            mz = -2.0f * fz;
            tl = lo - r2;
            th = hi - r2;
        }
        const int hn = min(64, hc - h0);
        int mine = PART ? *lengths : 0;  // list length of the lane's own particle
        for (int u = 0; u < hn; ++u) {
            const int p = hb + h0 + u;
            const float ax = readlane_f(mx, u), ay = readlane_f(my, u), az = readlane_f(mz, u);
            const float al = readlane_f(tl, u), ah = readlane_f(th, u);
            auto r2of = [&](int q) {
                return __builtin_fmaf(ax, cx[q], __builtin_fmaf(ay, cy[q], __builtin_fmaf(az, cz[q], cq[q])));
            };
            unsigned long long guard = 0ull;
            const int before = PART ? __builtin_amdgcn_readlane(mine, u) : 0;
            const int base = before & ~7;  // the list's first entry in LDS
            int k = before & 7;
            if (PART && lane < k) list[lane] = tail[8 * u + lane];
            auto append = [&](int q, bool in) {
                const unsigned long long m = __ballot(in);
                const int at = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                         __builtin_amdgcn_mbcnt_lo((uint32_t)m, k));
                list[in ? at : NBC_VOID] = (E)ce[q];
                k += __popcll(m);
                return m;
            };
#pragma unroll
            for (int q = 0; q < NCH; ++q) {
                const float r2 = r2of(q);
                guard |= __ballot(r2 <= ah) ^ append(q, r2 < al);
            }
            if (guard) {  // candidates in the guard band (1 particle in 100): the reference's FP64 test
                const double4 xi = xm[p];
                k = before & 7;
                wave_lds_sync();  // other lanes write the same places again
#pragma unroll
                for (int q = 0; q < NCH; ++q) {
                    const float r2 = r2of(q);
                    bool in = r2 < al;
                    if (!in && r2 <= ah) {
                        const double4 xj = xm[cand[64 * q + lane] & NB_MASK];
                        const double d0 = xi.x - xj.x;
                        const double d1 = xi.y - xj.y;
                        const double d2 = xi.z - xj.z;
                        in = !(d0 * d0 + d1 * d1 + d2 * d2 > P.square_doubleh);
                    }
                    append(q, in);
                }
            }
            const int room = mj - base;  // entries that the list still takes from `base` on
            // entries to store; the last group filled with the particle itself, as often as it is formed
            const int kn = PART ? max(0, min(last ? k : k & ~7, room)) : min(k, mj);
            const int end = PART ? min(k, room) : kn;
            wave_lds_sync();
            if (FIT && lane < 8 && (!PART || ((last || room < k) && room >= 0)))
                list[end + lane] = (E)((uint32_t)(p + self) << 4);
            wave_lds_sync();
            auto run = [&](int e) {  // 16 bytes of the list, stored as entries of either width
                uint4 v;
                __builtin_memcpy(&v, __builtin_assume_aligned(list + e, 16), 16);
                return v;
            };
            if constexpr (FIT) {
                for (int e = 8 * lane; e < kn; e += 512)
                    *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(nbr) + nb16_index(N, p, base + e)) = run(e);
            } else {
                for (int e = 4 * lane; e < kn; e += 256)
                    *reinterpret_cast<uint4*>(nbr + nb_index(N, p, base + e)) = run(e);
            }
            if (PART && lane < 8) tail[8 * u + lane] = list[(k & ~7) + lane];
            wave_lds_sync();
            const int len = last ? min(base + k, mj) : base + k;
            mine = lane == u ? len : mine;
            if (last) {
                pairs += len - 1;
                over += base + k > mj;
            }
        }
        if (last && lane < hn) nnb[hb + h0 + lane] = mine;
        if (PART) {
            *lengths = mine;
            break;
        }
    }
    return pairs;
}

template <bool SG>
__global__ __launch_bounds__(256, 4) void k_neighbours(Seg S, const double4* __restrict__ xm,
                                                    const int4* __restrict__ xq,
                                                    const int* __restrict__ cell,
                                                    const int* __restrict__ start,
                                                    uint32_t* __restrict__ nbr, int* __restrict__ nnb,
                                                    int* iscal, unsigned long long* pairs, int slots) {
    __shared__ uint32_t s_cand[4][NBC_MAX];  // a wave's candidates: sorted index | stencil cell in list order
    __shared__ __align__(16) uint32_t s_list[4][NBC_VOID + 4];  // the list of its current particle
    __shared__ uint32_t s_tail[4][64 * 8];  // candidates in parts: entries that wait for the next part
    __shared__ int s_aux[4][28];  // per stencil cell: sorted index to slot, or the stencil code's bits
    __shared__ int s_pairs[4];
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int vb = xcd_block(gridDim.x);
    const int sg = SG ? __builtin_amdgcn_readfirstlane(S.pblk[(vb * 4 * slots) >> 8]) : 0;
    DPC& P = S.P[sg];
    iscal += sg * IS_COUNT;
    const int n = iscal[IS_N];
    if (vb * 4 * slots - P.base >= n) return;
    const int ni = P.ncd[0], nj = P.ncd[1], nk = P.ncd[2];
    const float sq = (float)(P.square_doubleh * P.inv_lsb * P.inv_lsb);
    const float band = 4.0e-5f * fmaxf(1.0f, P.f_side * P.f_side / (float)P.square_doubleh);
    const float lo = sq * (1.0f - band), hi = sq * (1.0f + band);
    const int s0 = (vb * 4 + wid) * slots;
    uint32_t* cand = s_cand[wid];
    uint32_t* list = s_list[wid];
    int mypairs = 0, over = 0;
    int cl = 0;
    bool first = false;  // the lane's slot starts a cell
    if (lane < slots && s0 + lane - P.base < n) {
        cl = cell[s0 + lane];
        first = s0 + lane == P.base || cell[s0 + lane - 1] != cl;
    }
    int tile = -1, delta = 0;
    bool fits = false;
    unsigned long long todo = __ballot(first);
    while (todo) {
        const int l = __ffsll((long long)todo) - 1;
        todo &= todo - 1ull;
        int ic, jc, kc;
        d_cell_indices(P, __builtin_amdgcn_readlane(cl, l), ic, jc, kc);
        // lane r: row r of the cell's tile, its slots' offset from the sorted indices
        const int ti = div_inv(ic - 1, P.inv_tdim[0]), tj = div_inv(jc - 1, P.inv_tdim[1]),
                  tk = div_inv(kc - 1, P.inv_tdim[2]);
        const int id = __builtin_amdgcn_readfirstlane((tk * P.ntile[1] + tj) * P.ntile[0] + ti);
        if (id != tile) {
            tile = id;
            int g0, g1, h0, h1;
            tile_row(P, start, ti, tj, tk, lane, g0, g1, h0, h1);
            const int rincl = wave_incl_scan(g1 - g0);
            fits = __builtin_amdgcn_readlane(rincl, 63) <= P.tcap;
            delta = rincl - (g1 - g0) - g0;
        }
        // lane t: the t-th stencil cell in the order dy, dx, dz
        int b = 0, cnt = 0, row = 0;
        const int dy = lane / 9 - 1, dx = (lane / 3) % 3 - 1, dz = lane % 3 - 1;
        if (lane < 27) {
            const int ii = ic + dx, jj = jc + dy, kk = kc + dz;
            if (ii >= 1 && ii <= ni && jj >= 1 && jj <= nj && kk >= 1 && kk <= nk) {
                const int key = P.koff + ((kk - 1) * nj + (jj - 1)) * ni + ii - 1;
                b = start[key];
                cnt = start[key + 1] - b;
                row = (kk - tk * P.tdim[2]) * (P.tdim[1] + 2) + (jj - tj * P.tdim[1]);
            }
        }
        const int dt = __shfl(delta, row, 64);
        if (lane < 27) s_aux[wid][lane] = fits ? dt : (int)((uint32_t)((dx + 1) + 3 * (dy + 1) + 9 * (dz + 1)) << NB_SHIFT);
        const int incl = wave_incl_scan(cnt);
        const int total = __builtin_amdgcn_readlane(incl, 63);
        const int hb = __builtin_amdgcn_readlane(b, 13), hc = __builtin_amdgcn_readlane(cnt, 13);
        wave_lds_sync();
#define NB_LISTS(n, fit) mypairs += nb_cell_lists<n, fit>(P, xm, xq, cand, s_aux[wid], list, total, hb, hc, lo, hi, nbr, nnb, over)
#define NB_PART(n, fit)                                                                                               \
    mypairs += nb_cell_lists<n, fit, true>(P, xm, xq, cand, s_aux[wid], list, c1 - c0, hb, hc, lo, hi, nbr, nnb, over, \
                                           h0, c1 == total, s_tail[wid], &lengths)
        if (__builtin_expect(total > NBC_MAX || P.far_y, 0)) {
            if (P.far_y) {
                for (int q = lane; q < hc; q += 64) {
                    const int found = nb_particle_global(P, hb + q, xm, xq, cell, start, nbr, s_aux[wid], fits, hi);
                    const int k = min(found, P.nmaxpartj);
                    nnb[hb + q] = k;
                    if (found > k) atomicAdd(&iscal[IS_NB_OVERFLOW], 1);
                    atomicAdd(&pairs[(vb % NBC_PAIRS) * NBC_PSTRIDE], (unsigned long long)(k - 1));
                }
                wave_lds_sync();  // s_aux is reused
                continue;
            }
            const int chunks = (total + 63) >> 6, parts = (chunks + 7) / 8;
            const int per = (chunks + parts - 1) / parts;  // chunks of a part: 5 to 8
            for (int h0 = 0; h0 < hc; h0 += 64) {
                int lengths = 0;
                for (int c0 = 0; c0 < total; c0 += 64 * per) {
                    const int c1 = min(total, c0 + 64 * per);
                    const int first = incl - cnt;  // the lane's cell: its first candidate
                    for (int c = max(first, c0); c < min(incl, c1); ++c)
                        cand[c - c0] = (uint32_t)(b + c - first) | ((uint32_t)lane << NB_SHIFT);
                    wave_lds_sync();
                    if (per == 5) {
                        if (fits) NB_PART(5, true);
                        else NB_PART(5, false);
                    } else if (per == 6) {
                        if (fits) NB_PART(6, true);
                        else NB_PART(6, false);
                    } else if (per == 7) {
                        if (fits) NB_PART(7, true);
                        else NB_PART(7, false);
                    } else {
                        if (fits) NB_PART(8, true);
                        else NB_PART(8, false);
                    }
                }
            }
            continue;
        }
        for (int u = 0, pre = incl - cnt; u < cnt; ++u) cand[pre + u] = (uint32_t)(b + u) | ((uint32_t)lane << NB_SHIFT);
        wave_lds_sync();
        if (fits) {
            switch ((total + 63) >> 6) {
                case 1: NB_LISTS(1, true); break;
                case 2: NB_LISTS(2, true); break;
                case 3: NB_LISTS(3, true); break;
                case 4: NB_LISTS(4, true); break;
                case 5: NB_LISTS(5, true); break;
                case 6: NB_LISTS(6, true); break;
                case 7: NB_LISTS(7, true); break;
                case 8: NB_LISTS(8, true); break;
                case 9: NB_LISTS(9, true); break;
            }
        } else {
            switch ((total + 63) >> 6) {
                case 1: NB_LISTS(1, false); break;
                case 2: NB_LISTS(2, false); break;
                case 3: NB_LISTS(3, false); break;
                case 4: NB_LISTS(4, false); break;
                case 5: NB_LISTS(5, false); break;
                case 6: NB_LISTS(6, false); break;
                case 7: NB_LISTS(7, false); break;
                case 8: NB_LISTS(8, false); break;
                case 9: NB_LISTS(9, false); break;
            }
        }
#undef NB_LISTS
#undef NB_PART
    }
    // pair-interaction counter: sum_i (nPartIntorno(i) - 1), self excluded
    if (lane == 0) {
        s_pairs[wid] = mypairs;
        if (over) atomicAdd(&iscal[IS_NB_OVERFLOW], over);
    }
    __syncthreads();
    if (threadIdx.x == 0)
        atomicAdd(&pairs[(vb % NBC_PAIRS) * NBC_PSTRIDE],
                  (unsigned long long)((long long)s_pairs[0] + s_pairs[1] + s_pairs[2] + s_pairs[3]));
}

// kernel-table values at rob times the weight da, FP64 (InterpolateTable.f90:58-82)
__device__ __forceinline__ void d_kt_values(DPC& P, const double* __restrict__ kt, double rob, double da, double J[4]) {
    const double deltaX = P.ktdelta;
    const int nr0 = (int)((rob - kt[0]) / deltaX);
    if (nr0 <= 0) {
        for (int c = 0; c < 4; ++c) J[c] = kt[1 + c] * da;
    } else if (nr0 >= 40) {
        for (int c = 0; c < 4; ++c) J[c] = kt[40 * 5 + 1 + c] * da;
    } else {
        const double* r0 = &kt[nr0 * 5];
        const double* r1 = &kt[(nr0 + 1) * 5];
        const double csi = (rob - r0[0]) / deltaX;
        for (int c = 0; c < 4; ++c) J[c] = (r0[1 + c] + csi * (r1[1 + c] - r0[1 + c])) * da;
    }
}

// lane u's value for the lanes of its group of four
__device__ __forceinline__ int quad_lane(int v, int u) {
    return u == 0 ? __builtin_amdgcn_mov_dpp(v, 0x00, 0xF, 0xF, true)
         : u == 1 ? __builtin_amdgcn_mov_dpp(v, 0x55, 0xF, 0xF, true)
         : u == 2 ? __builtin_amdgcn_mov_dpp(v, 0xAA, 0xF, 0xF, true)
                  : __builtin_amdgcn_mov_dpp(v, 0xFF, 0xF, 0xF, true);
}
__device__ __forceinline__ double quad_lane(double v, int u) {
    return __hiloint2double(quad_lane(__double2hiint(v), u), quad_lane(__double2loint(v), u));
}

// ----------------------------------------------------------------------------
// SA-SPH volume integrals (FP64)
// ----------------------------------------------------------------------------
__device__ __attribute__((noinline)) void d_volume_integrals(DPC& P, const DFace& F, const double* __restrict__ kt,
                                   const double* __restrict__ bit, const double locx[3],
                                   double bi[8], double ig[9]) {
    double IntWdV = 0.0, IntdWrm1dV = 0.0, IntGWZrm1dV = 0.0;
    double G0 = 0.0, G1 = 0.0, G2 = 0.0;
    double M00 = 0.0, M01 = 0.0, M02 = 0.0, M11 = 0.0, M12 = 0.0, M22 = 0.0;
    double J0 = 0.0, J1 = 0.0, J2 = 0.0, J3 = 0.0;
    for (int q = 0; q < 8; ++q) bi[q] = 0.0;
    for (int q = 0; q < 9; ++q) ig[q] = 0.0;
    const double zpmin = 0.05 * P.h;
    double L0 = locx[0], L1 = locx[1], L2 = locx[2];
    if (L2 < 0.0) return;
    if (L2 < zpmin) L2 = zpmin;
    double robpre = 2.1;
    const PIC pic = pic_of(F);
    for (int ipk = 0; ipk < 256; ++ipk) {
        const double* b = &bit[ipk * 7];
        const double Pj0 = L0 + b[0], Pj1 = L1 + b[1], Pj2 = L2 + b[2];
        if (!(Pj2 <= 0.0)) continue;
        const double ts = L2 / (L2 - Pj2);
        const double X0 = L0 + (Pj0 - L0) * ts;
        const double X1 = L1 + (Pj1 - L1) * ts;
        if (!d_point_internal(pic, X0, X1)) continue;
        double dist = 0.0;
        {
            const double d0 = X0 - L0, d1 = X1 - L1, d2 = 0.0 - L2;
            dist = dist + d0 * d0;
            dist = dist + d1 * d1;
            dist = dist + d2 * d2;
        }
        dist = sqrt(dist);
        const double da = b[3];
        const double rob = dist / P.h;
        if (fabs(rob - robpre) > 1.0e-3) {
            double J[4];
            d_kt_values(P, kt, rob, da, J);
            J0 = J[0];
            J1 = J[1];
            J2 = J[2];
            J3 = J[3];
            robpre = rob;
        }
        const double R0 = b[4], R1 = b[5], R2 = b[6];
        const double RZ2 = R2 * R2;
        IntWdV = IntWdV + J0;
        IntdWrm1dV = IntdWrm1dV + J1;
        IntGWZrm1dV = IntGWZrm1dV + RZ2 * J1;
        G0 = G0 + R0 * J2;
        M00 = M00 + R0 * R0 * J3;
        M01 = M01 + R0 * R1 * J3;
        M02 = M02 + R0 * R2 * J3;
        G1 = G1 + R1 * J2;
        M11 = M11 + R1 * R1 * J3;
        M12 = M12 + R1 * R2 * J3;
        G2 = G2 + R2 * J2;
        M22 = M22 + R2 * R2 * J3;
    }
    if (L2 == zpmin) IntWdV = d_point_internal(F, L0, L1) ? 0.5 : 0.0;
    bi[1] = IntWdV;
    bi[2] = IntdWrm1dV;
    bi[3] = G0;
    bi[4] = G1;
    bi[5] = G2;
    bi[6] = IntGWZrm1dV;
    // IntGiWrRdV column-major
    ig[0] = M00; ig[1] = M01; ig[2] = M02;
    ig[3] = M01; ig[4] = M11; ig[5] = M12;
    ig[6] = M02; ig[7] = M12; ig[8] = M22;
}

// ----------------------------------------------------------------------------
// boundary table: ComputeBoundaryDataTab_3D.f90:62-106 in two kernels.
// k_boundary_find: FindCloseBoundaryFaces3D.f90:78-188 per particle, appends
// every (particle, close face) pair to a compact work list; k_boundary_int:
// ComputeBoundaryVolumeIntegrals_P0.f90:76-155 over that list.
// ----------------------------------------------------------------------------
template <bool SG>
__global__ __launch_bounds__(256) void k_boundary_find(Seg S, const DFace* __restrict__ faces,
                                                       const int* __restrict__ ncount,
                                                       const int* __restrict__ nstart,
                                                       const int* __restrict__ nvec,
                                                       const double4* __restrict__ xm,
                                                       int* __restrict__ bn, BTab* __restrict__ bt,
                                                       int* __restrict__ work, int* nwork, int* iscal) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int sg = SG ? __builtin_amdgcn_readfirstlane(S.pblk[(blockIdx.x * blockDim.x) >> 8]) : 0;
    DPC& P = S.P[sg];
    iscal += sg * IS_COUNT;
    if (i - P.base >= iscal[IS_N]) return;
    const double4 x = xm[i];
    const double xc[3] = {x.x, x.y, x.z};
    const int nc = d_particle_cell(P, x.x, x.y, x.z);
    // the faces listed in the 27 cells around the particle's cell, each once
    // and in the order the reference's cell walk meets them (a face accepted
    // once is skipped when met again; one rejected is rejected again)
    const int nf = nc > 0 ? ncount[P.koff + nc - 1] : 0;
    if (nf == 0) {  // no frontier face listed within reach
        bn[i] = 0;
        return;
    }
    int ncbf = 0;
    int clob[SPH_MB];
    double lz[SPH_MB];
    const int ini = nstart[P.koff + nc - 1];
    for (int fl = ini; fl < ini + nf; ++fl) {
        const int f = nvec[fl];
        const DFace& F = faces[f];
        const double pinmin = (F.btype == 3) ? -P.doubleh : 0.0;
        const double* ref = &F.GX[3 * (F.nodes - 1)];
        double PX[3];
        for (int sdi = 0; sdi < 3; ++sdi) {
            double s = 0.0;
            for (int sdj = 0; sdj < 3; ++sdj) s = s + F.T[3 * sdi + sdj] * (xc[sdj] - ref[sdj]);
            PX[sdi] = s;
        }
        const double pin = PX[2];
        if (pin >= pinmin && pin < P.doubleh) {
            const bool need_in = (F.btype == 3 || F.btype == 4 || F.btype == 5);
            if (!need_in || d_point_internal(F, PX[0], PX[1])) {
                if (ncbf >= SPH_MB) {
                    atomicAdd(&iscal[IS_BT_OVERFLOW], 1);
                    continue;
                }
                clob[ncbf] = f;
                lz[ncbf] = pin;
                ++ncbf;
            }
        }
    }
    bn[i] = ncbf;
    if (ncbf == 0) return;
    const int w0 = atomicAdd(nwork, ncbf);
    for (int q = 0; q < ncbf; ++q) {
        const DFace& F = faces[clob[q]];
        const double* ref = &F.GX[3 * (F.nodes - 1)];
        BTab& rec = bt[(size_t)q * P.cap + i];
        for (int sdi = 0; sdi < 2; ++sdi) {
            double s = 0.0;
            for (int sdj = 0; sdj < 3; ++sdj) s = s + F.T[3 * sdi + sdj] * (xc[sdj] - ref[sdj]);
            rec.loc[sdi] = s;
        }
        rec.loc[2] = lz[q];
        rec.face = clob[q];
        work[w0 + q] = i | (q << NB_SHIFT);
    }
}

// ----------------------------------------------------------------------------
// 2D form (x-z plane): boundary table over the boundary sides.
// FindCloseBoundarySides2D.f90:68-170, SelectCloseBoundarySides2D.f90:66-120,
// ComputeBoundaryDataTab_2D.f90:71-162 with FindBoundaryIntersection2D.f90:
// 59-86, ComputeSurfaceIntegral_WdS2D.f90:57-85, BoundaryVolumeIntegrals2D
// .f90:60-97, ComputeVolumeIntegral_WdV2D.f90:69-132 and
// InterpolateBoundaryIntegrals2D.f90:61-70.  One lane per particle over the
// sides (a tank has a handful); every expression in the reference's order.
// The integrals use the device's sin, cos, tan and atan2 (the host reference
// calls the C library's).
// ----------------------------------------------------------------------------
constexpr double PIGRECO_D = 3.14159265358979;
constexpr double KERNELCONST2D_D = 0.454728408833987;
constexpr double DELTAX_BIT_D = 0.1;

// w.f90:48-57
__device__ __forceinline__ double d_w2(double r, double h, double coef) {
    const double sq = r / h;
    double q;
    if (sq <= 1.0) {
        q = 0.666666667 + sq * sq * (sq * 0.5 - 1.0);
    } else if (sq >= 2.0) {
        q = 0.0;
    } else {
        const double dms = 2.0 - sq;
        q = dms * dms * dms / 6.0;
    }
    return q * coef;
}
// WIntegr.f90:60-82
__device__ __forceinline__ double d_wintegr(double ri, double hh) {
    const double ro = ri / hh;
    if (0.0 <= ro && ro < 1.0) {
        const double ro2 = ro * ro, ro3 = ro2 * ro;
        const double w1 = (0.5 + -0.375 * ro2 + 0.15 * ro3) * ro2;
        return KERNELCONST2D_D * (0.35 - w1);
    } else if (1.0 <= ro && ro < 2.0) {
        const double q1 = 2.0 - ro, q2 = q1 * q1, q4 = q2 * q2;
        return -KERNELCONST2D_D * ((-0.125 + 0.05 * q1) * q4);
    }
    return 0.0;
}
// J2Wro2.f90:55-70
__device__ __forceinline__ double d_j2wro2(double ro) {
    const double a1 = 0.00833333333333333, a2 = 0.26666666666666667;
    const double ro2 = ro * ro, ro3 = ro2 * ro;
    if (0.0 <= ro && ro < 1.0) return KERNELCONST2D_D * (0.25 - (a1 * (40.0 - 36.0 * ro2 + 15.0 * ro3) * ro3));
    if (1.0 <= ro && ro < 2.0)
        return KERNELCONST2D_D * (a2 - (a1 * (80.0 - 90.0 * ro + 36.0 * ro2 - 5.0 * ro3) * ro3));
    return 0.0;
}
// BoundIntegralTab2D row r (0-based), column c; 22 x 6 row-major
__device__ __forceinline__ void d_interp2d(const double* __restrict__ tab, int ncols, const int* cols,
                                           double xx, double* func) {
    if (xx < tab[0]) xx = tab[0];
    // rows 1..21 hold ii (0 <= delta < 2 for a selected side); the clamp only
    // keeps a non-finite position inside the table
    const int ii = min(max((int)((xx - tab[0]) / DELTAX_BIT_D) + 1, 1), 21);
    const double xi = tab[(ii - 1) * 6];
    for (int nc = 0; nc < ncols; ++nc) {
        const int jj = cols[nc];
        const double fi = tab[(ii - 1) * 6 + jj], fip1 = tab[ii * 6 + jj];
        func[nc] = fi + (fip1 - fi) * (xx - xi) / DELTAX_BIT_D;
    }
}

constexpr int BT2_WG = 512;
struct Corner2D {  // a particle with two close sides
    int i, side[2];
    double x[2], y[2];
};

__global__ __launch_bounds__(BT2_WG) void k_boundary_2d(DPC* Pp, const DFace* __restrict__ sides,
                                                     const double* __restrict__ tab,
                                                     const double4* __restrict__ xm,
                                                     const int* __restrict__ cell,
                                                     int* __restrict__ bn, BTab* __restrict__ bt,
                                                     int* iscal) {
    DPC& P = *Pp;
    __shared__ Corner2D corners[BT2_WG];
    __shared__ int ncorner;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (threadIdx.x == 0) ncorner = 0;
    __syncthreads();
    const bool live = i < P.cap && i < iscal[IS_N];
    int nint = 0;
    double4 X = make_double4(0.0, 0.0, 0.0, 0.0);
    if (live) X = xm[i];
    const double px = X.x, pz = X.z;
    const double dh = P.doubleh;
    int ncbs = 0;
    int clo[4];
    double loc[8];
    bool bad = !live;
    for (int isi = 0; isi < P.nf && !bad; ++isi) {
        const DFace& S = sides[isi];
        if (S.btype == 6) continue;  // peri
        const double P1P0 = px - S.v1[0], P1P1 = pz - S.v1[1];
        const double s0 = S.T[0], s1 = S.T[2], n0 = S.T[6], n1 = S.T[8];
        const double sidel = S.len;
        const double xp = P1P0 * s0 + P1P1 * s1;
        const double yp = P1P0 * n0 + P1P1 * n1;
        const double xpmin = -dh, xpmax = sidel + dh, ypmin = -dh, ypmax = dh;
        if ((xpmin < xp && xp < xpmax) && (ypmin < yp && yp < ypmax)) {
            double ypmx = 0.0, ypmn = 0.0;
            if (xp < 0.0) {
                ypmx = sqrt(P.square_doubleh - xp * xp);
                ypmn = -ypmx;
            } else if (xp <= sidel) {
                ypmx = ypmax;
                ypmn = ypmin;
            } else if (xp < xpmax) {
                const double Lmxpq = (sidel - xp) * (sidel - xp);
                ypmx = sqrt(P.square_doubleh - Lmxpq);
                ypmn = -ypmx;
            }
            if (ypmn < yp && yp < ypmx) {
                if (ncbs >= 4) {
                    bad = true;
                    break;
                }
                clo[ncbs] = isi;
                loc[2 * ncbs] = xp;
                loc[2 * ncbs + 1] = yp;
                ncbs = ncbs + 1;
            }
        }
    }
    for (int q = 0; q < ncbs && !bad; ++q) {
        const int b = sides[clo[q]].btype;
        if (b != 0 && b != 1 && b != 2) {
            atomicAdd(&iscal[IS_UNSUPPORTED], 1);
            bad = true;
        }
    }
    if (bad && ncbs >= 4) atomicAdd(&iscal[IS_BT_OVERFLOW], 1);
    if (bad) ncbs = 0;
    if (ncbs == 2) {
        const int a = clo[0], b = clo[1];
        if (sides[a].prev == b + 1)
            loc[2] = sides[b].len - loc[2];
        else if (sides[b].prev == a + 1)
            loc[0] = sides[a].len - loc[0];
    }
    // SelectCloseBoundarySides2D.f90:66-120: fixe/tapi sides with y > 0; open
    // sides with y > 0 and 0 < x < side length
    int iside[4];
    double iloc[8];
    for (int q = 0; q < ncbs; ++q) {
        bool keep = loc[2 * q + 1] > 0.0;
        if (sides[clo[q]].btype == 2) keep = keep && loc[2 * q] > 0.0 && loc[2 * q] < sides[clo[q]].len;
        if (keep) {
            iside[nint] = clo[q];
            iloc[2 * nint] = loc[2 * q];
            iloc[2 * nint + 1] = loc[2 * q + 1];
            nint = nint + 1;
        }
    }
    if (nint > 2) {
        atomicAdd(&iscal[IS_BT_OVERFLOW], 1);
        nint = 0;
    }
    const double h = P.h;
    const double yplimite = 0.05 * h;
    const double dalfarif = PIGRECO_D / 10;
    for (int icbs = 0; icbs < nint; ++icbs) {
        BTab& B = bt[(size_t)icbs * P.cap + i];
        const double ypi = iloc[2 * icbs + 1];
        B.face = iside[icbs];
        B.loc[0] = iloc[2 * icbs];
        B.loc[1] = ypi;
        B.loc[2] = 0.0;
        if (nint == 2) continue;
        double F[5];
        const int cols[5] = {1, 2, 3, 4, 5};
        d_interp2d(tab, 5, cols, ypi / h, F);
        B.bi[0] = F[0] / h;
        B.bi[1] = F[1];
        B.bi[2] = F[1];
        B.bi[3] = 0.0;
        B.bi[4] = 0.0;
        B.bi[5] = F[2] / P.squareh;
        B.bi[6] = F[3] / P.squareh;
        B.bi[7] = F[4] / P.squareh;
    }
    if (i < P.cap) bn[i] = nint;
    // The particles near a corner: three quadratures of about ten points a side.
    // Bound by their latency (sin, cos, tan, atan2; one point after the other
    // and one side after the other took 32 us at 5,000 particles), so a point is
    // a lane's, a side 16 lanes', and the third quadrature the other half of the
    // workgroup's; the sums are formed in order: 13 us.
    if (nint == 2) {
        Corner2D& C = corners[atomicAdd(&ncorner, 1)];
        C.i = i;
        for (int q = 0; q < 2; ++q) {
            C.side[q] = iside[q];
            C.x[q] = iloc[2 * q];
            C.y[q] = iloc[2 * q + 1];
        }
    }
    __syncthreads();
    constexpr int HALF = BT2_WG / 2;
    const int g = threadIdx.x % 16;
    const bool third = threadIdx.x >= HALF;
    for (int n = (threadIdx.x % HALF) / 16; n < 2 * ncorner; n += HALF / 16) {
        const Corner2D& C = corners[n >> 1];
        const int icbs = n & 1;
        // point k (from 1) of a sum that steps by d from x0: the running sum itself
        auto step = [](double x0, double d, int k) {
            double x = x0;
            for (int t = 0; t < k; ++t) x = x + d;
            return x;
        };
        BTab& B = bt[(size_t)icbs * P.cap + C.i];
        const double xpi = C.x[icbs], ypi = C.y[icbs];
        const double deltai = ypi / h;
        double F[5];
        // FindBoundaryIntersection2D (ypi > 0 here)
        const double halfchord = sqrt(P.square_doubleh - ypi * ypi);
        const double XA = xpi - halfchord, XB = xpi + halfchord;
        double xpmin = 0.0;
        if (XA > xpmin) xpmin = XA;
        double xpmax = sides[C.side[icbs]].len;
        if (XB < xpmax) xpmax = XB;
        double interlen = xpmax - xpmin;
        if (interlen <= 0.01 * h) interlen = 0.0;
        // ComputeSurfaceIntegral_WdS2D
        double IntWdS[1] = {0.0};
        if (!third && interlen > 0.0) {
            const double dsrif = h / 2.0;
            const double ypiq = ypi * ypi;
            int ndiv = (int)(interlen / dsrif + 0.5);
            if (ndiv < 2) ndiv = 2;
            const double deltas = interlen / ndiv;
            for (int k0 = 1; k0 <= ndiv; k0 += 16) {
                double t[1] = {0.0};
                if (k0 + g <= ndiv) {
                    const double dxpip = step(xpmin - 0.5 * deltas, deltas, k0 + g) - xpi;
                    const double ris = sqrt(dxpip * dxpip + ypiq);
                    t[0] = d_w2(ris, h, P.coefke) * deltas;
                }
                add_lanes<16>(IntWdS, t);
            }
        }
        // BoundaryVolumeIntegrals2D
        double V[3] = {0.0, 0.0, 0.0};  // IntWdV, Dp
        if (!third && interlen > 0.0) {
            double yb = ypi;
            if (yb < yplimite) yb = yplimite;
            const double alfaA = atan2(xpmin - xpi, yb), alfaB = atan2(xpmax - xpi, yb);
            const double intalfa = alfaB - alfaA;
            int ndiv = (int)(intalfa / dalfarif + 0.5);
            if (ndiv < 1) ndiv = 1;
            const double dalfa = intalfa / ndiv;
            for (int k0 = 1; k0 <= ndiv; k0 += 16) {
                double t[3] = {0.0, 0.0, 0.0};
                if (k0 + g <= ndiv) {
                    const double alfa_k = step(alfaA - 0.5 * dalfa, dalfa, k0 + g);
                    const double sa = sin(alfa_k), ca = cos(alfa_k);
                    const double rb = yb / ca;
                    const double mult = h * d_j2wro2(rb / h) * dalfa;
                    t[0] = d_wintegr(rb, h) * dalfa;
                    t[1] = sa * mult;
                    t[2] = -(ca * mult);
                }
                add_lanes<16>(V, t);
            }
            if (yb == yplimite) V[0] = 0.5;
        }
        // ComputeVolumeIntegral_WdV2D (Ncbslocal = 2)
        double IntWdV1[1] = {0.0};
        if (third && interlen > 0.0) {
            if (ypi >= yplimite) {
                const double alfaA = atan2(xpmin - xpi, ypi), alfaB = atan2(xpmax - xpi, ypi);
                const double intalfa = alfaB - alfaA;
                int ndiv = (int)(intalfa / dalfarif + 0.5);
                if (ndiv < 2) ndiv = 2;
                const double dalfa = intalfa / ndiv;
                for (int k0 = 1; k0 <= ndiv; k0 += 16) {
                    double t[1] = {0.0};
                    if (k0 + g <= ndiv) {
                        const double ta = tan(step(alfaA - 0.5 * dalfa, dalfa, k0 + g));
                        const double ris = ypi * sqrt(1.0 + ta * ta);
                        t[0] = d_wintegr(ris, h) * dalfa;
                    }
                    add_lanes<16>(IntWdV1, t);
                }
            } else {
                const double ypj = C.y[1 - icbs];
                if (ypj <= yplimite) {
                    double angle = 0.0;
                    if (sides[C.side[0]].prev == C.side[1] + 1)
                        angle = sides[C.side[0]].angle;
                    else if (sides[C.side[1]].prev == C.side[0] + 1)
                        angle = sides[C.side[1]].angle;
                    else if (g == 0)
                        atomicAdd(&iscal[IS_UNSUPPORTED], 1);  // sides not consecutive
                    IntWdV1[0] = 0.5 * (angle + PIGRECO_D) / (2.0 * PIGRECO_D);
                } else {
                    IntWdV1[0] = (xpmin >= xpi && xpi <= xpmax) ? 0.5 : 0.0;
                }
            }
        }
        if (g == 0 && third) {
            const int cols[3] = {3, 4, 5};
            d_interp2d(tab, 3, cols, deltai, F);
            B.bi[2] = IntWdV1[0];
            B.bi[5] = F[0] / P.squareh;
            B.bi[6] = F[1] / P.squareh;
            B.bi[7] = F[2] / P.squareh;
        } else if (g == 0) {
            B.bi[0] = IntWdS[0];
            B.bi[1] = V[0];
            B.bi[3] = V[1];
            B.bi[4] = V[2];
        }
    }
}

// ----------------------------------------------------------------------------
// FP32-mixed form of the same quadrature, eight lanes per (particle, face)
// pair, lane r taking ring r of BoundIntegralTab.  The rays of a ring meet
// the face plane on one circle of radius ts |b_xy| around (L0, L1), all at
// the same distance rob h = L2 |b| / (-b_z).  IsPointInternal's area
// coordinates are affine over the plane, so over that circle each stays
// within its centre value +- radius |grad|: a circle that clears every bound
// (or lies beyond one) by BT_MARGIN has every direction inside (outside) the
// face, as the FP64 per-direction test finds it; other rings run that test
// per direction (FP64, with -1/b_z precomputed).  The reference's reuse of
// the kernel-table values (refresh when rob moves by more than 1e-3) changes
// state only at the first kept direction of a ring, so the lanes replay it
// over the rings' (count, rob) in ring order; interpolation and sums are
// FP32 and the eight ring sums are reduced across the lanes.
// ----------------------------------------------------------------------------
constexpr double BT_MARGIN = 1.0e-10;

// 1: the circle (centre c0, c1, radius rad) lies inside the face, -1: outside,
// 0: undecided
__device__ __forceinline__ int ring_side(const DFace& F, const PIC& c, double c0, double c1, double rad) {
    if (c.fkod != 1 && c.fkod != 2) return -1;
    const double u0 = (c.a0 + c.b0 * c0 + c.c0 * c1) * c.pu;
    const double u1 = (c.a1 + c.b1 * c0 + c.c1 * c1) * c.pu;
    const double m0 = rad * F.pg[0] + BT_MARGIN, m1 = rad * F.pg[1] + BT_MARGIN;
    bool in = u0 - m0 >= 0.0 && u0 + m0 <= 1.0 && u1 - m1 >= 0.0 && u1 + m1 <= 1.0;
    bool out = u0 + m0 < 0.0 || u0 - m0 > 1.0 || u1 + m1 < 0.0 || u1 - m1 > 1.0;
    if (c.fkod == 1) {
        const double u2 = 1.0 - (u0 + u1), m2 = rad * F.pg[2] + BT_MARGIN;
        in = in && u2 - m2 >= 0.0 && u2 + m2 <= 1.0;
        out = out || u2 + m2 < 0.0 || u2 - m2 > 1.0;
    }
    return in ? 1 : (out ? -1 : 0);
}

// The volume integrals in FP64, bit for bit as d_volume_integrals sums them
// over the 256 directions, by four lanes of a pair.  One lane a pair walked the
// directions one after the other: 101 us at 72,000 particles, 134 at 576,000.
// A ring's directions share b_z and the weight (RingC), so the plane test, ts
// and the table values belong to the ring: each lane takes two rings, decides
// them whole by ring_side where it can and tests direction by direction where
// it cannot.  Then every lane adds three of the twelve sums over the kept
// directions in order, the factors from an LDS table: 32 and 60 us.  The
// table values are refreshed where rob moves by more than 1e-3: within a ring
// it moves by rounding only, so a ring is refreshed by its first kept direction
// or not at all; a pair in which a ring's move is within 1e-9 of 1e-3 goes through
// d_volume_integrals, and so does every pair of a table whose rings are not of
// this form, one lane a pair.
// Segmented contexts: BT_SPLIT workgroups take the pairs of a 256-slot block,
// which share a segment and so these tables.  (From the work list, which holds
// the segments' pairs mixed, with the tables in global memory, 2 solves of 1,440
// particles took 186 us, now 60; 256 of them 1760, 402; 16 of 11,000 482, 146.)
constexpr int BT_SPLIT = 4;
template <bool SG>
__global__ __launch_bounds__(256) void k_boundary_int(Seg S, const DFace* __restrict__ faces,
                                                      const double* __restrict__ kt_g,
                                                      const double* __restrict__ bit_g,
                                                      const BtF32* __restrict__ tab, BTab* __restrict__ bt,
                                                      const int* __restrict__ work, const int* nwork,
                                                      const int* __restrict__ bn, const int* iscal) {
    constexpr int ND = BT_RINGS * BT_RDIRS, G = 4;
    __shared__ double kt_s[41 * 5];
    __shared__ double2 b_s[ND];
    __shared__ double f_s[ND * 12];  // lane l's factors of direction k: [12 k + 3 l, + 3)
    __shared__ uint16_t pair_s[SG ? 256 * SPH_MB : 1];  // slot of the block, table slot << 8
    __shared__ int wsum[4];
    const int blk = SG ? blockIdx.x / BT_SPLIT : blockIdx.x, first = SG ? blockIdx.x % BT_SPLIT : blockIdx.x;
    const int stride = SG ? BT_SPLIT : gridDim.x;
    const int sg = SG ? __builtin_amdgcn_readfirstlane(S.pblk[blk]) : 0;
    DPC& P = S.P[sg];
    int nw;
    if (SG) {
        const int i = blk * 256 + threadIdx.x, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
        const int n = i - P.base < iscal[sg * IS_COUNT + IS_N] ? bn[i] : 0;
        const int incl = wave_incl_scan(n);
        if (lane == 63) wsum[wid] = incl;
        __syncthreads();
        int at = incl - n;
        for (int v = 0; v < wid; ++v) at += wsum[v];
        nw = wsum[0] + wsum[1] + wsum[2] + wsum[3];
        for (int q = 0; q < n; ++q) pair_s[at + q] = (uint16_t)(threadIdx.x | (q << 8));
    } else {
        nw = *nwork;
    }
    if (first * (256 / G) >= nw) return;  // no pair for this workgroup
    const double* ktg = kt_g + (size_t)sg * (41 * 5);
    const double* bitg = bit_g + (size_t)sg * (ND * 7);
    const BtF32& T = tab[sg];
    auto factors = [](const double* R, int l, double f[3]) {
        f[0] = l == 0 ? 1.0 : l == 1 ? R[0] : l == 2 ? R[0] * R[0] : R[1] * R[1];
        f[1] = l == 0 ? 1.0 : l == 1 ? R[1] : l == 2 ? R[0] * R[1] : R[1] * R[2];
        f[2] = l == 0 ? R[2] * R[2] : l == 1 ? R[2] : l == 2 ? R[0] * R[2] : R[2] * R[2];
    };
    for (int t = threadIdx.x; t < 41 * 5; t += 256) kt_s[t] = ktg[t];
    for (int t = threadIdx.x; t < ND; t += 256) {
        const double* b = &bitg[t * 7];
        b_s[t] = make_double2(b[0], b[1]);
        for (int l = 0; l < G; ++l) factors(b + 4, l, &f_s[12 * t + 3 * l]);
    }
    __syncthreads();
    auto record = [&](int w) -> BTab& {
        const int e = SG ? pair_s[w] : work[w];
        const int i = SG ? blk * 256 + (e & 255) : e & (int)NB_MASK;
        const int q = SG ? e >> 8 : (int)((uint32_t)e >> NB_SHIFT);
        return bt[(size_t)q * P.cap + i];
    };
    auto serially = [&](BTab& rec) {
        const double loc[3] = {rec.loc[0], rec.loc[1], rec.loc[2]};
        double bi[8], ig[9];
        d_volume_integrals(P, faces[rec.face], ktg, bitg, loc, bi, ig);
        for (int t = 0; t < 8; ++t) rec.bi[t] = bi[t];
        for (int t = 0; t < 9; ++t) rec.ig[t] = ig[t];
    };
    if (!T.all_ok) {  // no rings: one lane a pair
        for (int w = first * 256 + threadIdx.x; w < nw; w += stride * 256) serially(record(w));
        return;
    }
    const int l = threadIdx.x % G;
    for (int w = (first * 256 + threadIdx.x) / G; w < nw; w += stride * (256 / G)) {
        const double* kt = kt_s;
        auto dir = [&](int k) { return b_s[k]; };
        BTab& rec = record(w);
        const DFace& F = faces[rec.face];
        const double loc[3] = {rec.loc[0], rec.loc[1], rec.loc[2]};
        const double zpmin = 0.05 * P.h;
        const double L0 = loc[0], L1 = loc[1], L2 = loc[2] < zpmin ? zpmin : loc[2];
        const PIC pic = pic_of(F);
        uint32_t mask[2] = {0u, 0u};  // the kept directions of the rings l and l + 4
        double rob[2] = {0.0, 0.0}, J[2][4];
        bool serial = false;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            J[u][0] = J[u][1] = J[u][2] = J[u][3] = 0.0;
            const int r = l + 4 * u;
            const double Pj2 = L2 + T.rc[r].bz;
            if (loc[2] < 0.0 || !(Pj2 <= 0.0)) continue;
            const double ts = L2 / (L2 - Pj2);
            auto point = [&](int k, double& X0, double& X1) {
                const double2 b = dir(r * BT_RDIRS + k);
                const double Pj0 = L0 + b.x, Pj1 = L1 + b.y;
                X0 = L0 + (Pj0 - L0) * ts;
                X1 = L1 + (Pj1 - L1) * ts;
            };
            double X0, X1;
            const int side = ring_side(F, pic, L0, L1, ts * T.rc[r].rho);
            uint32_t m = side > 0 ? ~0u : 0u;
            if (side == 0)
                for (int k = 0; k < BT_RDIRS; ++k) {
                    point(k, X0, X1);
                    if (d_point_internal(pic, X0, X1)) m |= 1u << k;
                }
            mask[u] = m;
            if (m == 0u) continue;
            point(__ffs(m) - 1, X0, X1);
            double dist = 0.0;
            const double d0 = X0 - L0, d1 = X1 - L1, d2 = 0.0 - L2;
            dist = dist + d0 * d0;
            dist = dist + d1 * d1;
            dist = dist + d2 * d2;
            dist = sqrt(dist);
            rob[u] = dist / P.h;
            d_kt_values(P, kt, rob[u], bitg[r * BT_RDIRS * 7 + 3], J[u]);
        }
        double s[3] = {0.0, 0.0, 0.0}, ja = 0.0, jb = 0.0, robpre = 2.1;
#pragma unroll
        for (int r = 0; r < BT_RINGS; ++r) {
            const int u = r / G;
            const uint32_t m = (uint32_t)quad_lane((int)mask[u], r % G);
            const double rr = quad_lane(rob[u], r % G);
            double Jr[4];
            for (int c = 0; c < 4; ++c) Jr[c] = quad_lane(J[u][c], r % G);
            const double move = fabs(rr - robpre);
            if (m != 0u && fabs(move - 1.0e-3) < 1.0e-9) serial = true;
            if (m != 0u && move > 1.0e-3) {
                ja = l == 0 ? Jr[0] : l == 1 ? Jr[2] : Jr[3];
                jb = l == 0 ? Jr[1] : ja;
                robpre = rr;
            }
            if (!__any(m != 0u)) continue;
            const bool part = __any(m != 0u && m != ~0u);
            const double ma = m ? ja : 0.0, mb = m ? jb : 0.0;  // a direction left out adds a zero
#pragma unroll 4
            for (int k = 0; k < BT_RDIRS; ++k) {
                const int d = r * BT_RDIRS + k;
                const double f[3] = {f_s[12 * d + 3 * l], f_s[12 * d + 3 * l + 1], f_s[12 * d + 3 * l + 2]};
                const bool on = !part || ((m >> k) & 1u);
                const double ka = on ? ma : 0.0, kb = on ? mb : 0.0;
                s[0] = s[0] + f[0] * ka;
                s[1] = s[1] + f[1] * kb;
                s[2] = s[2] + f[2] * kb;
            }
        }
        if (serial) {
            if (l == 0) serially(rec);
        } else if (l == 0) {
            rec.bi[0] = 0.0;
            rec.bi[1] = loc[2] >= 0.0 && L2 == zpmin ? (d_point_internal(F, L0, L1) ? 0.5 : 0.0) : s[0];
            rec.bi[2] = s[1];
            rec.bi[6] = s[2];
            rec.bi[7] = 0.0;
        } else if (l == 1) {
            for (int t = 0; t < 3; ++t) rec.bi[3 + t] = s[t];
        } else if (l == 2) {
            for (int t = 0; t < 3; ++t) rec.ig[t] = s[t];
            rec.ig[3] = s[1];
            rec.ig[6] = s[2];
        } else {
            rec.ig[4] = s[0];
            rec.ig[5] = rec.ig[7] = s[1];
            rec.ig[8] = s[2];
        }
    }
}

// kernel-table values at rob times the weight da (InterpolateTable.f90:58-82)
__device__ __forceinline__ void kt_values_f32(const BtF32& T, float rob, float da, float J[4]) {
#pragma clang fp contract(fast)
    const float* kt = T.kt;
    const int nr0 = (int)((rob - kt[0]) * T.kt_inv_delta);
    if (nr0 <= 0) {
        for (int c = 0; c < 4; ++c) J[c] = kt[1 + c] * da;
    } else if (nr0 >= 40) {
        for (int c = 0; c < 4; ++c) J[c] = kt[40 * 5 + 1 + c] * da;
    } else {
        const float* r0 = &kt[nr0 * 5];
        const float csi = (rob - r0[0]) * T.kt_inv_delta;
        for (int c = 0; c < 4; ++c) J[c] = (r0[1 + c] + csi * (r0[6 + c] - r0[1 + c])) * da;
    }
}

// accumulators: IntWdV, IntdWrm1dV, IntGWZrm1dV, G0..2, M00 M01 M02 M11 M12 M22;
// n directions with common R_z and unit-vector sums s = (R0, R1, R0^2, R0R1, R1^2)
__device__ __forceinline__ void bt_add(float a[12], const float J[4], float n, float R2, const float s[5]) {
#pragma clang fp contract(fast)
    a[0] += n * J[0];
    a[1] += n * J[1];
    a[2] += R2 * R2 * n * J[1];
    a[3] += J[2] * s[0];
    a[4] += J[2] * s[1];
    a[5] += J[2] * R2 * n;
    a[6] += J[3] * s[2];
    a[7] += J[3] * s[3];
    a[8] += J[3] * R2 * s[0];
    a[9] += J[3] * s[4];
    a[10] += J[3] * R2 * s[1];
    a[11] += J[3] * R2 * R2 * n;
}

// a table without the ring structure: one lane, direction by direction
__device__ void bt_pair_f32_dirs(const BtF32& T, const DFace& F, double L0, double L1, double L2,
                                 float a[12]) {
    const PIC pic = pic_of(F);
    const float L2f = (float)L2;
    float robpre = 2.1f, J[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < BT_RINGS * BT_RDIRS; ++k) {
        const BitF64 g = T.bd[k];
        if (!(L2 + g.b2 <= 0.0)) continue;
        const double ts = L2 * g.nr;
        if (!d_point_internal(pic, L0 + g.b0 * ts, L1 + g.b1 * ts)) continue;
        const float* f = T.bf[k];
        const float rob = L2f * f[0];
        if (fabsf(rob - robpre) > 1.0e-3f) {
            kt_values_f32(T, rob, f[1], J);
            robpre = rob;
        }
        const float s[5] = {f[2], f[3], f[2] * f[2], f[2] * f[3], f[3] * f[3]};
        bt_add(a, J, 1.f, T.br2[k], s);
    }
}

// Segmented contexts: the lanes of a pair read their segment's table (one
// per segment, consecutive) from global memory.
template <bool SG>
__global__ __launch_bounds__(256) void k_boundary_int_f32(Seg S, const DFace* __restrict__ faces,
                                                          const BtF32* __restrict__ tab,
                                                          BTab* __restrict__ bt,
                                                          const int* __restrict__ work,
                                                          const int* nwork) {
    __shared__ BtF32 T_s;
    const int nw = *nwork;
    const int per_block = blockDim.x / BT_RINGS;
    if (blockIdx.x * per_block >= nw) return;  // no pair for this workgroup
    if (!SG) {
        const int4* src = reinterpret_cast<const int4*>(tab);
        int4* dst = reinterpret_cast<int4*>(&T_s);
        for (int t = threadIdx.x; t < (int)(sizeof(BtF32) / 16); t += blockDim.x) dst[t] = src[t];
        __syncthreads();
    }
    const int gt = blockIdx.x * blockDim.x + threadIdx.x;
    const int r = gt & (BT_RINGS - 1);
    const int stride = (gridDim.x * blockDim.x) / BT_RINGS;
    // the eight lanes of a pair stay together: same w, same trip count
    for (int w = gt / BT_RINGS; w < nw; w += stride) {
        const int e = work[w];
        const int i = e & (int)NB_MASK, q = (int)((uint32_t)e >> NB_SHIFT);
        const int sg = SG ? S.pblk[i >> 8] : 0;
        DPC& P = S.P[sg];
        const BtF32& T = SG ? tab[sg] : T_s;
        BTab& rec = bt[(size_t)q * P.cap + i];
        const double L0 = rec.loc[0], L1 = rec.loc[1];
        double L2 = rec.loc[2];
        const DFace& F = faces[rec.face];
        const double zpmin = 0.05 * P.h;
        float a[12];
        for (int t = 0; t < 12; ++t) a[t] = 0.f;
        const bool neg = L2 < 0.0;
        if (L2 < zpmin) L2 = zpmin;
        if (!neg && !T.all_ok) {
            if (r == 0) bt_pair_f32_dirs(T, F, L0, L1, L2, a);
        } else if (!neg) {
            const RingC R = T.rc[r];
            const PIC pic = pic_of(F);
            float n = 0.f, s[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
            if (L2 + R.bz <= 0.0) {  // the plane test, common to the ring
                const double ts = L2 * R.nr;
                const int side = ring_side(F, pic, L0, L1, ts * R.rho);
                if (side > 0) {
                    n = (float)BT_RDIRS;
                    s[0] = R.s0; s[1] = R.s1; s[2] = R.s00; s[3] = R.s01; s[4] = R.s11;
                } else if (side == 0) {
                    for (int k = r * BT_RDIRS; k < (r + 1) * BT_RDIRS; ++k) {
                        const BitF64 g = T.bd[k];
                        if (!d_point_internal(pic, L0 + g.b0 * ts, L1 + g.b1 * ts)) continue;
                        const float* f = T.bf[k];
                        n += 1.f;
                        s[0] += f[2];
                        s[1] += f[3];
                        s[2] += f[2] * f[2];
                        s[3] += f[2] * f[3];
                        s[4] += f[3] * f[3];
                    }
                }
            }
            const float L2f = (float)L2;
            const float rob = L2f * R.ck;
            // the reuse rule over the rings in order: the ring whose values ring r uses
            float robpre = 2.1f;
            int src = -1;
            for (int k = 0; k < BT_RINGS; ++k) {
                const float nk = __shfl(n, k, BT_RINGS), rk = __shfl(rob, k, BT_RINGS);
                if (nk > 0.f && fabsf(rk - robpre) > 1.0e-3f) {
                    robpre = rk;
                    if (k <= r) src = k;
                }
            }
            if (n > 0.f && src >= 0) {
                float J[4];
                kt_values_f32(T, L2f * T.rc[src].ck, T.rc[src].da, J);
                bt_add(a, J, n, R.R2, s);
            }
        }
        for (int o = BT_RINGS / 2; o > 0; o >>= 1)
            for (int t = 0; t < 12; ++t) a[t] += __shfl_xor(a[t], o, BT_RINGS);
        // bi(1:8), then IntGiWrRdV column-major: 17 doubles, spread over the lanes
        double v[17];
        v[0] = 0.0;
        v[1] = neg ? 0.0 : (L2 == zpmin ? (d_point_internal(F, L0, L1) ? 0.5 : 0.0) : (double)a[0]);
        v[2] = a[1]; v[3] = a[3]; v[4] = a[4]; v[5] = a[5]; v[6] = a[2]; v[7] = 0.0;
        v[8] = a[6]; v[9] = a[7]; v[10] = a[8];
        v[11] = a[7]; v[12] = a[9]; v[13] = a[10];
        v[14] = a[8]; v[15] = a[10]; v[16] = a[11];
        double lo = 0.0, hi = 0.0;
#pragma unroll
        for (int t = 0; t < BT_RINGS; ++t)
            if (t == r) {
                lo = v[t];
                hi = v[t + 8];
            }
        double* out = rec.bi;  // bi[8] and ig[9] are contiguous
        out[r] = lo;
        out[r + 8] = hi;
        if (r == 0) out[16] = v[16];
    }
}

// ----------------------------------------------------------------------------
// Global quantities of the fluid (fluid_global_quantities.f90:66-72: mass,
// linear momentum, angular momentum about the origin, volume) as compensated
// FP64 sums: every partial sum is a double-double (s + c, Knuth's TwoSum on
// each addition), so the result is the exact sum of the terms rounded once,
// whatever the reduction order.
// ----------------------------------------------------------------------------
struct DD {
    double s, c;
};
__device__ __forceinline__ DD dd_add(DD x, DD y) {
    const double s = x.s + y.s;
    const double bp = s - x.s;
    const double e = (x.s - (s - bp)) + (y.s - bp);
    const double c = e + (x.c + y.c);
    const double s2 = s + c;  // renormalise (|s| >= |c|)
    return DD{s2, c - (s2 - s)};
}
__device__ __forceinline__ DD dd_shfl_xor(DD v, int o) {
    return DD{__shfl_xor(v.s, o, 64), __shfl_xor(v.c, o, 64)};
}

constexpr int GQ_N = 8;  // mass, lin mom x3, ang mom x3, volume

__global__ __launch_bounds__(256) void k_global_partial(const double4* __restrict__ xm,
                                                        const double4* __restrict__ vel,
                                                        const double2* __restrict__ rp,
                                                        double* __restrict__ part, const int* iscal) {
    __shared__ double red[4][GQ_N][2];
    const int n = iscal[IS_N];
    DD acc[GQ_N];
    for (int q = 0; q < GQ_N; ++q) acc[q] = DD{0.0, 0.0};
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const double4 x = xm[i];
        const double4 v = vel[i];
        const double m = x.w;
        // Vector_Product(coord, vel)
        const double a0 = x.y * v.z - x.z * v.y;
        const double a1 = x.z * v.x - x.x * v.z;
        const double a2 = x.x * v.y - x.y * v.x;
        const double t[GQ_N] = {m, m * v.x, m * v.y, m * v.z, m * a0, m * a1, m * a2, m / rp[i].x};
#pragma unroll
        for (int q = 0; q < GQ_N; ++q) acc[q] = dd_add(acc[q], DD{t[q], 0.0});
    }
#pragma unroll
    for (int q = 0; q < GQ_N; ++q)
        for (int o = 32; o > 0; o >>= 1) acc[q] = dd_add(acc[q], dd_shfl_xor(acc[q], o));
    const int wid = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
        for (int q = 0; q < GQ_N; ++q) {
            red[wid][q][0] = acc[q].s;
            red[wid][q][1] = acc[q].c;
        }
    __syncthreads();
    if (threadIdx.x < GQ_N) {
        const int q = threadIdx.x;
        DD r = DD{red[0][q][0], red[0][q][1]};
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w) r = dd_add(r, DD{red[w][q][0], red[w][q][1]});
        part[(size_t)blockIdx.x * GQ_N * 2 + 2 * q] = r.s;
        part[(size_t)blockIdx.x * GQ_N * 2 + 2 * q + 1] = r.c;
    }
}

__global__ void k_global_final(const double* __restrict__ part, int nblocks, double* __restrict__ out) {
    const int q = threadIdx.x;
    if (q >= GQ_N) return;
    DD r = DD{0.0, 0.0};
    for (int b = 0; b < nblocks; ++b)
        r = dd_add(r, DD{part[(size_t)b * GQ_N * 2 + 2 * q], part[(size_t)b * GQ_N * 2 + 2 * q + 1]});
    out[q] = r.s + r.c;
}

// ----------------------------------------------------------------------------
// The state in pg order (row = particle id), one array per field: a
// permutation that is a latency-bound sort on the host (576,000 particles:
// state() 45 -> 6.6 ms) and a pass of scattered 8-byte stores here.
// bad: set where an id is not a row (a sort that could not renumber).
// ----------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_pack_state(const double4* __restrict__ xm, const double4* __restrict__ vel,
                                                    const double4* __restrict__ acc,
                                                    const double2* __restrict__ rp,
                                                    const double* __restrict__ dden,
                                                    const double* __restrict__ vpres, int n,
                                                    double* __restrict__ o_x, double* __restrict__ o_v,
                                                    double* __restrict__ o_a, double* __restrict__ o_s, int* bad) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const double4 v = vel[p];
    const int r = (int)v.w;
    if (r < 0 || r >= n) {
        *bad = 1;
        return;
    }
    const double4 x = xm[p], a = acc[p];
    const double2 q = rp[p];
    double* ox = o_x + 3 * (size_t)r;
    double* ov = o_v + 3 * (size_t)r;
    double* oa = o_a + 3 * (size_t)r;
    ox[0] = x.x; ox[1] = x.y; ox[2] = x.z;
    ov[0] = v.x; ov[1] = v.y; ov[2] = v.z;
    oa[0] = a.x; oa[1] = a.y; oa[2] = a.z;
    double* os = o_s + r;
    const size_t m = (size_t)n;
    os[0] = q.x;
    os[m] = q.y;
    os[2 * m] = dden[p];
    os[3 * m] = vpres[p];
}

// ----------------------------------------------------------------------------
// Free-surface monitor lines: calc_pelo.f90:82-131.  One workgroup per line;
// each thread takes one point of a FS_WG-point chunk: its cell (the ceiling
// form of CalcVarp.f90:66-72, with out-of-range indices giving cell 0 before
// any integer conversion), then the two particles of that cell closest to
// the point.  The reference takes them with two minloc passes over an array
// preset to 9e12; a running (first, second) minimum with strict comparisons
// in cell order (ascending particle index, as NPartOrd) picks the same pair,
// because a point and a particle of the same cell are closer than 9e12.  A
// cell holding one particle gives that particle twice.  Thread 0 then runs
// the reference's sequential flags over the chunk: pelolib takes the last
// filled cell, z_lower_fluid_top stops at the first empty cell above fluid;
// cells outside the grid are skipped.
// icont: control_lines(:)%Icont, 1-based (first, last); the reference starts
// at Icont(1)+1, which is 0-based index Icont(1).
// out[3*line + d] = pelolib, out[3*(nlines + line) + d] = z_lower_fluid_top.
// ----------------------------------------------------------------------------
constexpr int FS_WG = 256;

__device__ __forceinline__ int d_point_cell(DPC& P, double x, double y, double z) {
    const double q[3] = {x, y, z};
    int ijk[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const double f = ceil((q[d] - P.extr_lo[d]) / P.dcd[d]);
        if (!(f >= 1.0 && f <= (double)P.ncd[d])) return 0;  // also NaN
        ijk[d] = (int)f;
    }
    return d_cell_number(P, ijk[0], ijk[1], ijk[2]);
}

__global__ __launch_bounds__(FS_WG) void k_free_surface(DPC* Pp, const double4* __restrict__ xm,
                                                       const int* __restrict__ start,
                                                       const double* __restrict__ pts,
                                                       const int* __restrict__ icont, int nlines,
                                                       double* __restrict__ out) {
    DPC& P = *Pp;
    __shared__ double val[FS_WG][3];
    __shared__ int st[FS_WG];  // 0 outside the grid, 1 empty cell, 2 filled cell
    const int line = blockIdx.x;
    const int j0 = icont[2 * line], j1 = icont[2 * line + 1];
    bool zflag = true, below = false;
    double pel[3] = {0.0, 0.0, 0.0}, zl[3] = {0.0, 0.0, 0.0};
    const double half_dx = P.dx / 2.0;
    for (int base = j0; base < j1; base += FS_WG) {
        const int j = base + (int)threadIdx.x;
        int s = 0;
        if (j < j1) {
            const double qx = pts[3 * j], qy = pts[3 * j + 1], qz = pts[3 * j + 2];
            const int c = d_point_cell(P, qx, qy, qz);
            if (c > 0) {
                const int b = start[c - 1], e = start[c];
                s = e > b ? 2 : 1;
                if (s == 2) {
                    double m1 = 0.0, m2 = 0.0;
                    int i1 = -1, i2 = -1;
                    for (int m = b; m < e; ++m) {
                        const double4 x = xm[m];
                        const double r0 = qx - x.x, r1 = qy - x.y, r2 = qz - x.z;
                        const double d2 = r0 * r0 + r1 * r1 + r2 * r2;
                        if (i1 < 0 || d2 < m1) {
                            m2 = m1;
                            i2 = i1;
                            m1 = d2;
                            i1 = m;
                        } else if (i2 < 0 || d2 < m2) {
                            m2 = d2;
                            i2 = m;
                        }
                    }
                    if (i2 < 0) i2 = i1;
                    const double4 a = xm[i1], bb = xm[i2];
                    val[threadIdx.x][0] = (a.x + bb.x) * 0.5 + half_dx;
                    val[threadIdx.x][1] = (a.y + bb.y) * 0.5 + half_dx;
                    val[threadIdx.x][2] = (a.z + bb.z) * 0.5 + half_dx;
                }
            }
        }
        st[threadIdx.x] = s;
        __syncthreads();
        if (threadIdx.x == 0) {
            const int nt = min(FS_WG, j1 - base);
            for (int t = 0; t < nt; ++t) {
                if (st[t] == 0) continue;
                if (st[t] == 1) {
                    if (below) zflag = false;
                    continue;
                }
                for (int d = 0; d < 3; ++d) {
                    pel[d] = val[t][d];
                    if (zflag) zl[d] = val[t][d];
                }
                below = true;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int d = 0; d < 3; ++d) {
            out[3 * line + d] = pel[d];
            out[3 * (nlines + line) + d] = zl[d];
        }
}

// ----------------------------------------------------------------------------
// dt: time_step_duration.f90:74-116.  Positive doubles order like their bit
// patterns, so the minimum over particles is an exact atomicMin on uint64.
// ----------------------------------------------------------------------------
__device__ __forceinline__ double d_dt_cfl(DPC& P, double vx, double vy, double vz) {
    const double U = sqrt(vx * vx + vy * vy + vz * vz);
    return P.cfl * 2.0 * P.h / (P.celerita + U);
}

__device__ __forceinline__ void block_min_to(unsigned long long v, unsigned long long* dst) {
    __shared__ unsigned long long red[16];
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long t = __shfl_xor(v, o, 64);
        v = t < v ? t : v;
    }
    const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) red[wid] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long m = red[0];
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w) m = red[w] < m ? red[w] : m;
        atomicMin(dst, m);
    }
}

// The wave's minimum of v into *dst, and v reset.  The minimum only falls: a
// value read before the atomic is an upper bound of it.
__device__ __forceinline__ void wave_min_to(unsigned long long& v, unsigned long long* dst) {
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long t = __shfl_xor(v, o, 64);
        v = t < v ? t : v;
    }
    if ((threadIdx.x & 63) == 0 && v < *(volatile unsigned long long*)dst) atomicMin(dst, v);
    v = 0x7FF0000000000000ull;
}

template <bool SG>
__global__ __launch_bounds__(256) void k_dtmin(Seg S, const double4* __restrict__ vel,
                                               unsigned long long* dtmin, const int* iscal) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int sg = SG ? __builtin_amdgcn_readfirstlane(S.pblk[(blockIdx.x * blockDim.x) >> 8]) : 0;
    DPC& P = S.P[sg];
    dtmin += sg;
    unsigned long long v = 0x7FF0000000000000ull;
    if (i - P.base < iscal[sg * IS_COUNT + IS_N]) {
        const double4 u = vel[i];
        v = (unsigned long long)__double_as_longlong(d_dt_cfl(P, u.x, u.y, u.z));
    }
    block_min_to(v, dtmin);
}

// step prologue (time_step_loop.f90:180-186): dt_previous_step, dt, time
// Segmented contexts: one lane per segment.
template <bool SG>
__global__ void k_dt_begin(Seg S, double* scal, unsigned long long* dtmin, int* iscal, int advance) {
    const int sg = SG ? (int)(blockIdx.x * blockDim.x + threadIdx.x) : 0;
    if (SG ? sg >= S.nseg : (threadIdx.x != 0 || blockIdx.x != 0)) return;
    DPC& P = S.P[sg];
    scal += sg * SC_COUNT;
    iscal += sg * IS_COUNT;
    dtmin += sg;
    if (advance) {
        iscal[IS_IT] += 1;
        iscal[IS_ONGOING] = iscal[IS_IT];
        scal[SC_DTPREV] = scal[SC_DT];
    }
    const int og = iscal[IS_ONGOING];
    double dtmin_v = 3.4e38;
    double dt_vis = 3.4e38;
    if (P.kin_visc > 1.0e-24) {
        dt_vis = P.vsc_coeff * P.squareh / (0.5 * P.kin_visc);
        dtmin_v = fmin(dtmin_v, dt_vis);
    }
    const double mparts = __longlong_as_double((long long)*dtmin);
    if (iscal[IS_N] == 0) {
        scal[SC_DT] = 0.0;
    } else {
        dtmin_v = fmin(dtmin_v, fmin(mparts, dt_vis));
        if (og == 0) scal[SC_DT] = dtmin_v;
        else scal[SC_DT] = (1.0 - P.pesodt) * dtmin_v + P.pesodt * scal[SC_DTAVG];
    }
    const double dt = scal[SC_DT];
    if (og == 0) scal[SC_DTAVG] = dt;
    else scal[SC_DTAVG] = (scal[SC_DTAVG] * (double)(og - 1) + dt) / (double)og;
    if (advance) scal[SC_TIME] = scal[SC_TIME] + dt;
    scal[SC_DTVEL] = 0.5 * (dt + scal[SC_DTPREV]);
    scal[SC_TV1] = P.tetav * P.celerita * dt / P.h;
    scal[SC_TP1] = P.tetap * P.celerita * dt / P.h;
    *dtmin = 0x7FF0000000000000ull;
}

// the row a with pre[a] <= x < pre[a + 1] of the prefix sums pre[0..rows]
__device__ __forceinline__ int tile_find(const int* pre, int rows, int x) {
    int a = 0;
#pragma unroll
    for (int s = 32; s > 0; s >>= 1)
        if (a + s < rows && pre[a + s] <= x) a += s;
    return a;
}

// Runs the tiles that hold particles: stage(P, segment, sorted index, slot)
// for every slot of a tile that fits, then part(P, segment, sorted index,
// slot, fits) with G lanes for every home particle, then done(P, segment).  A
// workgroup takes the tiles of its XCD's contiguous share, so tiles that share
// halo rows share an L2.  TILED false: G lanes for every particle, 256 threads
// a block (its slots lie in one segment), nothing staged.
template <bool SG, int G, int U, bool TILED = true, class Stage, class Part, class Done>
__device__ __forceinline__ void for_tiles(const Seg& S, const Tiles& T,
                                          const int* __restrict__ start, Stage&& stage, Part&& part,
                                          Done&& done) {
    if constexpr (!TILED) {
        const int vb = xcd_block(gridDim.x), i = (vb * 256 + (int)threadIdx.x) / G;
        const int sg = SG ? __builtin_amdgcn_readfirstlane(S.pblk[(vb * 256 / G) >> 8]) : 0;
        DPC& P = S.P[sg];
        if (i < start[P.koff + P.nmax]) part(P, sg, i, 0, false);
        done(P, sg);
        return;
    }
    __shared__ TileS ts;
    const int nt = *T.n;
    const int per = gridDim.x >> 3, xcd = blockIdx.x & 7;  // gridDim.x is a multiple of 8
    const int t1 = (int)((long long)nt * (xcd + 1) / 8);
    const int lane = threadIdx.x & 63;
    for (int t = (int)((long long)nt * xcd / 8) + (blockIdx.x >> 3); t < t1; t += per) {
        const int id = __builtin_amdgcn_readfirstlane(T.list[t]);
        const int sg = SG ? __builtin_amdgcn_readfirstlane(S.tblk[id >> 8]) : 0;
        DPC& P = S.P[sg];
        const int rows = tile_rows(P);
        if (threadIdx.x < 64) {
            int ti, tj, tk, g0, g1, h0, h1;
            tile_coords(P, id, ti, tj, tk);
            tile_row(P, start, ti, tj, tk, lane, g0, g1, h0, h1);
            const int a = wave_incl_scan(g1 - g0), b = wave_incl_scan(h1 - h0);
            ts.g[lane] = g0;
            ts.h0[lane] = h0;
            ts.l[lane + 1] = a;
            ts.hp[lane + 1] = b;
            if (lane == 0) ts.l[0] = ts.hp[0] = 0;
        }
        __syncthreads();
        const int total = ts.l[rows], nhome = ts.hp[rows];
        const bool fits = total <= P.tcap;
        if (fits) {
            // U slots per thread at a time, so that their loads are in flight
            // together (a slot past the end repeats the last one)
            const int bs = blockDim.x;
            for (int e0 = threadIdx.x; e0 < total; e0 += U * bs) {
                int e[U], g[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    e[u] = min(e0 + u * bs, total - 1);
                    const int r = tile_find(ts.l, rows, e[u]);
                    g[u] = ts.g[r] + e[u] - ts.l[r];
                }
#pragma unroll
                for (int u = 0; u < U; ++u) stage(P, sg, g[u], e[u]);
            }
        }
        __syncthreads();
        for (int q = threadIdx.x / G; q < nhome; q += blockDim.x / G) {
            const int a = tile_find(ts.hp, rows, q);
            const int i = ts.h0[a] + q - ts.hp[a];
            part(P, sg, i, i - ts.g[a] + ts.l[a], fits);
        }
        done(P, sg);
        __syncthreads();  // the slots and rows are reused
    }
}

// Particles in tiles that have more than cap slots, or whose solve's records do
// not fit the LDS form (FP64 with several masses), added to *out: a wavefront a
// tile.
template <bool SG>
__global__ __launch_bounds__(256) void k_tile_unfit(Seg S, Tiles T, const int* __restrict__ start, int cap, int* out) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    int n = 0;
    for (int t = blockIdx.x * 4 + wid; t < *T.n; t += gridDim.x * 4) {
        const int id = __builtin_amdgcn_readfirstlane(T.list[t]);
        DPC& P = S.P[SG ? __builtin_amdgcn_readfirstlane(S.tblk[id >> 8]) : 0];
        int ti, tj, tk, g0, g1, h0, h1;
        tile_coords(P, id, ti, tj, tk);
        tile_row(P, start, ti, tj, tk, lane, g0, g1, h0, h1);
        const int total = __builtin_amdgcn_readlane(wave_incl_scan(g1 - g0), 63);
        if (total > (P.f32 || P.umass ? cap : 0)) n += __builtin_amdgcn_readlane(wave_incl_scan(h1 - h0), 63);
    }
    if (lane == 0 && n) atomicAdd(out, n);
}

// 16 bytes at byte offset o of an LDS array
__device__ __forceinline__ float4 lds16(const float4* a, uint32_t o) {
    return *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(a) + o);
}

// wall_function_for_SASPH.f90:56-80 (no land-cover map), FP64: slip
// coefficient and mixing-length viscosity of one particle-frontier pair at
// distance r; d50 is ten times the frontier's roughness length.  Nepero_number
// and k_v: Static_allocation_module.f90:51,53.
__device__ __forceinline__ void wall_function(double u_t, double d50, double r, double dx,
                                              double& slip, double& nut) {
    const double e = 2.718281828, kv2 = 0.41 * 0.41;
    slip = 0.0;
    nut = 1.0e-15;
    if (r <= 0.5 * dx) {
        const double z0 = d50 / 10.0;
        if (r < z0 * e) {
            slip = 1.0;
            nut = kv2 * u_t * z0 * e;
        } else {
            const double L = log(r / z0);
            slip = 1.0 / L;
            nut = kv2 * u_t * r / L;
        }
    }
}

// line_plane_intersection.f90:39-76 with three_plane_intersection.f90:42-66
// and Matrix_Inversion_3x3.f90:39-58, FP64: the point where the line through
// P1 and P2 meets the plane through A, B and C (two planes through the line,
// each with a point 999 away from P1, and the plane); false when the 3x3
// system's |determinant| is below 1e-36.
__device__ bool d_line_plane(const double P1[3], const double P2[3], const double A[3], const double B[3],
                             const double C[3], double X[3]) {
    const double Q1[3] = {P1[0] - 999.0, P1[1], P1[2]};
    const double Q2[3] = {P1[0], P1[1] - 999.0, P2[2] == P2[2] ? P1[2] - 999.0 : P1[2]};
    double m[3][3], dv[3];
    for (int r = 0; r < 2; ++r) {
        const double* Q = r == 0 ? Q1 : Q2;
        m[r][0] = (P2[1] - P1[1]) * (Q[2] - P1[2]) - (Q[1] - P1[1]) * (P2[2] - P1[2]);
        m[r][1] = -((P2[0] - P1[0]) * (Q[2] - P1[2]) - (Q[0] - P1[0]) * (P2[2] - P1[2]));
        m[r][2] = (P2[0] - P1[0]) * (Q[1] - P1[1]) - (Q[0] - P1[0]) * (P2[1] - P1[1]);
        dv[r] = -(m[r][0] * P1[0] + m[r][1] * P1[1] + m[r][2] * P1[2]);
    }
    m[2][0] = (B[1] - A[1]) * (C[2] - A[2]) - (C[1] - A[1]) * (B[2] - A[2]);
    m[2][1] = -((B[0] - A[0]) * (C[2] - A[2]) - (C[0] - A[0]) * (B[2] - A[2]));
    m[2][2] = (B[0] - A[0]) * (C[1] - A[1]) - (C[0] - A[0]) * (B[1] - A[1]);
    dv[2] = -(m[2][0] * A[0] + m[2][1] * A[1] + m[2][2] * A[2]);
    const double det = m[0][0] * m[1][1] * m[2][2] + m[1][0] * m[2][1] * m[0][2] +
                       m[2][0] * m[0][1] * m[1][2] - m[0][0] * m[2][1] * m[1][2] -
                       m[2][0] * m[1][1] * m[0][2] - m[1][0] * m[0][1] * m[2][2];
    if (!(fabs(det) >= 1.0e-36)) return false;
    double inv[3][3];
    inv[0][0] = m[1][1] * m[2][2] - m[1][2] * m[2][1];
    inv[0][1] = m[0][2] * m[2][1] - m[0][1] * m[2][2];
    inv[0][2] = m[0][1] * m[1][2] - m[0][2] * m[1][1];
    inv[1][0] = m[1][2] * m[2][0] - m[1][0] * m[2][2];
    inv[1][1] = m[0][0] * m[2][2] - m[0][2] * m[2][0];
    inv[1][2] = m[0][2] * m[1][0] - m[0][0] * m[1][2];
    inv[2][0] = m[1][0] * m[2][1] - m[1][1] * m[2][0];
    inv[2][1] = m[0][1] * m[2][0] - m[0][0] * m[2][1];
    inv[2][2] = m[0][0] * m[1][1] - m[0][1] * m[1][0];
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) inv[i][j] = inv[i][j] / det;
    const double b[3] = {-dv[0], -dv[1], -dv[2]};
    for (int i = 0; i < 3; ++i) X[i] = inv[i][0] * b[0] + inv[i][1] * b[1] + inv[i][2] * b[2];
    return true;
}

// CancelOutgoneParticles_3D.f90:67-158 for one open face, FP64: the step from
// xo to xn ends on the face's outer side, started on its inner side, and
// the segment crosses the face's plane inside the face.
__device__ bool open_face_crossed(const DFace& F, const double xo[3], const double xn[3]) {
    const int nodes = F.nodes;
    const double* G1 = &F.GX[0];
    const double* G2 = &F.GX[3];
    const double* G3 = &F.GX[6];
    const double* Gn = &F.GX[3 * (nodes - 1)];
    const double dx21 = G2[0] - G1[0], dx31 = G3[0] - G1[0];
    const double dy21 = G2[1] - G1[1], dy31 = G3[1] - G1[1];
    const double dz21 = G2[2] - G1[2], dz31 = G3[2] - G1[2];
    auto det_of = [&](const double* X) {
        const double dx = X[0] - G1[0], dy = X[1] - G1[1], dz = X[2] - G1[2];
        return dx21 * dy31 * dz + dx31 * dy * dz21 + dx * dy21 * dz31 - dx21 * dy * dz31 - dx31 * dy21 * dz -
               dx * dy31 * dz21;
    };
    const double dn = det_of(xn);
    if (!(dn <= 0.0)) return false;
    const double dpo = det_of(xo);
    if (copysign(1.0, dn) == copysign(1.0, dpo)) return false;
    // local coordinates (T(:,i) . (X - node(nodes))) of the face's nodes 1-3 and of both ends
    double Pp[3][3], Ln[3], Lo[3];
    const double* Gk[3] = {G1, G2, G3};
    for (int sdi = 0; sdi < 3; ++sdi) {
        for (int k = 0; k < 3; ++k) {
            double a = 0.0;
            for (int sdj = 0; sdj < 3; ++sdj) a = a + F.T[3 * sdi + sdj] * (Gk[k][sdj] - Gn[sdj]);
            Pp[k][sdi] = a;
        }
        double a = 0.0, b = 0.0;
        for (int sdj = 0; sdj < 3; ++sdj) {
            a = a + F.T[3 * sdi + sdj] * (xn[sdj] - Gn[sdj]);
            b = b + F.T[3 * sdi + sdj] * (xo[sdj] - Gn[sdj]);
        }
        Ln[sdi] = a;
        Lo[sdi] = b;
    }
    double LX[3];
    if (!d_line_plane(Ln, Lo, Pp[0], Pp[1], Pp[2], LX)) return false;
    return d_point_internal(pic_of(F), LX[0], LX[1]);
}

// CancelOutgoneParticles_2D.f90:80-101 for one open side (x-z plane), FP64:
// the step from xo to xn ends on the outer side of the side's line
// (determinant <= 0), started on the other, and the side's two vertices lie
// on opposite sides of the step's line.
__device__ bool open_side_crossed(const DFace& S, const double xo[3], const double xn[3]) {
    const double o1x = S.v1[0], o1z = S.v1[1], o2x = S.v2[0], o2z = S.v2[1];
    const double dn = (xn[2] - o1z) * (o2x - o1x) - (xn[0] - o1x) * (o2z - o1z);
    if (!(dn <= 0.0)) return false;
    const double dold = (xo[2] - o1z) * (o2x - o1x) - (xo[0] - o1x) * (o2z - o1z);
    if (copysign(1.0, dn) == copysign(1.0, dold)) return false;
    const double d1 = (o1z - xo[2]) * (xn[0] - xo[0]) - (o1x - xo[0]) * (xn[2] - xo[2]);
    const double d2 = (o2z - xo[2]) * (xn[0] - xo[0]) - (o2x - xo[0]) * (xn[2] - xo[2]);
    return copysign(1.0, d1) != copysign(1.0, d2);
}

// SA-SPH terms of the momentum equation (AddBoundaryContributions_to_ME3D.f90:
// 118-336), FP64; tp/td/tv start at zero
__device__ __forceinline__ void sa_momentum(DPC& P, const DFace* __restrict__ faces,
                                            const BTab* __restrict__ bt, int i, int ncbf,
                                            const double v_i[3], double2 rpi, int lam_prev,
                                            double tp[3], double td[3], double tv[3], int* iscal) {
    const double h = P.h;
    double ALEt[3] = {0, 0, 0}, gradpt[3] = {0, 0, 0}, VM[3] = {0, 0, 0}, VS[3] = {0, 0, 0};
    for (int q = 0; q < ncbf; ++q) {
        const BTab& B = bt[(size_t)q * P.cap + i];
        const DFace& F = faces[B.face];
        if (F.btype == 2) continue;
        if (F.btype != 0 && F.btype != 1) {
            atomicAdd(&iscal[IS_UNSUPPORTED], 1);
            break;
        }
        if (!(B.loc[2] > 0.0)) continue;
        double dvij[3], dvn = 0.0;
        for (int sd = 0; sd < 3; ++sd) {
            dvij[sd] = 2.0 * (v_i[sd] - F.vel[sd]);
            dvn = dvn + F.T[6 + sd] * dvij[sd];
        }
        double gl[3];
        for (int sd = 0; sd < 3; ++sd) {
            double a = 0.0;
            for (int sj = 0; sj < 3; ++sj) a = a + F.T[3 * sd + sj] * P.grav[sj];
            gl[sd] = a;
        }
        double gloc[3];
        for (int r = 0; r < 3; ++r) {
            double a = 0.0;
            for (int k = 0; k < 3; ++k) a = a + B.ig[3 * k + r] * gl[k];
            gloc[r] = a;
        }
        for (int r = 0; r < 3; ++r) {
            double a = 0.0;
            for (int k = 0; k < 3; ++k) a = a + F.T[3 * k + r] * gloc[k];
            gradpt[r] = gradpt[r] + a;
        }
        double aloc[3];
        for (int d = 0; d < 3; ++d) aloc[d] = 2.0 * rpi.y / rpi.x * B.bi[3 + d];
        for (int r = 0; r < 3; ++r) {
            double a = 0.0;
            for (int k = 0; k < 3; ++k) a = a + F.T[3 * k + r] * aloc[k];
            ALEt[r] = ALEt[r] + a;
        }
        if (P.alfamon > 0.0) {
            const double Monvisc = P.alfamon * P.celerita * h;
            const double Mmult = -Monvisc * dvn * B.bi[6];
            for (int d = 0; d < 3; ++d) VM[d] = VM[d] + Mmult * F.T[6 + d];
        }
        double slip = 0.0, cinv = 0.0;
        if (F.mode == 1) {
            slip = F.slip;
            cinv = P.kin_visc;
        } else if (F.mode == 2) {
            // AddBoundaryContributions_to_ME3D.f90:207-227
            double ut[3];
            for (int d = 0; d < 3; ++d) ut[d] = 0.5 * (dvij[d] - dvn * F.T[6 + d]);
            wall_function(sqrt(ut[0] * ut[0] + ut[1] * ut[1] + ut[2] * ut[2]), F.slip * 10.0,
                          B.loc[2], P.dx, slip, cinv);
        }
        if (cinv > 0.0 && (lam_prev == 1 || F.lam == 0)) {
            const double cm = cinv * B.bi[2] * slip;
            for (int d = 0; d < 3; ++d) VS[d] = VS[d] + cm * (2.0 * (v_i[d] - F.vel[d]));
        }
    }
    for (int d = 0; d < 3; ++d) {
        tp[d] = tp[d] + ALEt[d] + gradpt[d];
        td[d] = td[d] - VM[d];
        tv[d] = tv[d] + VS[d];
    }
}

// AddBoundaryContributions_to_ME2D.f90:121-405 for fixe/tapi sides (2D form);
// tp/td/tv start at zero, as the reference's tpres/tdiss/tvisc do
__device__ __forceinline__ void sa_momentum_2d(DPC& P, const DFace* __restrict__ sides,
                                               const BTab* __restrict__ bt, int i, int ncbf,
                                               const double v_i[3], double2 rpi, int lam_prev,
                                               double tp[3], double td[3], double tv[3]) {
    const double ro0 = P.den0, roi = rpi.x, pressi = rpi.y;
    const double distpimin = P.dx;
    double VMo0 = 0.0, VMo1 = 0.0, VSh0 = 0.0, VSh1 = 0.0, RG0s = 0.0, RG1s = 0.0;
    double ALE0 = 0.0, ALE2 = 0.0;
    const double g0 = P.grav[0], g1 = P.grav[2];
    for (int q = 0; q < ncbf; ++q) {
        const BTab& B = bt[(size_t)q * P.cap + i];
        const DFace& S = sides[B.face];
        if (S.btype == 2) continue;  // AddBoundaryContributions_to_ME2D.f90:124
        const double xpi = B.loc[0], ypi = B.loc[1];
        const double IntWdS = B.bi[0], IntWdV = B.bi[2], IntWd1s0 = B.bi[5], IntWd3s0 = B.bi[6];
        const double n0 = S.T[6], n1 = S.T[8];
        double GravN = 0.0;
        GravN = GravN + P.grav[0] * n0;
        GravN = GravN + P.grav[2] * n1;
        const double sv0 = S.btype == 1 ? S.vel[0] : 0.0, sv1 = S.btype == 1 ? S.vel[2] : 0.0;
        const double Dv0 = 2.0 * (v_i[0] - sv0), Dv1 = 2.0 * (v_i[2] - sv1);
        const double DvelN = Dv0 * n0 + Dv1 * n1;
        const double distpi = fmax(ypi, distpimin);
        double pressib = pressi;
        const double pressibmin = 10.0 * ro0 * distpimin;
        if (DvelN <= 0.0) {
            if (pressib < pressibmin) pressib = pressibmin;
        }
        const double PressB = pressib - ro0 * GravN * distpi;
        const double Qii = IntWdS * (pressib + PressB) / roi;
        double RG0 = 0.0, RG1 = 0.0;
        RG0 = RG0 + S.RN[0] * g0;
        RG0 = RG0 + S.RN[1] * g1;
        RG0 = RG0 * IntWdV;
        RG1 = RG1 + S.RN[2] * g0;
        RG1 = RG1 + S.RN[3] * g1;
        RG1 = RG1 * IntWdV;
        RG0s = RG0s + RG0;
        RG1s = RG1s + RG1;
        ALE0 = ALE0 - n0 * Qii;
        ALE2 = ALE2 - n1 * Qii;
        if (xpi >= 0.0 && xpi <= S.len) {
            double slip = 0.0, cinv = 0.0;
            if (S.mode == 1) {
                slip = S.slip;
                cinv = P.kin_visc;
            } else if (S.mode == 2) {
                // AddBoundaryContributions_to_ME2D.f90:314-326
                double ut[3];
                for (int k = 0; k < 3; ++k) ut[k] = (v_i[k] - S.vel[k]) - (0.5 * DvelN * S.T[6 + k]);
                wall_function(sqrt(ut[0] * ut[0] + ut[1] * ut[1] + ut[2] * ut[2]), S.slip * 10.0, ypi,
                              P.dx, slip, cinv);
            }
            const double Monvisc = P.alfamon * P.celerita * P.h;
            const double TN = Monvisc * DvelN * IntWd3s0;
            double SVforce = 0.0;
            if (lam_prev == 1 || S.lam == 0) SVforce = 2.0 * cinv * slip * IntWd1s0;
            VMo0 = VMo0 + TN * n0;
            VMo1 = VMo1 + TN * n1;
            VSh0 = VSh0 + (2.0 * v_i[0]) * SVforce;
            VSh1 = VSh1 + (2.0 * v_i[2]) * SVforce;
        }
    }
    tp[0] = tp[0] - RG0s - ALE0;
    tp[2] = tp[2] - RG1s - ALE2;
    td[0] = td[0] - VMo0;
    td[2] = td[2] - VMo1;
    tv[0] = tv[0] - VSh0;
    tv[2] = tv[2] - VSh1;
}

// AddElasticBoundaryReaction_2D.f90:66-99 over the selected sides
__device__ __forceinline__ void elastic_2d(DPC& P, const DFace* __restrict__ sides,
                                           const BTab* __restrict__ bt, int i, int ncbf,
                                           const double v_i[3], double br[3]) {
    const double h = P.h;
    const double ypimin = 0.25 * P.dx;
    const double celer02 = P.eps / P.den0;
    for (int q = 0; q < ncbf; ++q) {
        const BTab& B = bt[(size_t)q * P.cap + i];
        const DFace& S = sides[B.face];
        if (S.btype != 0 && S.btype != 1) continue;  // AddElasticBoundaryReaction_2D.f90:75
        const double xpi = B.loc[0], ypi = B.loc[1];
        if (ypi < ypimin && xpi > 0.0 && xpi < S.len) {
            double vin = 0.0;
            for (int k = 0; k < 3; ++k) vin = vin + v_i[k] * S.T[6 + k];
            if (vin < 0.0) {
                const double nr = -1.0 * celer02 * log((h + ypi - ypimin) / h) / h;
                for (int d = 0; d < 3; ++d) br[d] = br[d] + nr * S.T[6 + d];
            }
        }
    }
}

// ----------------------------------------------------------------------------
// Per-particle parts of the four passes outside the pair sums, FP64 in both
// forms.
// ----------------------------------------------------------------------------
// elastic wall reaction (AddElasticBoundaryReaction_3D.f90:67-152, _2D) of a
// particle with ncbf > 0 close frontiers
__device__ __forceinline__ void elastic_walls(DPC& P, const DFace* __restrict__ faces,
                                              const DEdge* __restrict__ edges, const BTab* __restrict__ bt,
                                              const double4* __restrict__ xm, int i, int ncbf, double4 vi,
                                              double br[3]) {
    const double v_i[3] = {vi.x, vi.y, vi.z};
    if (P.dim == 2) {
        elastic_2d(P, faces, bt, i, ncbf, v_i, br);
        return;
    }
    const double h = P.h;
    const double zimin = 0.25 * P.dx;
    const double celer02 = P.eps / P.den0;
    // AddElasticBoundaryReaction_3D.f90:72-104 (faces); rea: the
    // slots whose face reacted (ReaFace), for the edges below
    static_assert(SPH_MB <= 32, "one ReaFace bit per boundary-table slot");
    unsigned rea = 0u;
    for (int q = 0; q < ncbf; ++q) {
        const BTab& B = bt[(size_t)q * P.cap + i];
        const DFace& F = faces[B.face];
        if (F.btype != 0 && F.btype != 1) continue;
        const double zi = B.loc[2];
        if (zi < zimin && d_point_internal(F, B.loc[0], B.loc[1])) {
            double vin = 0.0;
            for (int sd = 0; sd < 3; ++sd) vin = vin + v_i[sd] * F.T[6 + sd];
            if (vin < 0.0) {
                const double nr = -1.0 * celer02 * log((h + zi - zimin) / h) / h;
                for (int d = 0; d < 3; ++d) br[d] = br[d] + nr * F.T[6 + d];
            }
            rea |= 1u << q;
        }
    }
    // AddElasticBoundaryReaction_3D.f90:106-152 (convex edges, in
    // order; the reference returns at the first edge whose two
    // faces are not both among the particle's non-reacting faces)
    for (int ne = 0; ne < P.ne; ++ne) {
        const DEdge& E = edges[P.eoff + ne];
        int nclose = 0;
        for (int q = 0; q < ncbf; ++q) {
            const int f = bt[(size_t)q * P.cap + i].face;
            const bool rq = (rea >> q) & 1u;
            if (f == E.face[0] && !rq) ++nclose;
            else if (f == E.face[1] && !rq) ++nclose;
        }
        if (nclose != 2) break;
        const double4 xi = xm[i];
        const double x[3] = {xi.x, xi.y, xi.z};
        double scaprod = 0.0;
        for (int sd = 0; sd < 3; ++sd) scaprod = scaprod + (x[sd] - E.gx[sd]) * E.comp[sd];
        const double tau = scaprod / (E.len * E.len);
        if (tau >= 0.0 && tau <= 1.0) {
            double QP[3], d2 = 0.0;
            for (int sd = 0; sd < 3; ++sd) QP[sd] = x[sd] - (E.gx[sd] + E.comp[sd] * tau);
            for (int sd = 0; sd < 3; ++sd) d2 = d2 + QP[sd] * QP[sd];
            const double zi = sqrt(d2);
            if (zi < zimin) {
                double cd[3], vin = 0.0;
                for (int sd = 0; sd < 3; ++sd) cd[sd] = QP[sd] / zi;
                for (int sd = 0; sd < 3; ++sd) vin = vin + v_i[sd] * cd[sd];
                if (vin < 0.0) {
                    const double nr = -1.0 * celer02 * log(zi / zimin) / zimin;
                    for (int d = 0; d < 3; ++d) br[d] = br[d] + nr * cd[d];
                }
            }
        }
    }
}

// The wall terms of the FP32-mixed momentum pass as calls: inlined, their FP64
// values raise the kernel above the 128 registers that two workgroups a CU
// allow, and it spills (576,000 particles: 151 us
// against 116).  Few particles take them.
struct Walls6 {
    double tp[3], tdv[3];  // pressure terms; Monaghan's and the shear terms
};
struct Walls3 {
    double r[3];
};
__device__ __attribute__((noinline)) Walls6 wall_terms(DPC* P, const DFace* __restrict__ faces,
                                                       const BTab* __restrict__ bt, int i, int ncbf, double vx,
                                                       double vy, double vz, double rho, double p, int lam,
                                                       int* iscal) {
    double tp[3] = {0.0, 0.0, 0.0}, td[3] = {0.0, 0.0, 0.0}, tv[3] = {0.0, 0.0, 0.0};
    const double v_i[3] = {vx, vy, vz};
    if (P->dim == 2)
        sa_momentum_2d(*P, faces, bt, i, ncbf, v_i, make_double2(rho, p), lam, tp, td, tv);
    else
        sa_momentum(*P, faces, bt, i, ncbf, v_i, make_double2(rho, p), lam, tp, td, tv, iscal);
    return Walls6{{tp[0], tp[1], tp[2]}, {td[0] + tv[0], td[1] + tv[1], td[2] + tv[2]}};
}
__device__ __attribute__((noinline)) Walls3 wall_elastic(DPC* P, const DFace* __restrict__ faces,
                                                         const DEdge* __restrict__ edges,
                                                         const BTab* __restrict__ bt,
                                                         const double4* __restrict__ xm, int i, int ncbf,
                                                         double vx, double vy, double vz) {
    double br[3] = {0.0, 0.0, 0.0};
    elastic_walls(*P, faces, edges, bt, xm, i, ncbf, make_double4(vx, vy, vz, 0.0), br);
    return Walls3{{br[0], br[1], br[2]}};
}

// laminar flag, acceleration and Leapfrog_momentum.f90:66-86 (RK1:
// Euler.f90:85-93); br: the elastic wall reaction, for ncbf > 0.  Returns the
// new velocity.
__device__ __forceinline__ double4 momentum_end(DPC& P, int i, int ncbf, double4 vi, double dtvel,
                                                const double tp[3], const double td[3], const double tv[3],
                                                const double rvs[3], const double br[3],
                                                int* __restrict__ lam_out, double4* __restrict__ acc_out,
                                                double4* __restrict__ vel_out) {
    int lam = 0;
    if (P.kin_visc > 0.0) {
        const double apg = sqrt(tp[0] * tp[0] + tp[1] * tp[1] + tp[2] * tp[2]) + P.GI;
        const double amo = sqrt(rvs[0] * rvs[0] + rvs[1] * rvs[1] + rvs[2] * rvs[2]);
        double w = 0.0;
        if (apg != 0.0) w = amo / apg * 100.0;
        lam = (w > 5.0 || apg == 0.0) ? 1 : 0;
    }
    lam_out[i] = lam;
    double a[3];
    for (int d = 0; d < 3; ++d) a[d] = tp[d] + td[d] + tv[d] + P.grav[d];
    if (ncbf > 0)
        for (int d = 0; d < 3; ++d) a[d] = a[d] + br[d];
    acc_out[i] = make_double4(a[0], a[1], a[2], 0.0);
    // vel = vel + dtvel*acc (kodvel == 0)
    const double4 vn =
        make_double4(vi.x + dtvel * a[0], vi.y + dtvel * a[1], vi.z + dtvel * a[2], vi.w);
    vel_out[i] = vn;
    return vn;
}

// wall terms of the velocity smoothing (velocity_smoothing_SA_SPH_3D.f90:64-122, _2D)
__device__ __forceinline__ void vsmooth_walls(DPC& P, const DFace* __restrict__ faces,
                                              const BTab* __restrict__ bt, int i, int ncbf, double4 vi,
                                              double v[3]) {
    // velocity_smoothing_SA_SPH_2D.f90:64-118 (fixe/tapi sides)
    for (int q = 0; q < ncbf && P.dim == 2; ++q) {
        const BTab& B = bt[(size_t)q * P.cap + i];
        const DFace& S = faces[B.face];
        if (S.btype != 0 && S.btype != 1) continue;
        const double s0 = S.T[0], s1 = S.T[2], n0 = S.T[6], n1 = S.T[8];
        const double DVG0 = 2.0 * (S.tvel[0] - vi.x), DVG1 = 2.0 * (S.tvel[2] - vi.z);
        const double DVL0 = s0 * DVG0 + s1 * DVG1;
        const double DVL1 = n0 * DVG0 + n1 * DVG1;
        const double IntWdV = B.bi[2];
        double slip = S.mode == 1 ? S.slip : 0.0;
        if (S.mode == 2) {
            // velocity_smoothing_SA_SPH_2D.f90:93-106
            const double u0 = (S.tvel[0] - vi.x) - (0.5 * DVL1 * S.T[6]);
            const double u1 = (S.tvel[1] - vi.y) - (0.5 * DVL1 * S.T[7]);
            const double u2 = (S.tvel[2] - vi.z) - (0.5 * DVL1 * S.T[8]);
            double nut;
            wall_function(sqrt(u0 * u0 + u1 * u1 + u2 * u2), S.slip * 10.0, B.loc[1], P.dx,
                          slip, nut);
        }
        const double BCL0 = DVL0 * IntWdV * slip;
        const double BCL1 = DVL1 * IntWdV;
        v[0] = v[0] + (s0 * BCL0 + n0 * BCL1);
        v[2] = v[2] + (s1 * BCL0 + n1 * BCL1);
    }
    for (int q = 0; q < ncbf && P.dim == 3; ++q) {
        const BTab& B = bt[(size_t)q * P.cap + i];
        const DFace& F = faces[B.face];
        if (F.btype == 3 || F.btype == 4 || F.btype == 5) {
            v[0] = v[1] = v[2] = 0.0;
            break;
        }
        if (F.btype != 0 && F.btype != 1) continue;
        const double DVG[3] = {2.0 * (F.tvel[0] - vi.x), 2.0 * (F.tvel[1] - vi.y),
                               2.0 * (F.tvel[2] - vi.z)};
        double DVL[3];
        for (int ii = 0; ii < 3; ++ii) {
            double a = 0.0;
            for (int jj = 0; jj < 3; ++jj) a = a + F.T[3 * ii + jj] * DVG[jj];
            DVL[ii] = a;
        }
        const double IntWdV = B.bi[1];
        double slip = F.mode == 1 ? F.slip : 0.0;
        if (F.mode == 2) {
            // velocity_smoothing_SA_SPH_3D.f90:89-110
            double ut[3], nut;
            for (int d = 0; d < 3; ++d) ut[d] = 0.5 * (DVG[d] - DVL[2] * F.T[6 + d]);
            wall_function(sqrt(ut[0] * ut[0] + ut[1] * ut[1] + ut[2] * ut[2]), F.slip * 10.0,
                          B.loc[2], P.dx, slip, nut);
        }
        const double BCL[3] = {DVL[0] * IntWdV * slip, DVL[1] * IntWdV * slip,
                               DVL[2] * IntWdV};
        for (int ii = 0; ii < 3; ++ii) {
            double a = 0.0;
            for (int jj = 0; jj < 3; ++jj) a = a + F.T[3 * jj + ii] * BCL[jj];
            v[ii] = v[ii] + a;
        }
    }
}

// CancelOutgoneParticles_3D / _2D: the step from xo to xn crosses an open frontier
__device__ __forceinline__ int open_crossed(DPC& P, const DFace* __restrict__ faces, const double xo[3],
                                            const double xn[3]) {
    int g = 0;
    for (int f = P.foff; f < P.foff + P.nf; ++f)
        if (faces[f].btype == 2 &&
            (P.dim == 2 ? open_side_crossed(faces[f], xo, xn) : open_face_crossed(faces[f], xo, xn)))
            g = 1;
    return g;
}

// The same two as calls, for the FP32-mixed pass (see wall_terms)
__device__ __attribute__((noinline)) int open_crossed_call(DPC* P, const DFace* __restrict__ faces, double x0,
                                                           double y0, double z0, double x1, double y1, double z1) {
    const double xo[3] = {x0, y0, z0}, xn[3] = {x1, y1, z1};
    return open_crossed(*P, faces, xo, xn);
}
__device__ __attribute__((noinline)) Walls3 wall_smooth(DPC* P, const DFace* __restrict__ faces,
                                                        const BTab* __restrict__ bt, int i, int ncbf, double vx,
                                                        double vy, double vz, double sx, double sy, double sz) {
    double v[3] = {sx, sy, sz};
    vsmooth_walls(*P, faces, bt, i, ncbf, make_double4(vx, vy, vz, 0.0), v);
    return Walls3{{v[0], v[1], v[2]}};
}

// velocity_smoothing_2.f90:59-103, Leapfrog_trajectories.f90:48-76, the open
// faces, RK1's density update and the particle part of the next
// time_step_duration; returns the bits of the particle's time step limit
template <bool CALL>
__device__ __forceinline__ unsigned long long vsmooth_end(
    DPC& P, const DFace* __restrict__ faces, int i, double4 xi, double4 vi, const double v[3],
    bool smooth, double tv1, double dt, bool eos, const double* __restrict__ dden_in,
    const double2* __restrict__ rp, double4* __restrict__ vel_out, double4* __restrict__ xm_out,
    double2* __restrict__ rp_out, float* __restrict__ dr_out, int* __restrict__ gone) {
    double4 vn = vi;
    if (smooth) vn = make_double4(vi.x + tv1 * v[0], vi.y + tv1 * v[1], vi.z + tv1 * v[2], vi.w);
    vel_out[i] = vn;

    const double xn[3] = {xi.x + dt * vn.x, xi.y + dt * vn.y, xi.z + dt * vn.z};
    xm_out[i] = make_double4(xn[0], xn[1], xn[2], xi.w);
    // the next time_step_duration runs over the particles the coming
    // OrdGrid1 keeps: not those out of the grid, nor those that left
    // through an open face
    bool stays = d_particle_cell(P, xn[0], xn[1], xn[2]) > 0;
    if (P.nopen > 0) {  // open frontiers, on the step just made
        const double xo[3] = {xi.x, xi.y, xi.z};
        const int g = CALL ? open_crossed_call(&P, faces, xo[0], xo[1], xo[2], xn[0], xn[1], xn[2])
                           : open_crossed(P, faces, xo, xn);
        gone[i] = g;
        stays = stays && !g;
    }
    if (P.rk1 && !P.dbsph) {
        // explicit RK1: Euler.f90:231-241 (dens = dens + dt dden) and
        // EoS_fluid_loop.f90:59-70 (time_integration.f90:52-65); the
        // pressure smoothing that follows reads these with the
        // stage's kernel values, hence the old positions
        const double2 rpi = rp[i];
        const double rho1 = rpi.x + dt * dden_in[i];
        const double p1 = eos ? P.eps / P.den0 * (rho1 - P.den0) + P.prif : rpi.y;
        rp_out[i] = make_double2(rho1, p1);
        if (P.f32) dr_out[i] = (float)(rho1 - P.den0);
    }
    if (!stays) return 0x7FF0000000000000ull;
    return (unsigned long long)__double_as_longlong(d_dt_cfl(P, vn.x, vn.y, vn.z));
}

// wall part of the continuity equation: AddBoundaryContribution_to_CE3D.f90:82-169, _CE2D
__device__ __forceinline__ double continuity_walls(DPC& P, const DFace* __restrict__ faces,
                                                   const BTab* __restrict__ bt, int i, int ncbf, double4 vi,
                                                   double rhoi, int* iscal) {
    double dd = 0.0;
    if (ncbf > 0 && P.dim == 2) {
        // SASPH_continuity.f90:126-169 with AddBoundaryContribution_to_CE2D
        // .f90:74-150 (fixe/tapi sides): grad_u_SA(1) and grad_w_SA(3)
        double gu0 = 0.0, gw2 = 0.0;
        for (int q = 0; q < ncbf; ++q) {
            const BTab& B = bt[(size_t)q * P.cap + i];
            const DFace& S = faces[B.face];
            if (S.btype != 0 && S.btype != 1) continue;
            const double IntWdS = B.bi[0];
            double dv0, dv1;
            if (S.btype == 0) {
                dv0 = 2.0 * (-vi.x);
                dv1 = 2.0 * (-vi.z);
            } else {
                dv0 = 2.0 * (S.vel[0] - vi.x);
                dv1 = 2.0 * (S.vel[2] - vi.z);
            }
            gu0 = gu0 - dv0 * S.T[6] * IntWdS;
            gw2 = gw2 - dv1 * S.T[8] * IntWdS;
        }
        dd = dd - rhoi * (gu0 + 0.0 + gw2);
    } else if (ncbf > 0) {
        double gu = 0.0, gv = 0.0, gw = 0.0;
        const double v_i[3] = {vi.x, vi.y, vi.z};
        for (int q = 0; q < ncbf; ++q) {
            const BTab& B = bt[(size_t)q * P.cap + i];
            const DFace& F = faces[B.face];
            if (F.btype == 0 || F.btype == 1) {
                if (B.loc[2] > 0.0) {
                    double a2[3];
                    for (int d = 0; d < 3; ++d) a2[d] = 2.0 * (F.vel[d] - v_i[d]);
                    const double dp = a2[0] * F.T[6] + a2[1] * F.T[7] + a2[2] * F.T[8];
                    double av[3];
                    for (int r = 0; r < 3; ++r) {
                        double a = 0.0;
                        for (int k = 0; k < 3; ++k) a = a + F.T[3 * k + r] * B.bi[3 + k];
                        av[r] = a;
                    }
                    gu = gu - dp * F.T[6] * av[0];
                    gv = gv - dp * F.T[7] * av[1];
                    gw = gw - dp * F.T[8] * av[2];
                }
            } else if (F.btype >= 3) {
                atomicAdd(&iscal[IS_UNSUPPORTED], 1);
                break;
            }
        }
        dd = dd - rhoi * (gu + gv + gw);
    }
    return dd;
}

// Leapfrog_continuity.f90:51-68 (with the density_thresholds clamp) and
// EoS_fluid_loop.f90:59-70.  RK1: the density is integrated after the
// velocities and positions (Euler.f90:231-241, in vsmooth_end).
__device__ __forceinline__ void continuity_end(DPC& P, int i, double2 rpi, double dden, double dt, bool eos,
                                               double* __restrict__ dden_out, double2* __restrict__ rp_out,
                                               float* __restrict__ dr_out) {
    dden_out[i] = dden;
    if (P.rk1) return;
    double rho1 = rpi.x + dt * dden;
    if (P.dthr) {  // Leapfrog_continuity.f90:61-68
        if (rho1 < 0.9 * P.den0) rho1 = 0.9 * P.den0;
        if (rho1 > 1.1 * P.den0) rho1 = 1.1 * P.den0;
    }
    const double p1 = eos ? P.eps / P.den0 * (rho1 - P.den0) + P.prif : rpi.y;
    rp_out[i] = make_double2(rho1, p1);
    if (P.f32) dr_out[i] = (float)(rho1 - P.den0);
}

// the wall part of PressureSmoothing_3D.f90 / _2D.f90 and the update of p and rho;
// returns the new rho
__device__ __forceinline__ double psmooth_end(DPC& P, const DFace* __restrict__ faces,
                                              const int* __restrict__ bn, const BTab* __restrict__ bt, int i,
                                              int nsp, double2 rpi, double tp1, double somp, double app,
                                              double* __restrict__ vpres_out, double2* __restrict__ rp_out) {
    const double p0i = P.prif, pi = rpi.y;
    double diffp = 0.0;
    if (nsp > 0) {
    const int ncbf = P.semi ? bn[i] : 0;
    if (P.dim == 2) {
        // PressureSmoothing_2D.f90:124-214, SmoothVersion "b", fixe/tapi
        // sides; vpres is the smoothed pressure itself
        double VFT = 0.0;
        for (int q = 0; q < ncbf; ++q) {
            const BTab& B = bt[(size_t)q * P.cap + i];
            const DFace& S = faces[B.face];
            if (S.btype != 0 && S.btype != 1) continue;
            const double mf0 = S.T[0] * P.grav[0] + S.T[2] * P.grav[2];
            const double mf1 = S.T[6] * P.grav[0] + S.T[8] * P.grav[2];
            VFT = VFT + B.bi[1];
            somp = somp + P.den0 * (mf0 * B.bi[3] + mf1 * B.bi[4]);
        }
        app = app + VFT + 0.0 + 0.0 + 0.0;
        const double pz = (pi - pi) * 0.0;
        diffp = pi + tp1 * (somp + pz + pz + (p0i - pi) * (1.0 - app));
    } else {
        for (int q = 0; q < ncbf; ++q) {
            const BTab& B = bt[(size_t)q * P.cap + i];
            if (B.loc[2] > 0.0) app = app + B.bi[1];
        }
        if (P.dbsph) diffp = somp / app;  // PressureSmoothing_3D.f90:110-112
        else if (app < 0.95) diffp = somp + (p0i - pi) * (1.0 - app);
        else diffp = somp / app;
    }
    } else if (P.dim == 2) {
        diffp = rpi.y;  // no list (never: self is listed): pressure unchanged
    }
    vpres_out[i] = diffp;
    double p2 = rpi.y, rho2 = rpi.x;
    if (P.dim == 2) {  // PressureSmoothing_2D.f90:217-231: p = vpres, rho = EoS^-1(p)
        if (P.tetap > 0.0) {
            p2 = diffp;
            rho2 = P.den0 * (1.0 + (p2 - P.prif) / P.eps);
        }
    } else if (P.tetap > 0.0) {
        p2 = rpi.y + tp1 * diffp;
        rho2 = P.den0 * (1.0 + (p2 - P.prif) / P.eps);
    }
    rp_out[i] = make_double2(rho2, p2);
    return rho2;
}

// ----------------------------------------------------------------------------
// The four passes in FP64, one workgroup per tile: as the FP32-mixed ones
// below, with FP64 records (48 to 64 bytes a slot, so the largest tiles leave
// one workgroup of eight wavefronts a CU).  The expressions are the
// reference's, operation for operation, and every sum is formed in list order.
// They were bound by their gathers, five 16-byte loads a neighbour from records
// of three cell planes, more than an XCD's L2 (0.9-1.9 GB a launch from HBM);
// now by FP64 issue (measured: an operation every 4.9-5.7 cycles of a SIMD, a
// reciprocal or root 16.5), so the quotients share reciprocals and nothing
// branches on a pair.  576,000 particles: momentum 499 -> 448 us, velocity
// smoothing 595 -> 203, continuity 527 -> 206, pressure smoothing 315 -> 170;
// 72,000: 102 -> 80, 58 -> 38, 58 -> 37, 46 -> 31.  Twice the wavefronts (two
// lanes a particle, 1024 threads) measured the same, reading a neighbour's
// records ahead of the previous one's arithmetic 1% slower.
// Tiles that do not fit, solves of several masses, and lists that carry stencil
// codes (DB-SPH walls) gather from global memory with the same expressions;
// choose_form takes such solves off the tiles (CAP TILE_CAP_0).
// ----------------------------------------------------------------------------
#define TILE_ARGS Seg S, Tiles T, const int* __restrict__ start

// Adds particle i's NS pair terms to sum in list order, by G lanes (lane g of
// them; LDS form: 1, 2 or 4): each lane forms the terms of two entries, the lanes' entries
// consecutive, and lane 0 adds them all in order.  lds(byte offset of a
// neighbour's 16-byte records) and glob(its sorted index) read a neighbour,
// term(terms, one, other, one counts, other counts).  Past the list's end they
// are given the particle itself (`self`, i), whose differences vanish: a term
// that is a multiple of one is then a zero and leaves the sum as it is.
template <int G, int NS, class Lds, class Glob, class Term>
__device__ __forceinline__ void pair_sums64(const uint32_t* __restrict__ nbr, size_t N, int i, int nn, int g,
                                            bool fits, uint32_t self, double (&sum)[NS], Lds&& lds, Glob&& glob,
                                            Term&& term) {
    auto add = [&](const d2 (&t)[NS]) {
        double v[NS];
#pragma unroll
        for (int c = 0; c < NS; ++c) v[c] = t[c].x;
        add_lanes<G>(sum, v);
#pragma unroll
        for (int c = 0; c < NS; ++c) v[c] = t[c].y;
        add_lanes<G>(sum, v);
    };
    if (fits) {
        const uint4* L = reinterpret_cast<const uint4*>(nbr) + 2 * (size_t)i;
        uint4 next = *L;
        for (int k0 = 0; k0 < nn; k0 += 8) {
            const uint4 cur = next;
            L += (k0 & 8) ? 2 * N - 1 : (size_t)1;
            if (k0 + 8 < nn) next = *L;
            const uint32_t w[4] = {cur.x, cur.y, cur.z, cur.w};
            auto slot = [&](int u) {  // this lane's of the G entries from u on
                uint32_t o = w[u >> 1];
                if constexpr (G == 4) {
                    const uint32_t o2 = w[(u >> 1) + 1];
                    o = g & 2 ? o2 : o;
                }
                o = (G == 1 ? u & 1 : g & 1) ? o >> 16 : o & 0xFFFFu;
                return k0 + u + g < nn ? o : self;
            };
#pragma unroll
            for (int u = 0; u < 8; u += 2 * G) {
                __builtin_amdgcn_sched_barrier(0);
                d2 t[NS];
                term(t, lds(slot(u)), lds(slot(u + G)), k0 + u + g < nn, k0 + u + G + g < nn);
                add(t);
            }
        }
    } else {
        // a step's records are gathered during the step before it, and their
        // list entries a step earlier
        auto entry = [&](int k) { return k < nn ? (int)(nbr[nb_index(N, i, k)] & NB_MASK) : i; };
        int ja = entry(g), jb = entry(G + g);
        auto a = glob(ja), b = glob(jb);
        ja = entry(2 * G + g);
        jb = entry(3 * G + g);
        for (int k0 = 0; k0 < nn; k0 += 2 * G) {
            const auto ca = a, cb = b;
            a = glob(ja);
            b = glob(jb);
            ja = entry(k0 + 4 * G + g);
            jb = entry(k0 + 5 * G + g);
            d2 t[NS];
            term(t, ca, cb, k0 + g < nn, k0 + G + g < nn);
            add(t);
        }
    }
}

// 16 bytes at byte offset o of an LDS array, 8 bytes of the slot at offset o
__device__ __forceinline__ double2 lds16(const double2* a, uint32_t o) {
    return *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(a) + o);
}
__device__ __forceinline__ double lds8(const double* a, uint32_t o) {
    return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(a) + (o >> 1));
}

struct Nb { double x, y, z, u, v, w, rho, p, inv, m; };  // a neighbour, as far as a pass needs it

// momentum: RHS_momentum_equation.f90:72-179, inter_EqMoto.f90:108-283,
// viscomon.f90:54-71, viscomorris.f90:60-71
template <int CAP, bool SG, int G>
__global__ __launch_bounds__(TILE_WG, 2) void k_momentum64(
    TILE_ARGS, const DFace* __restrict__ faces, const DEdge* __restrict__ edges,
    const int* __restrict__ bn, const BTab* __restrict__ bt, const double4* __restrict__ xm,
    const double4* __restrict__ vel, const double2* __restrict__ rp, const int* __restrict__ lam_in,
    int* __restrict__ lam_out, const uint32_t* __restrict__ nbr, const int* __restrict__ nnb,
    double4* __restrict__ acc_out, double4* __restrict__ vel_out, const double* scal0, int* iscal0) {
    __shared__ double2 sA[CAP], sB[CAP], sC[CAP], sD[CAP];  // (x, y), (z, vx), (vy, vz), (rho, p)
    const int g = threadIdx.x % G;
    for_tiles<SG, G, 3, CAP != TILE_CAP_0>(S, T, start,
        [&](DPC&, int, int j, int slot) {
            const double4 x = xm[j], v = vel[j];
            sA[slot] = make_double2(x.x, x.y);
            sB[slot] = make_double2(x.z, v.x);
            sC[slot] = make_double2(v.y, v.z);
            sD[slot] = rp[j];
        },
        [&](DPC& P, int sg, int i, int slot, bool fits) {
            const double* scal = scal0 + sg * SC_COUNT;
            const double h = P.h;
            const double4 vi = vel[i];  // var == vel here
            const double2 rpi = rp[i];
            double tp[3] = {0.0, 0.0, 0.0};
            // sums: td, tv (from the wall terms on), rvs, tpa, ale
            double s[15];
            for (int c = 0; c < 15; ++c) s[c] = 0.0;
            const int ncbf = P.semi ? bn[i] : 0;
            const double v_i[3] = {vi.x, vi.y, vi.z};
            if (ncbf > 0) {
                double td[3] = {0.0, 0.0, 0.0}, tv[3] = {0.0, 0.0, 0.0};
                if (P.dim == 2)
                    sa_momentum_2d(P, faces, bt, i, ncbf, v_i, rpi, lam_in[i], tp, td, tv);
                else
                    sa_momentum(P, faces, bt, i, ncbf, v_i, rpi, lam_in[i], tp, td, tv, iscal0 + sg * IS_COUNT);
                for (int c = 0; c < 3; ++c) {
                    s[c] = td[c];
                    s[3 + c] = tv[c];
                }
            }
            const double4 xi = xm[i];
            const double rhoi = rpi.x, pi = rpi.y;
            const double celt = P.celerita + P.celerita;
            const double nui = P.kin_visc, nuj = P.kin_visc;
            const bool morris = nui > 1.0e-12 && nuj > 1.0e-12;
            const d2 invi = inv64(d2(rhoi));
            pair_sums64<G, 15>(nbr, (size_t)P.cap, i, nnb[i], g, fits, (uint32_t)slot << 4, s,
                [&](uint32_t o) {
                    const double2 a = lds16(sA, o), b = lds16(sB, o), c = lds16(sC, o), d = lds16(sD, o);
                    return Nb{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y, 0.0, xi.w};
                },
                [&](int j) {
                    const double4 x = xm[j], v = vel[j];
                    const double2 q = rp[j];
                    return Nb{x.x, x.y, x.z, v.x, v.y, v.z, q.x, q.y, 0.0, x.w};
                },
                [&](d2 (&t)[15], const Nb& a, const Nb& b, bool, bool) {
                    const d2 R0 = xi.x - d2{a.x, b.x}, R1 = xi.y - d2{a.y, b.y}, R2 = xi.z - d2{a.z, b.z};
                    const d2 rij = R0 * R0 + R1 * R1 + R2 * R2;
                    const K64x2 K = kvals64x2(P, rij, true, true, false);
                    const d2 dv0 = d2{a.u, b.u} - vi.x, dv1 = d2{a.v, b.v} - vi.y, dv2 = d2{a.w, b.w} - vi.z;
                    const d2 rhoj = {a.rho, b.rho}, pj = {a.p, b.p}, amassj = {a.m, b.m};
                    const d2 rr = rhoi * rhoj;
                    const d2 inv = inv64(rr), invj = newton64(rhoj, inv * rhoi);
                    d2 alpha = div64(pj - pi, rr, inv);
                    t[9] = -amassj * alpha * R0 * K.K3;
                    t[10] = -amassj * alpha * R1 * K.K3;
                    t[11] = -amassj * alpha * R2 * K.K3;
                    alpha = div64(pi * (div64(rhoj, d2(rhoi), invi) + 1.0) + pj * (div64(d2(rhoi), rhoj, invj) - 1.0), rr,
                                  inv);
                    t[12] = -(amassj * alpha * R0 * K.K3);
                    t[13] = -(amassj * alpha * R1 * K.K3);
                    t[14] = -(amassj * alpha * R2 * K.K3);
                    const d2 vrij = -dv0 * R0 - dv1 * R1 - dv2 * R2;
                    const d2 rsum = rhoi + rhoj;
                    const d2 TermMon = div64(d2(P.alfamon * celt * h), rsum, inv64(rsum));
                    t[0] = amassj * TermMon * vrij * R0 * K.K2;
                    t[1] = amassj * TermMon * vrij * R1 * K.K2;
                    t[2] = amassj * TermMon * vrij * R2 * K.K2;
                    // no branch: the compiler would keep the entries' values across it
                    const d2 rtil = nui * rhoi + nuj * rhoj + 1.0e-3;
                    const double atil = 4.0 * (nui * nuj);
                    const d2 visc = div64(amassj * atil, rtil, inv64(rtil));
                    const d2 fac = {morris ? visc.x : 0.0, morris ? visc.y : 0.0};
                    t[3] = t[6] = fac * (-dv0 * K.K2 * rij);
                    t[4] = t[7] = fac * (-dv1 * K.K2 * rij);
                    t[5] = t[8] = fac * (-dv2 * K.K2 * rij);
                });
            if (g) return;
            for (int d = 0; d < 3; ++d) tp[d] = tp[d] + s[9 + d] + s[12 + d];
            double br[3] = {0.0, 0.0, 0.0};
            if (ncbf > 0) elastic_walls(P, faces, edges, bt, xm, i, ncbf, vi, br);
            // Leapfrog_momentum.f90:66-86 integrates with dtvel; the explicit RK1
            // branch (Euler.f90:85-93) with dt
            momentum_end(P, i, ncbf, vi, P.rk1 ? scal[SC_DT] : scal[SC_DTVEL], tp, s, s + 3, s + 6, br, lam_out,
                         acc_out, vel_out);
        },
        [](DPC&, int) {});
}

// velocity smoothing: velocity_smoothing.f90:74-133
template <int CAP, bool SG, int G>
__global__ __launch_bounds__(TILE_WG, 2) void k_vsmooth64(
    TILE_ARGS, const DFace* __restrict__ faces, const int* __restrict__ bn, const BTab* __restrict__ bt,
    const double4* __restrict__ xm, const double4* __restrict__ vel1, const double2* __restrict__ rp,
    const uint32_t* __restrict__ nbr, const int* __restrict__ nnb, double4* __restrict__ vel_out,
    double4* __restrict__ xm_out, const double* scal0, unsigned long long* dtmin, const int* iscal0,
    const double* __restrict__ dden_in, double2* __restrict__ rp_out, int* __restrict__ gone) {
    __shared__ double2 sA[CAP], sB[CAP], sC[CAP], sD[CAP];  // (x, y), (z, vx), (vy, vz), (rho, 1 / rho)
    const int g = threadIdx.x % G;
    unsigned long long dtbits = 0x7FF0000000000000ull;
    for_tiles<SG, G, 3, CAP != TILE_CAP_0>(S, T, start,
        [&](DPC& P, int, int j, int slot) {
            if (!(P.tetav > 1.0e-9)) return;
            const double4 x = xm[j], v = vel1[j];
            sA[slot] = make_double2(x.x, x.y);
            sB[slot] = make_double2(x.z, v.x);
            sC[slot] = make_double2(v.y, v.z);
            const double rho = rp[j].x;
            sD[slot] = make_double2(rho, 1.0 / rho);
        },
        [&](DPC& P, int sg, int i, int slot, bool fits) {
            const double* scal = scal0 + sg * SC_COUNT;
            const bool smooth = P.tetav > 1.0e-9;
            const double4 xi = xm[i];
            const double4 vi = vel1[i];
            double v[3] = {0.0, 0.0, 0.0};
            if (smooth) {
                pair_sums64<G, 3>(nbr, (size_t)P.cap, i, nnb[i], g, fits, (uint32_t)slot << 4, v,
                    [&](uint32_t o) {
                        const double2 a = lds16(sA, o), b = lds16(sB, o), c = lds16(sC, o), d = lds16(sD, o);
                        return Nb{a.x, a.y, b.x, b.y, c.x, c.y, d.x, 0.0, d.y, xi.w};
                    },
                    [&](int j) {
                        const double4 x = xm[j], u = vel1[j];
                        const double rho = rp[j].x;
                        return Nb{x.x, x.y, x.z, u.x, u.y, u.z, rho, 0.0, 0.0, x.w};
                    },
                    [&](d2 (&t)[3], const Nb& a, const Nb& b, bool, bool) {
                        const d2 R0 = xi.x - d2{a.x, b.x}, R1 = xi.y - d2{a.y, b.y}, R2 = xi.z - d2{a.z, b.z};
                        const K64x2 K = kvals64x2(P, R0 * R0 + R1 * R1 + R2 * R2, false, false, true);
                        const d2 rhoj = {a.rho, b.rho};
                        const d2 pes = div64(d2{a.m, b.m} * K.W, rhoj, fits ? d2{a.inv, b.inv} : inv64(rhoj));
                        t[0] = (d2{a.u, b.u} - vi.x) * pes;
                        t[1] = (d2{a.v, b.v} - vi.y) * pes;
                        t[2] = (d2{a.w, b.w} - vi.z) * pes;
                    });
            }
            if (g) return;
            if (smooth) vsmooth_walls(P, faces, bt, i, P.semi ? bn[i] : 0, vi, v);
            const unsigned long long b =
                vsmooth_end<false>(P, faces, i, xi, vi, v, smooth, scal[SC_TV1], scal[SC_DT],
                                   iscal0[sg * IS_COUNT + IS_ONGOING] > 0, dden_in, rp, vel_out, xm_out, rp_out,
                                   nullptr, gone);
            dtbits = b < dtbits ? b : dtbits;
        },
        [&](DPC&, int sg) { wave_min_to(dtbits, dtmin + sg); });
}

// continuity: SASPH_continuity.f90:89-169, Continuity_Equation.f90:97-235
template <int CAP, bool SG, int G>
__global__ __launch_bounds__(TILE_WG, 2) void k_continuity64(
    TILE_ARGS, const DFace* __restrict__ faces, const int* __restrict__ bn, const BTab* __restrict__ bt,
    const double4* __restrict__ xm, const double4* __restrict__ vel, const double2* __restrict__ rp,
    const uint32_t* __restrict__ nbr, const int* __restrict__ nnb, double* __restrict__ dden_out,
    double2* __restrict__ rp_out, const double* scal0, int* iscal0) {
    __shared__ double2 sA[CAP], sB[CAP], sC[CAP];  // (x, y), (z, vx), (vy, vz)
    __shared__ double sD[CAP];                     // m / rho
    const int g = threadIdx.x % G;
    for_tiles<SG, G, 3, CAP != TILE_CAP_0>(S, T, start,
        [&](DPC&, int, int j, int slot) {
            const double4 x = xm[j], v = vel[j];
            sA[slot] = make_double2(x.x, x.y);
            sB[slot] = make_double2(x.z, v.x);
            sC[slot] = make_double2(v.y, v.z);
            sD[slot] = x.w / rp[j].x;
        },
        [&](DPC& P, int sg, int i, int slot, bool fits) {
            const double4 xi = xm[i];
            const double4 vi = vel[i];
            const double2 rpi = rp[i];
            const double rhoi = rpi.x;
            double s[3] = {0.0, 0.0, 0.0};
            pair_sums64<G, 3>(nbr, (size_t)P.cap, i, nnb[i], g, fits, (uint32_t)slot << 4, s,
                [&](uint32_t o) {
                    const double2 a = lds16(sA, o), b = lds16(sB, o), c = lds16(sC, o);
                    return Nb{a.x, a.y, b.x, b.y, c.x, c.y, 0.0, 0.0, 0.0, lds8(sD, o)};
                },
                [&](int j) {
                    const double4 x = xm[j], v = vel[j];
                    return Nb{x.x, x.y, x.z, v.x, v.y, v.z, 0.0, 0.0, 0.0, x.w / rp[j].x};
                },
                [&](d2 (&t)[3], const Nb& a, const Nb& b, bool, bool) {  // m: the neighbour's volume
                    const d2 R0 = xi.x - d2{a.x, b.x}, R1 = xi.y - d2{a.y, b.y}, R2 = xi.z - d2{a.z, b.z};
                    const K64x2 K = kvals64x2(P, R0 * R0 + R1 * R1 + R2 * R2, true, false, false);
                    const d2 f = rhoi * d2{a.m, b.m} * K.K1;
                    t[0] = f * (d2{a.u, b.u} - vi.x) * R0;
                    t[1] = f * (d2{a.v, b.v} - vi.y) * R1;
                    t[2] = f * (d2{a.w, b.w} - vi.z) * R2;
                });
            if (g) return;
            int* iscal = iscal0 + sg * IS_COUNT;
            const double dd = continuity_walls(P, faces, bt, i, P.semi ? bn[i] : 0, vi, rhoi, iscal);
            const double inner = s[0] + s[1] + s[2];
            continuity_end(P, i, rpi, dd - inner, scal0[sg * SC_COUNT + SC_DT], iscal[IS_ONGOING] > 0, dden_out,
                           rp_out, nullptr);
        },
        [](DPC&, int) {});
}

// pressure smoothing: PressureSmoothing_3D.f90:80-161 (both loops)
template <int CAP, bool SG, int G>
__global__ __launch_bounds__(TILE_WG, 2) void k_psmooth64(
    TILE_ARGS, const DFace* __restrict__ faces, const int* __restrict__ bn, const BTab* __restrict__ bt,
    const double4* __restrict__ xm, const double2* __restrict__ rp, const uint32_t* __restrict__ nbr,
    const int* __restrict__ nnb, double* __restrict__ vpres_out, double2* __restrict__ rp_out,
    const double* scal0) {
    __shared__ double2 sA[CAP], sB[CAP], sC[CAP];  // (x, y), (z, p), (rho, 1 / rho)
    const int g = threadIdx.x % G;
    for_tiles<SG, G, 3, CAP != TILE_CAP_0>(S, T, start,
        [&](DPC&, int, int j, int slot) {
            const double4 x = xm[j];
            const double2 q = rp[j];
            sA[slot] = make_double2(x.x, x.y);
            sB[slot] = make_double2(x.z, q.y);
            sC[slot] = make_double2(q.x, 1.0 / q.x);
        },
        [&](DPC& P, int sg, int i, int slot, bool fits) {
            const double4 xi = xm[i];
            const double2 rpi = rp[i];
            const int nsp = nnb[i];
            const double pi = rpi.y;
            double s[2] = {0.0, 0.0};
            pair_sums64<G, 2>(nbr, (size_t)P.cap, i, nsp, g, fits, (uint32_t)slot << 4, s,
                [&](uint32_t o) {
                    const double2 a = lds16(sA, o), b = lds16(sB, o), c = lds16(sC, o);
                    return Nb{a.x, a.y, b.x, 0.0, 0.0, 0.0, c.x, b.y, c.y, xi.w};
                },
                [&](int j) {
                    const double4 x = xm[j];
                    const double2 q = rp[j];
                    return Nb{x.x, x.y, x.z, 0.0, 0.0, 0.0, q.x, q.y, 0.0, x.w};
                },
                [&](d2 (&t)[2], const Nb& a, const Nb& b, bool ona, bool onb) {
                    const d2 R0 = xi.x - d2{a.x, b.x}, R1 = xi.y - d2{a.y, b.y}, R2 = xi.z - d2{a.z, b.z};
                    const K64x2 K = kvals64x2(P, R0 * R0 + R1 * R1 + R2 * R2, false, false, true);
                    const d2 rhoj = {a.rho, b.rho};
                    const d2 pes = div64(d2{a.m, b.m} * K.W, rhoj, fits ? d2{a.inv, b.inv} : inv64(rhoj));
                    t[0] = d2{ona ? pes.x : 0.0, onb ? pes.y : 0.0};
                    t[1] = (d2{a.p, b.p} - pi) * pes;
                });
            if (g) return;
            psmooth_end(P, faces, bn, bt, i, nsp, rpi, scal0[sg * SC_COUNT + SC_TP1], s[1], s[0], vpres_out, rp_out);
        },
        [](DPC&, int) {});
}

// ----------------------------------------------------------------------------
// The four passes in FP32-mixed form, one workgroup per tile (see Tiles): the
// records of the tile's particles and of the cells around it are staged in
// LDS once, with the parts of a pair's term that belong to the neighbour
// alone (m_j / rho_j, p_j / rho_j^2) computed there, and a lane walks its
// particle's list of LDS slots.  The passes were bound by their gathers: 64
// lanes reading 64 different lines take about 75 cycles of the CU's L1 per
// 16-byte load, 78 neighbours and one or two loads each; a 16-byte LDS gather
// takes about a quarter of it, and the pair sums' own instructions bound now.
// The tile is as large as two workgroups a CU allow (80 KB of LDS each: one
// stages while the other computes), smaller for small solves (choose_tile).
// Pair math on xq's integer positions: a separation is exact to 2^-28 of a
// cell, in units of P.lsb, whose powers are taken out of the sums.
// Tiles with more candidates than the LDS holds gather from global memory
// with the same expressions, so a sum does not depend on the tile.  Solves in
// which most do (choose_form) take no LDS and two lanes a particle, eight
// neighbours in flight each: a cluster of three times water, 81,000 particles,
// four passes: on tiles 1199 us (one neighbour in flight) and 582 (four), 270.
// 576,000 particles: momentum 186 -> 120 us, velocity smoothing 202 -> 87,
// continuity 185 -> 79, pressure smoothing 101 -> 55; 25,000 particles: 33 ->
// 28, 24 -> 17, 23 -> 16, 19 -> 13.
// ----------------------------------------------------------------------------
// q = r/h from a squared separation in lsb^2
struct PairR {
    float R0, R1, R2, rij, r;
};
__device__ __forceinline__ PairR pair_r(int4 a, float4 b) {
    PairR d;
    d.R0 = (float)lsb_diff(a.x, __float_as_int(b.x));
    d.R1 = (float)lsb_diff(a.y, __float_as_int(b.y));
    d.R2 = (float)lsb_diff(a.z, __float_as_int(b.z));
    d.rij = __builtin_fmaf(d.R0, d.R0, __builtin_fmaf(d.R1, d.R1, d.R2 * d.R2));
    d.r = __builtin_amdgcn_sqrtf(d.rij);
    return d;
}
// the spline over coefke, and its derivative times h over coefke
// (CalcVarLength.f90:243-265); every listed pair has r <= 2h, where both
// branches vanish, so no cut-off test is needed
__device__ __forceinline__ float spline_w(float q) {
    const float b = 2.0f - q, q2 = q * q;
    const float in = __builtin_fmaf(q2, __builtin_fmaf(q, 0.5f, -1.0f), 0.666666667f);
    const float out = b * b * b * 0.166666666667f;
    return q >= 1.0f ? out : in;
}
__device__ __forceinline__ float spline_g(float q, float b2) {
    return q >= 1.0f ? -0.5f * b2 : q * __builtin_fmaf(1.5f, q, -2.0f);
}

__device__ __forceinline__ float4 bits4(int4 x, float w) {
    return make_float4(__int_as_float(x.x), __int_as_float(x.y), __int_as_float(x.z), w);
}

// The NS pair sums of particle i over its list, by G lanes (1 or 2, lane g of
// them).  The entries go by eights to two partial sums in turn, which are
// added at the end, so a sum is the same for both G: few particles take two
// lanes each (a lane's serial walk over 80 neighbours is then the time: 1,440
// particles, continuity 18 -> 14 us), many take one.  (Four partial sums: 12
// us there, but one lane holding 36 of them spilled: 116 -> 206 us for the
// momentum pass at 576,000.)
// fits: 16-bit entries (LDS slot times 16), 16 of them per 32 bytes, filled up
// with the particle itself to whole eights; lds(sums, byte offset of the
// neighbour's 16-byte record, place in the list).  Else term(sums, glob(sorted
// index), place), CH neighbours' records in flight, past the end the particle
// itself.  The next entries are loaded while some are used.
template <int G, int CH, int NS, class Lds, class Glob, class Term>
__device__ __forceinline__ void pair_sums(const uint32_t* __restrict__ nbr, size_t N, int i, int nn, int g,
                                          bool fits, float (&sum)[NS], Lds&& lds, Glob&& glob, Term&& term) {
#pragma unroll
    for (int c = 0; c < NS; ++c) sum[c] = 0.0f;
#pragma unroll 1
    for (int m = g; m < 2; m += G) {  // the partial sums of the lane, one walk each
        float a[NS];
#pragma unroll
        for (int c = 0; c < NS; ++c) a[c] = 0.0f;
        if (fits) {
            const uint4* L = reinterpret_cast<const uint4*>(nbr) + 2 * (size_t)i + m;
            uint4 next = *L;
            for (int k = 8 * m; k < nn; k += 16) {
                const uint4 cur = next;
                L += 2 * N;
                if (k + 16 < nn) next = *L;
                const uint32_t w[4] = {cur.x, cur.y, cur.z, cur.w};
#pragma unroll
                for (int u = 0; u < 8; ++u) lds(a, (u & 1) ? w[u >> 1] >> 16 : w[u >> 1] & 0xFFFFu, k + u);
            }
        } else if constexpr (CH == 1) {
            for (int k0 = 8 * m; k0 < nn; k0 += 16)
                for (int k = k0; k < min(nn, k0 + 8); ++k) term(a, glob((int)(nbr[nb_index(N, i, k)] & NB_MASK)), k);
        } else {
            const uint4* L = reinterpret_cast<const uint4*>(nbr) + 2 * ((size_t)m * N + (size_t)i);
            uint4 na = L[0], nb = L[1];
            for (int k0 = 8 * m; k0 < nn; k0 += 16) {
                const uint32_t w[8] = {na.x, na.y, na.z, na.w, nb.x, nb.y, nb.z, nb.w};
                L += 4 * N;
                if (k0 + 16 < nn) {
                    na = L[0];
                    nb = L[1];
                }
#pragma unroll
                for (int c = 0; c < 8; c += CH) {
                    decltype(glob(0)) r[CH];
#pragma unroll
                    for (int u = 0; u < CH; ++u) r[u] = glob(k0 + c + u < nn ? (int)(w[c + u] & NB_MASK) : i);
#pragma unroll
                    for (int u = 0; u < CH; ++u) term(a, r[u], k0 + c + u);
                }
            }
        }
#pragma unroll
        for (int c = 0; c < NS; ++c) sum[c] += a[c];
    }
    if constexpr (G == 2)
#pragma unroll
        for (int c = 0; c < NS; ++c) sum[c] += __shfl_xor(sum[c], 1, 64);
}

struct RecF { int4 x; float4 v; };  // a gathered neighbour
// neighbours in flight: the LDS form's registers leave room for fewer (the
// pressure smoothing's for one: four took its seventh wavefront, 56 -> 64 us)
constexpr int GATHER_CH(int cap) { return cap == TILE_CAP_0 ? 8 : 4; }

// momentum; UM: every particle of the context has its solve's mass
template <int CAP, bool SG, int G, bool UM>
__global__ __launch_bounds__(TILE_WG, 4) void k_momentum(
    TILE_ARGS, const DFace* __restrict__ faces, const DEdge* __restrict__ edges,
    const int* __restrict__ bn, const BTab* __restrict__ bt, const double4* __restrict__ xm,
    const double4* __restrict__ vel, const double2* __restrict__ rp, const int4* __restrict__ xq,
    const float4* __restrict__ vf, const int* __restrict__ lam_in, int* __restrict__ lam_out,
    const uint32_t* __restrict__ nbr, const int* __restrict__ nnb, double4* __restrict__ acc_out,
    double4* __restrict__ vel_out, float4* __restrict__ vf_out, const double* scal0, int* iscal0) {
    __shared__ float4 sA[CAP], sB[CAP];
    // UM: (position, p_j / rho_j^2), (velocity, rho - den0); else (position, rho - den0), (velocity, mass)
    auto rec_a = [](DPC& P, int4 x, float4 v) {
        if constexpr (!UM) return bits4(x, v.w);
        const float rhoj = P.f_den0 + v.w, pj = __builtin_fmaf(P.f_eosk, v.w, P.f_prif);
        return bits4(x, pj * __builtin_amdgcn_rcpf(rhoj * rhoj));
    };
    auto rec_b = [](int4 x, float4 v) {
        return make_float4(v.x, v.y, v.z, UM ? v.w : __int_as_float(x.w));
    };
    for_tiles<SG, G, TILE_U, CAP != TILE_CAP_0>(S, T, start,
        [&](DPC& P, int, int j, int slot) {
            const int4 x = xq[j];
            const float4 v = vf[j];
            sA[slot] = rec_a(P, x, v);
            sB[slot] = rec_b(x, v);
        },
        [&](DPC& P, int sg, int i, int, bool fits) {
            const double* scal = scal0 + sg * SC_COUNT;
            const int4 xi = xq[i];
            const float4 vf_i = vf[i];
            const double2 rpi = rp[i];
            const float rhoi = (float)rpi.x;
            const float pri = (float)rpi.y * __builtin_amdgcn_rcpf(rhoi * rhoi);
            const float nu = P.f_kin_visc;
            // symmetric form -m_j (p_i/rho_i^2 + p_j/rho_j^2) r K3 of the
            // reference's difference term plus its ALE1 complement, with
            // K3 = -3 (2-q)^2 kacl / (r + eta); Monaghan's and Morris's terms
            // with K2 = g ke / ((r + eta)(r^2 + eta2)).  The particle itself
            // adds zeros.
            auto pair = [&](float* s, float4 A, float4 B) {
                const PairR d = pair_r(xi, A);
                const float q = d.r * P.f_q, b = 2.0f - q, b2 = b * b;
                const float e2 = d.rij + P.f_eta2l;
                const float D2 = __builtin_amdgcn_rcpf((d.r + P.f_etal) * e2);
                float k2 = spline_g(q, b2) * D2, k3 = b2 * (e2 * D2);
                float prj = A.w, drj = B.w;
                if constexpr (!UM) {
                    drj = A.w;
                    const float rhoj = P.f_den0 + drj, pj = __builtin_fmaf(P.f_eosk, drj, P.f_prif);
                    prj = pj * __builtin_amdgcn_rcpf(rhoj * rhoj);
                    k2 *= B.w;
                    k3 *= B.w;
                }
                const float cp = (pri + prj) * k3;
                s[0] = __builtin_fmaf(cp, d.R0, s[0]);
                s[1] = __builtin_fmaf(cp, d.R1, s[1]);
                s[2] = __builtin_fmaf(cp, d.R2, s[2]);
                const float v0 = B.x - vf_i.x, v1 = B.y - vf_i.y, v2 = B.z - vf_i.z;
                const float vr = __builtin_fmaf(v0, d.R0, __builtin_fmaf(v1, d.R1, v2 * d.R2));
                // 1 / (rho_i + rho_j) and 1 / (nu (rho_i + rho_j) + 1e-3) from one reciprocal
                const float t = rhoi + (P.f_den0 + drj), nt = __builtin_fmaf(nu, t, 1.0e-3f);
                const float Dm = __builtin_amdgcn_rcpf(t * nt);
                const float cd = Dm * nt * vr * k2;
                s[3] = __builtin_fmaf(cd, d.R0, s[3]);
                s[4] = __builtin_fmaf(cd, d.R1, s[4]);
                s[5] = __builtin_fmaf(cd, d.R2, s[5]);
                const float cv = Dm * t * (k2 * d.rij);
                s[6] = __builtin_fmaf(cv, v0, s[6]);
                s[7] = __builtin_fmaf(cv, v1, s[7]);
                s[8] = __builtin_fmaf(cv, v2, s[8]);
            };
            float s[9];
            pair_sums<G, GATHER_CH(CAP)>(nbr, (size_t)P.cap, i, nnb[i], threadIdx.x % G, fits, s,
                         [&](float* a, uint32_t o, int) { pair(a, lds16(sA, o), lds16(sB, o)); },
                         [&](int j) { return RecF{xq[j], vf[j]}; },
                         [&](float* a, const RecF& r, int) { pair(a, rec_a(P, r.x, r.v), rec_b(r.x, r.v)); });
            if (threadIdx.x % G) return;
            const double m = UM ? (double)P.f_mass : 1.0, ke = P.ke_coef * P.inv_lsb;
            const double sp = 3.0 * P.kacl_coef * m;
            const double sd = -(P.alfamon * (P.celerita + P.celerita) * P.h * m * ke);
            const double sv = P.kin_visc > 1.0e-12 ? -(4.0 * (P.kin_visc * P.kin_visc) * m * ke) : 0.0;
            // wall terms (AddBoundaryContributions_to_ME3D.f90), then the sums
            const double4 vi = vel[i];  // var == vel here
            const int ncbf = P.semi ? bn[i] : 0;
            Walls6 W = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
            Walls3 E = {{0.0, 0.0, 0.0}};
            if (ncbf > 0) {
                W = wall_terms(&P, faces, bt, i, ncbf, vi.x, vi.y, vi.z, rpi.x, rpi.y, lam_in[i], iscal0 + sg * IS_COUNT);
                E = wall_elastic(&P, faces, edges, bt, xm, i, ncbf, vi.x, vi.y, vi.z);
            }
            const double rvs[3] = {sv * (double)s[6], sv * (double)s[7], sv * (double)s[8]};
            const double tp[3] = {W.tp[0] + sp * (double)s[0], W.tp[1] + sp * (double)s[1], W.tp[2] + sp * (double)s[2]};
            const double td[3] = {W.tdv[0] + sd * (double)s[3], W.tdv[1] + sd * (double)s[4], W.tdv[2] + sd * (double)s[5]};
            const double dtvel = P.rk1 ? scal[SC_DT] : scal[SC_DTVEL];
            const double4 vn = momentum_end(P, i, ncbf, vi, dtvel, tp, td, rvs, rvs, E.r, lam_out, acc_out, vel_out);
            vf_out[i] = make_float4((float)vn.x, (float)vn.y, (float)vn.z, (float)(rpi.x - P.den0));
        },
        [](DPC&, int) {});
}

// velocity smoothing
template <int CAP, bool SG, int G>
__global__ __launch_bounds__(TILE_WG, 4) void k_vsmooth(
    TILE_ARGS, const DFace* __restrict__ faces, const int* __restrict__ bn, const BTab* __restrict__ bt,
    const double4* __restrict__ xm, const double4* __restrict__ vel1, const double2* __restrict__ rp,
    const int4* __restrict__ xq, const float4* __restrict__ vf, const uint32_t* __restrict__ nbr,
    const int* __restrict__ nnb, double4* __restrict__ vel_out, double4* __restrict__ xm_out,
    const double* scal0, unsigned long long* dtmin, const int* iscal0, const double* __restrict__ dden_in,
    double2* __restrict__ rp_out, float* __restrict__ dr_out, int* __restrict__ gone) {
    __shared__ float4 sA[CAP], sB[CAP];  // (position, m_j / rho_j), velocity
    auto rec_a = [](DPC& P, int4 x, float4 v) {
        return bits4(x, __int_as_float(x.w) * __builtin_amdgcn_rcpf(P.f_den0 + v.w));
    };
    unsigned long long dtbits = 0x7FF0000000000000ull;
    for_tiles<SG, G, TILE_U, CAP != TILE_CAP_0>(S, T, start,
        [&](DPC& P, int, int j, int slot) {
            if (!(P.tetav > 1.0e-9)) return;
            const float4 v = vf[j];
            sA[slot] = rec_a(P, xq[j], v);
            sB[slot] = v;
        },
        [&](DPC& P, int sg, int i, int, bool fits) {
            const double* scal = scal0 + sg * SC_COUNT;
            const bool smooth = P.tetav > 1.0e-9;
            double v[3] = {0.0, 0.0, 0.0};
            if (smooth) {
                const int4 xi = xq[i];
                const float4 vi = vf[i];
                auto pair = [&](float* s, float4 A, float4 B) {
                    const PairR d = pair_r(xi, A);
                    const float pes = A.w * spline_w(d.r * P.f_q);
                    s[0] = __builtin_fmaf(B.x - vi.x, pes, s[0]);
                    s[1] = __builtin_fmaf(B.y - vi.y, pes, s[1]);
                    s[2] = __builtin_fmaf(B.z - vi.z, pes, s[2]);
                };
                float s[3];
                pair_sums<G, GATHER_CH(CAP)>(nbr, (size_t)P.cap, i, nnb[i], threadIdx.x % G, fits, s,
                             [&](float* a, uint32_t o, int) { pair(a, lds16(sA, o), lds16(sB, o)); },
                             [&](int j) { return RecF{xq[j], vf[j]}; },
                             [&](float* a, const RecF& r, int) { pair(a, rec_a(P, r.x, r.v), r.v); });
                v[0] = P.coefke * (double)s[0];
                v[1] = P.coefke * (double)s[1];
                v[2] = P.coefke * (double)s[2];
            }
            if (threadIdx.x % G) return;
            const double4 vi = vel1[i];
            const int ncbf = smooth && P.semi ? bn[i] : 0;
            if (ncbf > 0) {
                const Walls3 W = wall_smooth(&P, faces, bt, i, ncbf, vi.x, vi.y, vi.z, v[0], v[1], v[2]);
                for (int d = 0; d < 3; ++d) v[d] = W.r[d];
            }
            const unsigned long long b =
                vsmooth_end<true>(P, faces, i, xm[i], vi, v, smooth, scal[SC_TV1], scal[SC_DT],
                            iscal0[sg * IS_COUNT + IS_ONGOING] > 0, dden_in, rp, vel_out, xm_out, rp_out,
                            dr_out, gone);
            dtbits = b < dtbits ? b : dtbits;
        },
        [&](DPC&, int sg) { wave_min_to(dtbits, dtmin + sg); });
}

// continuity
template <int CAP, bool SG, int G>
__global__ __launch_bounds__(TILE_WG, 4) void k_continuity(
    TILE_ARGS, const DFace* __restrict__ faces, const int* __restrict__ bn, const BTab* __restrict__ bt,
    const double4* __restrict__ vel, const double2* __restrict__ rp, const int4* __restrict__ xq,
    const float4* __restrict__ vf, const uint32_t* __restrict__ nbr, const int* __restrict__ nnb,
    double* __restrict__ dden_out, double2* __restrict__ rp_out, float* __restrict__ dr_out,
    const double* scal0, int* iscal0) {
    __shared__ float4 sA[CAP], sB[CAP];  // (position, m_j / rho_j), velocity
    auto rec_a = [](DPC& P, int4 x, float4 v) {
        return bits4(x, __int_as_float(x.w) * __builtin_amdgcn_rcpf(P.f_den0 + v.w));
    };
    for_tiles<SG, G, TILE_U, CAP != TILE_CAP_0>(S, T, start,
        [&](DPC& P, int, int j, int slot) {
            const float4 v = vf[j];
            sA[slot] = rec_a(P, xq[j], v);
            sB[slot] = v;
        },
        [&](DPC& P, int sg, int i, int, bool fits) {
            const int4 xi = xq[i];
            const float4 vi = vf[i];
            auto pair = [&](float* s, float4 A, float4 B) {
                const PairR d = pair_r(xi, A);
                const float q = d.r * P.f_q, b = 2.0f - q;
                const float k = A.w * spline_g(q, b * b) * __builtin_amdgcn_rcpf(d.r + P.f_etal);
                const float dv = __builtin_fmaf(B.x - vi.x, d.R0, __builtin_fmaf(B.y - vi.y, d.R1, (B.z - vi.z) * d.R2));
                s[0] = __builtin_fmaf(k, dv, s[0]);
            };
            float s[1];
            pair_sums<G, GATHER_CH(CAP)>(nbr, (size_t)P.cap, i, nnb[i], threadIdx.x % G, fits, s,
                         [&](float* a, uint32_t o, int) { pair(a, lds16(sA, o), lds16(sB, o)); },
                         [&](int j) { return RecF{xq[j], vf[j]}; },
                         [&](float* a, const RecF& r, int) { pair(a, rec_a(P, r.x, r.v), r.v); });
            if (threadIdx.x % G) return;
            const double2 rpi = rp[i];
            int* iscal = iscal0 + sg * IS_COUNT;
            const double dd = continuity_walls(P, faces, bt, i, P.semi ? bn[i] : 0, vel[i], rpi.x, iscal);
            const double inner = rpi.x * (P.ke_coef * (double)s[0]);
            continuity_end(P, i, rpi, dd - inner, scal0[sg * SC_COUNT + SC_DT], iscal[IS_ONGOING] > 0, dden_out,
                           rp_out, dr_out);
        },
        [](DPC&, int) {});
}

// pressure smoothing; p_j - p_i is the linear EoS of the density difference
template <int CAP, bool SG, int G>
__global__ __launch_bounds__(TILE_WG, 4) void k_psmooth(
    TILE_ARGS, const DFace* __restrict__ faces, const int* __restrict__ bn, const BTab* __restrict__ bt,
    const double2* __restrict__ rp, const int4* __restrict__ xq, const float* __restrict__ dr,
    const uint32_t* __restrict__ nbr, const int* __restrict__ nnb, double* __restrict__ vpres_out,
    double2* __restrict__ rp_out, float4* __restrict__ vf_out, const double* scal0) {
    __shared__ float4 sA[CAP];  // (position, m_j / rho_j)
    __shared__ float sD[CAP];   // rho_j - den0
    auto rec_a = [](DPC& P, int4 x, float d) {
        return bits4(x, __int_as_float(x.w) * __builtin_amdgcn_rcpf(P.f_den0 + d));
    };
    for_tiles<SG, G, TILE_U, CAP != TILE_CAP_0>(S, T, start,
        [&](DPC& P, int, int j, int slot) {
            const float d = dr[j];
            sA[slot] = rec_a(P, xq[j], d);
            sD[slot] = d;
        },
        [&](DPC& P, int sg, int i, int, bool fits) {
            const int4 xi = xq[i];
            const float di = dr[i];
            const int nn = nnb[i];
            auto pair = [&](float* s, float4 A, float dj, bool in) {
                const PairR d = pair_r(xi, A);
                const float pes = in ? A.w * spline_w(d.r * P.f_q) : 0.0f;
                s[0] += pes;
                s[1] = __builtin_fmaf(dj - di, pes, s[1]);
            };
            float s[2];
            struct RecD { int4 x; float d; };
            pair_sums<G, CAP == TILE_CAP_0 ? 8 : 1>(nbr, (size_t)P.cap, i, nn, threadIdx.x % G, fits, s,
                         [&](float* a, uint32_t o, int k) {
                             const float dj = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(sD) + (o >> 2));
                             pair(a, lds16(sA, o), dj, k < nn);
                         },
                         [&](int j) { return RecD{xq[j], dr[j]}; },
                         [&](float* a, const RecD& r, int k) { pair(a, rec_a(P, r.x, r.d), r.d, k < nn); });
            if (threadIdx.x % G) return;
            const double rho2 = psmooth_end(P, faces, bn, bt, i, nn, rp[i], scal0[sg * SC_COUNT + SC_TP1],
                                            P.eps / P.den0 * P.coefke * (double)s[1], P.coefke * (double)s[0],
                                            vpres_out, rp_out);
            // the density slot of the velocity record the next momentum pass reads
            reinterpret_cast<float*>(vf_out + i)[3] = (float)(rho2 - P.den0);
        },
        [](DPC&, int) {});
}

}  // namespace sph
