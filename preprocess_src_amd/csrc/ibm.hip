// Immersed-boundary coupling on gfx950.
//
// Spreading: ibm_st1 = ibm_st1a (zero) + ibm_st1b (4x4x4 cosine-delta
// spread) + ibm_st1c (fold of halo contributions onto periodic images)
// (ibm.cu:27-131, 214-369).  Interpolation + advection: ibm_st2a
// (ibm.cu:372-639).
//
// The stencil of a vertex is selected exactly as the reference does in its
// padded frame (xtr = X + (nx_p-1) dx/2, first node floor(xtr/dx)-1, nodes at
// ix_p*dx) and then mapped to the unpadded lattice by ix = ix_p - 2 with
// periodic wrapping, which is what the halo fold achieves; nodes beyond the
// walls are dropped (spread) or contribute zero velocity (interpolation).
// Vertex positions and stencil selection are FP64 in every precision mode;
// weights, lattice fields (u, F) and nodal forces use the arithmetic type T.
//
// Both directions work on lattice tiles of 8x8x8 nodes (16x8x8 left a third of
// the CUs idle on a few dozen cells, and its boxes let one or two work groups
// share a CU where these let three).  After each change
// of the positions the vertices are binned by the tile of their first stencil
// node (counting sort, counters combined per work group).
//   - Spreading: one work group per tile takes the vertices of its own bin
//     and of its 7 lower neighbours, keeps those whose stencil meets the tile
//     (per-wave queue), and accumulates their contributions into the tile in
//     LDS, one lane per vertex, with 64-bit integer LDS atomics on fixed-point
//     values (no global atomics).  The power-of-two scale per tile is fixed
//     by max |f| of the call and the tile's candidate count, so sums cannot
//     overflow and do not depend on the order of the additions (bitwise
//     reproducible); 64-bit integer LDS atomics also run about 4x faster
//     than FP32 LDS atomics here.  The tile then writes all of its nodes,
//     zeros included, which replaces the zeroing pass of ibm_st1a.
//   - Interpolation: one work group per tile stages the velocity of the tile
//     plus a 3/4-node halo in LDS once and runs the four frozen-field RK
//     stages of its vertices from LDS, one lane per vertex.
#include <type_traits>

#include "common.hpp"

namespace lbmibm {
namespace {

struct IbmGeom {
    int nx, ny, nz;     // unpadded
    int nxp, nyp, nzp;  // padded
    int walls;          // 1: y beyond [0,ny) is wall
    double dx;
};

struct TileGeom {
    int ntx, nty, ntz, ntiles;
    int tx;  // nodes of a tile in x
};

__device__ __forceinline__ bool wrap_index(int &i, int n) {
    if (i < 0) i += n;
    else if (i >= n) i -= n;
    return (unsigned)i < (unsigned)n;
}

__device__ __forceinline__ int pmod(int i, int n) {
    i %= n;
    return i < 0 ? i + n : i;
}

// sin and cos of (pi/2) t for t in [0, 1).  FP32: Taylor series of both to
// degree 13 / 12 in x = (pi/2) t (truncation below 1e-9 on [0, pi/2), so the
// result is within a few ulp of the correctly rounded value), evaluated by
// Horner in x^2 with no range reduction; explicit multiply-adds, so that the
// bits do not depend on where the compiler moves the terms.
__device__ __forceinline__ void sincos_quarter(float t, float *s, float *c) {
    const float x = 1.57079632679489662f * t, x2 = x * x;
    float ps = -1.0f / 6227020800.0f;
    ps = fmaf(ps, x2, 1.0f / 39916800.0f);
    ps = fmaf(ps, x2, -1.0f / 362880.0f);
    ps = fmaf(ps, x2, 1.0f / 5040.0f);
    ps = fmaf(ps, x2, -1.0f / 120.0f);
    ps = fmaf(ps, x2, 1.0f / 6.0f);
    // sin x = x (1 - x^2 (1/6 - x^2 (1/120 - ...)))
    *s = fmaf(-x * x2, ps, x);
    float pc = 1.0f / 479001600.0f;
    pc = fmaf(pc, x2, -1.0f / 3628800.0f);
    pc = fmaf(pc, x2, 1.0f / 40320.0f);
    pc = fmaf(pc, x2, -1.0f / 720.0f);
    pc = fmaf(pc, x2, 1.0f / 24.0f);
    pc = fmaf(pc, x2, -0.5f);
    *c = fmaf(x2, pc, 1.0f);
}
// FP64: the Taylor series of both to degree 17 / 16 of x = (pi/2) min(t, 1 - t)
// in [0, pi/4] (1 - t is exact for t >= 1/2; the first terms left out are below
// 1e-18), sine and cosine exchanged for t > 1/2.  No range reduction, and half
// the registers of the library's sincos.
__device__ __forceinline__ void sincos_quarter(double t, double *s, double *c) {
    const bool upper = t > 0.5;
    const double x = 1.57079632679489661923 * (upper ? 1.0 - t : t), x2 = x * x;
    double ps = 1.0 / 355687428096000.0;  // 1/17!
    ps = fma(ps, x2, -1.0 / 1307674368000.0);
    ps = fma(ps, x2, 1.0 / 6227020800.0);
    ps = fma(ps, x2, -1.0 / 39916800.0);
    ps = fma(ps, x2, 1.0 / 362880.0);
    ps = fma(ps, x2, -1.0 / 5040.0);
    ps = fma(ps, x2, 1.0 / 120.0);
    ps = fma(ps, x2, -1.0 / 6.0);
    double pc = 1.0 / 20922789888000.0;  // 1/16!
    pc = fma(pc, x2, -1.0 / 87178291200.0);
    pc = fma(pc, x2, 1.0 / 479001600.0);
    pc = fma(pc, x2, -1.0 / 3628800.0);
    pc = fma(pc, x2, 1.0 / 40320.0);
    pc = fma(pc, x2, -1.0 / 720.0);
    pc = fma(pc, x2, 1.0 / 24.0);
    pc = fma(pc, x2, -0.5);
    const double sn = fma(x * x2, ps, x), cs = fma(x2, pc, 1.0);
    *s = upper ? cs : sn;
    *c = upper ? sn : cs;
}

// Weights 1 + cos(pi |x_node - xtr| / (2h)) of the 4 nodes from
// floor(xtr/h)-1 (ibm.cu:103-121).  With t = frac(xtr/h) the distances are
// 1+t, t, 1-t, 2-t, so the four cosines are -sin, cos, sin, -cos of pi t/2:
// one sincos of an argument in [0, pi/2) per axis, evaluated in W.
// xtr / h; h == 1 (lattice units) skips the FP64 division, with the same result
__device__ __forceinline__ double over_h(double xtr, double h) { return h == 1.0 ? xtr : xtr / h; }

template <typename W>
__device__ __forceinline__ void stencil(double xtr, double h, int &first, W w[4], bool unit_spacing) {
    const double q = unit_spacing ? xtr : over_h(xtr, h);
    const double fl = floor(q);
    first = (int)fl - 1;
    const W t = (W)(q - fl);
    W sn, cs;
    sincos_quarter(t, &sn, &cs);
    w[0] = W(1) - sn;
    w[1] = W(1) + cs;
    w[2] = W(1) + sn;
    w[3] = W(1) - cs;
}

// First stencil node (padded frame, as stencil()) and fraction t = frac(xtr/h).
template <typename W>
__device__ __forceinline__ void stencil_first(double xtr, double h, int &first, W &t) {
    const double q = over_h(xtr, h);
    const double fl = floor(q);
    first = (int)fl - 1;
    t = (W)(q - fl);
}

// Weights of the 4 nodes from the fraction t (as stencil()).
template <typename W> __device__ __forceinline__ void stencil_weights(W t, W w[4]) {
    W sn, cs;
    sincos_quarter(t, &sn, &cs);
    w[0] = W(1) - sn;
    w[1] = W(1) + cs;
    w[2] = W(1) + sn;
    w[3] = W(1) - cs;
}

// Unpadded first stencil nodes (unwrapped) and weights at a position.
template <typename W>
__device__ __forceinline__ void stencil3(const IbmGeom &g, double x, double y, double z, bool unit, int &x1, int &y1,
                                         int &z1, W wx[4], W wy[4], W wz[4]) {
    if (!unit) {
        stencil<W>(x + (double)(g.nxp - 1) * g.dx / 2.0, g.dx, x1, wx, false);
        stencil<W>(y + (double)(g.nyp - 1) * g.dx / 2.0, g.dx, y1, wy, false);
        stencil<W>(z + (double)(g.nzp - 1) * g.dx / 2.0, g.dx, z1, wz, false);
    } else {  // RK2 / Euler branches use unit spacing (ibm.cu:524-551, 581-608)
        stencil<W>(x + (double)(g.nxp - 1) / 2.0, g.dx, x1, wx, true);
        stencil<W>(y + (double)(g.nyp - 1) / 2.0, g.dx, y1, wy, true);
        stencil<W>(z + (double)(g.nzp - 1) / 2.0, g.dx, z1, wz, true);
    }
    x1 -= 2;
    y1 -= 2;
    z1 -= 2;
}

// Mask of the 4 stencil nodes first..first+3 (periodic when wrap) that fall
// in [o, o+len) of an axis of n nodes; bit k for node first+k.
__device__ __forceinline__ unsigned axis_mask(int first, int o, int len, int n, bool wrap) {
    unsigned m = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        int a = first + k;
        if (wrap) {
            if (a < 0) a += n;
            else if (a >= n) a -= n;
        }
        if (a >= o && a < o + len && a >= 0 && a < n) m |= 1u << k;
    }
    return m;
}

// Tiles along one axis whose nodes can hold the first stencil node of a
// vertex reaching [o, o+len): the tile itself and the tiles of nodes o-3..o-1
// (periodic when wrap).  Returns the number of distinct tiles (1..4).
__device__ __forceinline__ int source_tiles(int t, int o, int n, int tile, bool wrap, int out[4]) {
    int cnt = 1;
    out[0] = t;
    for (int d = 1; d <= 3; d++) {
        int a = o - d;
        if (a < 0) {
            if (!wrap) break;
            a = ((a % n) + n) % n;
        }
        const int s = a / tile;
        bool seen = false;
        for (int i = 0; i < cnt; i++) seen |= out[i] == s;
        if (!seen) out[cnt++] = s;
    }
    return cnt;
}

// ---- binning ---------------------------------------------------------------

template <typename T>
__global__ __launch_bounds__(BIN_WG) void k_bin_count(const double *__restrict__ xs, const T *__restrict__ cf, int nv,
                                                      BinGeom bg, int *__restrict__ home,
                                                      int *__restrict__ tile_count, float *__restrict__ blk_fmax) {
    __shared__ float shm[BIN_WG / 64];
    __shared__ TileTable tab;
    tab.clear();
    __syncthreads();
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    const bool on = v < nv;
    int t = 0;
    float fm = 0.0f;
    if (on) {
        t = home_tile(bg, xs[v], xs[nv + v], xs[2 * (size_t)nv + v]);
        home[v] = t;
        fm = fmaxf(fabsf((float)cf[v]), fmaxf(fabsf((float)cf[nv + v]), fabsf((float)cf[2 * (size_t)nv + v])));
        fm *= 1.0001f;  // margin for the float rounding of |f|
    }
    int slot;
    (void)tab.add(t, on, slot);
    // per-block max |f| (one store per block; k_tile_scan reduces them)
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) fm = fmaxf(fm, __shfl_xor(fm, o));
    if ((threadIdx.x & 63) == 0) shm[threadIdx.x >> 6] = fm;
    __syncthreads();
    tab.flush(tile_count);
    if (threadIdx.x == 0) {
        for (int k = 1; k < BIN_WG / 64; k++) fm = fmaxf(fm, shm[k]);
        blk_fmax[blockIdx.x] = fm;
    }
}

// Heavy-first order of the tiles: a counting sort on a 256-level key of the
// per-tile load, largest first.  The tile kernels take their tiles in this
// order, so the dispatcher starts the longest work groups first and fills the
// tail with light ones (longest-processing-time-first scheduling); the order
// within a key level is arbitrary and does not affect any result.  The last level
// holds nearly all tiles of a sparse lattice: a wave counts it with one atomic.
__device__ void heavy_first_order(const int *load, int n, int *hist, int *order) {
    __shared__ int maxload;
    if (threadIdx.x == 0) maxload = 0;
    for (int i = threadIdx.x; i < 256; i += blockDim.x) hist[i] = 0;
    __syncthreads();
    int m = 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) m = max(m, load[i]);
    atomicMax(&maxload, m);
    __syncthreads();
    int shift = 0;
    while ((maxload >> shift) > 255) shift++;
    const int lane = threadIdx.x & 63;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int key = 255 - (load[i] >> shift);
        const unsigned long long last = __ballot(key == 255);
        if (key < 255) atomicAdd(&hist[key], 1);
        else if (lane == __ffsll((long long)last) - 1) atomicAdd(&hist[255], __popcll(last));
    }
    __syncthreads();
    if (threadIdx.x == 0) {  // exclusive scan of 256 bins
        int acc = 0;
        for (int k = 0; k < 256; k++) {
            const int c = hist[k];
            hist[k] = acc;
            acc += c;
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int key = 255 - (load[i] >> shift);
        const unsigned long long last = __ballot(key == 255);
        if (key < 255) {
            order[atomicAdd(&hist[key], 1)] = i;
        } else {
            const int first = __ffsll((long long)last) - 1;
            int at = 0;
            if (lane == first) at = atomicAdd(&hist[255], __popcll(last));
            order[__shfl(at, first) + __popcll(last & ((1ull << lane) - 1ull))] = i;
        }
    }
    __syncthreads();
}

// The heavy-first tile orders of the spreading from source bins, if that form is
// taken (by candidate count: own bin and the bins below on each axis), and of the
// interpolation and the home boxes (by own count).
// They only steer the dispatch order, and tile loads change slowly with the
// cells, so they are refreshed on every TILE_ORDER_PERIOD-th binning (a call
// counter on the device, so captured graphs refresh them too); any
// permutation is a valid order, the initial one is the identity.
constexpr int TILE_ORDER_PERIOD = 16;

template <bool BINS>
__device__ void tile_orders(const int *__restrict__ tile_count, int ntiles, const IbmGeom &g, const TileGeom &tg,
                            int *__restrict__ tile_cand, int *__restrict__ order_spread,
                            int *__restrict__ order_interp, int *__restrict__ calls) {
    __shared__ int sh[256];
    __shared__ int call;
    if (threadIdx.x == 0) call = (*calls)++;
    __syncthreads();
    if (call % TILE_ORDER_PERIOD != 0) return;
    for (int t = threadIdx.x; BINS && t < ntiles; t += 1024) {
        const int tx = t % tg.ntx, ty = (t / tg.ntx) % tg.nty, tz = t / (tg.ntx * tg.nty);
        int sxs[4], sys[4], szs[4];
        const int nsx = source_tiles(tx, tx * tg.tx, g.nx, tg.tx, true, sxs);
        const int nsy = source_tiles(ty, ty * TILE_Y, g.ny, TILE_Y, !g.walls, sys);
        const int nsz = source_tiles(tz, tz * TILE_Z, g.nz, TILE_Z, true, szs);
        int c = 0;
        for (int iz = 0; iz < nsz; iz++)
            for (int iy = 0; iy < nsy; iy++)
                for (int ix = 0; ix < nsx; ix++) c += tile_count[sxs[ix] + tg.ntx * (sys[iy] + tg.nty * szs[iz])];
        tile_cand[t] = c;
    }
    __syncthreads();
    if (BINS) heavy_first_order(tile_cand, ntiles, sh, order_spread);
    heavy_first_order(tile_count, ntiles, sh, order_interp);
}

// Vertices per work group of k_spread_box, and the work groups of a tile.
constexpr int SB_CHUNK = 800;
__host__ __device__ __forceinline__ int spread_chunks(int cnt) { return (cnt + SB_CHUNK - 1) / SB_CHUNK; }

// Exclusive scans over the tiles, in one work group, 4096 tiles per round (four
// consecutive ones per thread; one each took 79 us for the 65536 tiles of
// 512x256x256 nodes, this 29; the orders that follow 550 us when they were due,
// 80 now): the bins' offsets, and the extra chunks of the tiles that k_spread_box shares
// out (listed in `extra`, (-1, 0) behind the last); and the maximum of the
// per-block force maxima.  Both scans ride in one 64-bit wave scan, one barrier
// a round.  The tile orders follow in the same launch (of their own they took
// 5 us a step, nearly always to find that they are not due).
template <bool BINS>
__global__ __launch_bounds__(1024) void k_tile_scan(const int *__restrict__ tile_count, int *__restrict__ tile_off,
                                                    int *__restrict__ tile_cur, int ntiles,
                                                    const float *__restrict__ blk_fmax, int nblk,
                                                    unsigned *__restrict__ absmax, int *__restrict__ tile_ex,
                                                    int2 *__restrict__ extra, int maxextra, IbmGeom g, TileGeom tg,
                                                    int *__restrict__ tile_cand, int *__restrict__ order_spread,
                                                    int *__restrict__ order_interp, int *__restrict__ order_calls) {
    __shared__ unsigned long long wtot[2][16];
    __shared__ float wmax[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float fm = 0.0f;
    for (int i = threadIdx.x; i < nblk; i += 1024) fm = fmaxf(fm, blk_fmax[i]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) fm = fmaxf(fm, __shfl_xor(fm, o));
    if (lane == 0) wmax[wave] = fm;
    unsigned long long carry = 0ull;  // vertices in the low half, extra chunks in the high half
    int parity = 0;
    constexpr int PER = 4;
    for (int base = 0; base < ntiles; base += 1024 * PER, parity ^= 1) {
        const int i = base + PER * (int)threadIdx.x;
        const bool whole = i + PER <= ntiles;
        int cnt[PER];
        if (whole) {  // the arrays are aligned, i is a multiple of four
            const int4 c = *(const int4 *)(tile_count + i);
            cnt[0] = c.x; cnt[1] = c.y; cnt[2] = c.z; cnt[3] = c.w;
        } else {
#pragma unroll
            for (int j = 0; j < PER; j++) cnt[j] = i + j < ntiles ? tile_count[i + j] : 0;
        }
        unsigned long long own = 0ull;
#pragma unroll
        for (int j = 0; j < PER; j++)
            own += (unsigned)cnt[j] | ((unsigned long long)max(spread_chunks(cnt[j]) - 1, 0) << 32);
        unsigned long long incl = own;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned long long t = __shfl_up(incl, o);
            if (lane >= o) incl += t;
        }
        if (lane == 63) wtot[parity][wave] = incl;
        __syncthreads();
        unsigned long long b = carry + incl - own;
#pragma unroll 4  // all 16 would take the registers of a whole CU, and wait for a free one
        for (int w = 0; w < 16; w++) {
            const unsigned long long t = wtot[parity][w];
            if (w < wave) b += t;
            carry += t;
        }
        int off[PER], ex[PER];
#pragma unroll
        for (int j = 0; j < PER; j++) {
            off[j] = (int)(unsigned)b;
            ex[j] = (int)(b >> 32);
            const int n = max(spread_chunks(cnt[j]) - 1, 0);
#pragma unroll 1
            for (int c = 0; c < n; c++)
                if (ex[j] + c < maxextra) extra[ex[j] + c] = make_int2(i + j, c + 1);
            b += (unsigned)cnt[j] | ((unsigned long long)n << 32);
        }
        if (whole) {
            *(int4 *)(tile_off + i) = make_int4(off[0], off[1], off[2], off[3]);
            *(int4 *)(tile_ex + i) = make_int4(ex[0], ex[1], ex[2], ex[3]);
            *(int4 *)(tile_cur + i) = make_int4(0, 0, 0, 0);
        } else {
#pragma unroll
            for (int j = 0; j < PER; j++)
                if (i + j < ntiles) {
                    tile_off[i + j] = off[j];
                    tile_ex[i + j] = ex[j];
                    tile_cur[i + j] = 0;
                }
        }
    }
    for (int e = (int)(carry >> 32) + (int)threadIdx.x; e < maxextra; e += 1024) extra[e] = make_int2(-1, 0);
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; w++) fm = fmaxf(fm, wmax[w]);
        *absmax = __float_as_uint(fm);
    }
    tile_orders<BINS>(tile_count, ntiles, g, tg, tile_cand, order_spread, order_interp, order_calls);
}

// Spreading data of a vertex, stored in bin order next to its first stencil
// node (node0: x and z wrapped, y + 3): the stencil fractions and the force.
template <typename T> struct SpreadRec {
    T t[3];
    T f[3];
};

template <typename T>
__global__ __launch_bounds__(BIN_WG) void k_bin_scatter(const double *__restrict__ xs, const T *__restrict__ cf,
                                                     const int *__restrict__ home, int nv, IbmGeom g,
                                                     const int *__restrict__ tile_off, int *__restrict__ tile_cur,
                                                     int *__restrict__ home_list, short4 *__restrict__ node0,
                                                     SpreadRec<T> *__restrict__ rec) {
    __shared__ TileTable tab;
    tab.clear();
    __syncthreads();
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    const bool on = v < nv;
    const int t = on ? home[v] : 0;
    int slot;
    const int r = tab.add(t, on, slot);
    __syncthreads();
    tab.flush(tile_cur);
    __syncthreads();
    if (on) {
        const int pos = tile_off[t] + tab.cnt[slot] + r;
        home_list[pos] = v;
        int x1, y1, z1;
        SpreadRec<T> sr;
        stencil_first<T>(xs[v] + (double)(g.nxp - 1) * g.dx / 2.0, g.dx, x1, sr.t[0]);
        stencil_first<T>(xs[nv + v] + (double)(g.nyp - 1) * g.dx / 2.0, g.dx, y1, sr.t[1]);
        stencil_first<T>(xs[2 * (size_t)nv + v] + (double)(g.nzp - 1) * g.dx / 2.0, g.dx, z1, sr.t[2]);
        x1 -= 2; y1 -= 2; z1 -= 2;  // unpadded
        int xw = x1, zw = z1;
        wrap_index(xw, g.nx);
        wrap_index(zw, g.nz);
        xw = min(max(xw, -30000), 30000);
        zw = min(max(zw, -30000), 30000);
        node0[pos] = make_short4((short)xw, (short)min(max(y1 + 3, -30000), 30000), (short)zw, 0);
        // the forces read in vertex order (coalesced), written in bin order
        sr.f[0] = cf[v]; sr.f[1] = cf[nv + v]; sr.f[2] = cf[2 * (size_t)nv + v];
        rec[pos] = sr;
    }
}

// The force part of the spreading records, in bin order, and max |f|, when
// the bins of unchanged positions are reused for new forces (a gather of cf).
template <typename T>
__global__ __launch_bounds__(256) void k_bin_forces(const int *__restrict__ home_list, const T *__restrict__ cf, int nv,
                                                    SpreadRec<T> *__restrict__ rec, unsigned *__restrict__ absmax) {
    __shared__ float shm[4];
    const int pos = blockIdx.x * blockDim.x + threadIdx.x;
    float fm = 0.0f;
    if (pos < nv) {
        const int v = home_list[pos];
        const T f0 = cf[v], f1 = cf[nv + v], f2 = cf[2 * (size_t)nv + v];
        rec[pos].f[0] = f0; rec[pos].f[1] = f1; rec[pos].f[2] = f2;
        fm = fmaxf(fabsf((float)f0), fmaxf(fabsf((float)f1), fabsf((float)f2)));
        fm *= 1.0001f;  // margin for the float rounding of |f|
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) fm = fmaxf(fm, __shfl_xor(fm, o));
    if ((threadIdx.x & 63) == 0) shm[threadIdx.x >> 6] = fm;
    __syncthreads();
    // non-negative floats order as their bit patterns: an integer maximum
    if (threadIdx.x == 0) atomicMax(absmax, __float_as_uint(fmaxf(fmaxf(shm[0], shm[1]), fmaxf(shm[2], shm[3]))));
}

__global__ void k_zero_int(int *__restrict__ p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// a[k] for a runtime k by selects (a runtime index would put a in scratch)
template <typename T> __device__ __forceinline__ T sel4(const T (&a)[4], int k) {
    return k == 0 ? a[0] : k == 1 ? a[1] : k == 2 ? a[2] : a[3];
}

// ---- spreading ---------------------------------------------------------------

// LDS accumulator layout of a tile, rows padded to strides 20 and 176: the
// 64 (kx,ky,kz) offsets of one stencil fall on 32 distinct 8-byte bank slots.
constexpr int ACC_SX = 20, ACC_SXY = 176, ACC_N = ACC_SXY * TILE_Z;

// Accumulation into the tile in 64-bit fixed point with a power-of-two scale,
// so the integer sums do not depend on the order of the additions.
//   FP32: the scale keeps |sum| below 2^47; the product w*(f*scale) is formed
//   by one FP64 FMA with 1.5*2^52 added, which leaves round(w*f*scale) in the
//   low mantissa bits (valid for |value| < 2^51), see below.
//   FP64: the scale keeps |sum| below 2^62 and llrint converts.
template <typename T> struct FixedPoint;
// FP32: t = fma(w, f scale, 1.5 2^52) holds k = round(w f scale) as
// bits(t) = 0x4338 << 48 + k for |k| < 2^51.  The constant part is a multiple
// of 2^48, so the raw bits are summed as they are and the low 48 bits of the
// sum are the sum of the k modulo 2^48: exact whenever the final sum is below
// 2^47 in magnitude, which the per-tile scale guarantees (kBits = 47), however
// the partial sums wrap.  No per-term subtraction.
template <> struct FixedPoint<float> {
    static constexpr int kBits = 47;
    double f[3];
    __device__ __forceinline__ FixedPoint(float f0, float f1, float f2, double scale) {
        f[0] = (double)f0 * scale; f[1] = (double)f1 * scale; f[2] = (double)f2 * scale;
    }
    __device__ __forceinline__ void add(unsigned long long *acc, int li, float w, int stride = ACC_N) const {
        const double wd = (double)w;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const double t = fma(wd, f[d], 6755399441055744.0);  // + 1.5 * 2^52
            atomicAdd(&acc[d * stride + li], (unsigned long long)__double_as_longlong(t));
        }
    }
    // the fixed-point bits of v * scale, as add() forms them
    __device__ __forceinline__ static unsigned long long fixed(double v, double scale) {
        return (unsigned long long)__double_as_longlong(fma(v, scale, 6755399441055744.0));
    }
    __device__ __forceinline__ static long long value(unsigned long long a) {
        return (long long)(a << 16) >> 16;  // sign-extend the low 48 bits
    }
    // value(a) * inv, inv a power of two: value(a) + bits(1.5 2^52) are the
    // bits of value(a) + 1.5 2^52, and the subtraction is exact
    __device__ __forceinline__ static double real(unsigned long long a, double inv) {
        const double t = __longlong_as_double(value(a) + 0x4338000000000000ll);
        return fma(t, inv, -6755399441055744.0 * inv);
    }
};
template <> struct FixedPoint<double> {
    static constexpr int kBits = 62;
    double f[3], scale;
    __device__ __forceinline__ FixedPoint(double f0, double f1, double f2, double s) : scale(s) {
        f[0] = f0; f[1] = f1; f[2] = f2;
    }
    __device__ __forceinline__ void add(unsigned long long *acc, int li, double w, int stride = ACC_N) const {
#pragma unroll
        for (int d = 0; d < 3; d++) atomicAdd(&acc[d * stride + li], (unsigned long long)llrint(w * f[d] * scale));
    }
    __device__ __forceinline__ static unsigned long long fixed(double v, double scale) {
        return (unsigned long long)llrint(v * scale);
    }
    __device__ __forceinline__ static long long value(unsigned long long a) { return (long long)a; }
    __device__ __forceinline__ static double real(unsigned long long a, double inv) { return (double)value(a) * inv; }
};

template <typename T>
__device__ __forceinline__ void spread_vertex(const SpreadRec<T> &sr, short4 n0, const IbmGeom &g, int ox, int oy,
                                              int oz, int lx, int ly, int lz, double scale, T w64,
                                              unsigned long long *acc) {
    const int x1 = n0.x, y1 = n0.y - 3, z1 = n0.z;
    const unsigned mx = axis_mask(x1, ox, lx, g.nx, true);
    const unsigned my = axis_mask(y1, oy, ly, g.ny, !g.walls);
    const unsigned mz = axis_mask(z1, oz, lz, g.nz, true);
    if (!mx || !my || !mz) return;
    T wx[4], wy[4], wz[4];
    stencil_weights<T>(sr.t[0], wx);
    stencil_weights<T>(sr.t[1], wy);
    stencil_weights<T>(sr.t[2], wz);
    const FixedPoint<T> fp(sr.f[0], sr.f[1], sr.f[2], scale);
    // tile-relative offsets of the stencil nodes on each axis
    int ax[4], by[4], cz[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        int a = x1 + k, b = y1 + k, c = z1 + k;
        wrap_index(a, g.nx);
        wrap_index(c, g.nz);
        if (!g.walls) wrap_index(b, g.ny);
        ax[k] = a - ox;
        by[k] = ACC_SX * (b - oy);
        cz[k] = ACC_SXY * (c - oz);
    }
#pragma unroll
    for (int kz = 0; kz < 4; kz++) {
        if (!((mz >> kz) & 1u)) continue;
#pragma unroll
        for (int ky = 0; ky < 4; ky++) {
            if (!((my >> ky) & 1u)) continue;
            const T wyz = wy[ky] * wz[kz] * w64;
            const int row = by[ky] + cz[kz];
#pragma unroll
            for (int kx = 0; kx < 4; kx++) {
                if (!((mx >> kx) & 1u)) continue;
                fp.add(acc, row + ax[kx], wx[kx] * wyz);
            }
        }
    }
}

template <typename T>
__global__ __launch_bounds__(256) void k_spread_tiles(const SpreadRec<T> *__restrict__ rec,
                                                      const short4 *__restrict__ node0,
                                                      const int *__restrict__ tile_count,
                                                      const int *__restrict__ tile_off, T *__restrict__ F,
                                                      IbmGeom g, TileGeom tg, const unsigned *__restrict__ absmax,
                                                      const int *__restrict__ order) {
    __shared__ unsigned long long acc[3 * ACC_N];
    __shared__ int queue[4][128];
    const int tile = order[blockIdx.x];
    const int tx = tile % tg.ntx, ty = (tile / tg.ntx) % tg.nty, tz = tile / (tg.ntx * tg.nty);
    const int ox = tx * tg.tx, oy = ty * TILE_Y, oz = tz * TILE_Z;
    const int lx = min(tg.tx, g.nx - ox), ly = min(TILE_Y, g.ny - oy), lz = min(TILE_Z, g.nz - oz);
    for (int k = threadIdx.x; k < 3 * ACC_N; k += blockDim.x) acc[k] = 0ull;
    // source bins: tiles holding first stencil nodes that reach this tile
    int sxs[4], sys[4], szs[4];
    const int nsx = source_tiles(tx, ox, g.nx, tg.tx, true, sxs);
    const int nsy = source_tiles(ty, oy, g.ny, TILE_Y, !g.walls, sys);
    const int nsz = source_tiles(tz, oz, g.nz, TILE_Z, true, szs);
    // fixed-point scale: at most `total` vertices reach one node, each with a
    // weight at most 1/(8 dx^3), so |sum| <= total |f|max / (8 dx^3), which
    // the power of two keeps below 2^kBits / scale
    long long total = 0;
    for (int iz = 0; iz < nsz; iz++)
        for (int iy = 0; iy < nsy; iy++)
            for (int ix = 0; ix < nsx; ix++) total += tile_count[sxs[ix] + tg.ntx * (sys[iy] + tg.nty * szs[iz])];
    const double fmax = (double)__uint_as_float(*absmax);
    double scale = 1.0;
    if (fmax > 0.0 && total > 0) {
        const double bound = (double)total * fmax / (8.0 * g.dx * g.dx * g.dx);
        scale = ldexp(1.0, FixedPoint<T>::kBits - 1 - ilogb(bound));
    }
    const T w64 = (T)(1.0 / (64.0 * g.dx * g.dx * g.dx));
    __syncthreads();

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int *q = queue[wave];
    int qn = 0;
    for (int s = 0; s < nsx * nsy * nsz; s++) {
        const int bin = sxs[s % nsx] + tg.ntx * (sys[(s / nsx) % nsy] + tg.nty * szs[s / (nsx * nsy)]);
        const int cnt = tile_count[bin], off = tile_off[bin];
        // the bin read as 64 columns of R rows, lane l taking column l: the
        // lanes of a wave get vertices far apart in the bin, whose stencils
        // rarely share LDS addresses (64-bit LDS atomics to one address
        // serialise, and neighbouring vertices in a bin are close in space)
        const int R = (cnt + 63) >> 6;
        for (int r = wave; r < R; r += 4) {
            const int i = lane * R + r;
            int v = -1;  // position in bin order
            bool touch = false;
            if (i < cnt) {
                v = off + i;
                const short4 n0 = node0[v];
                touch = axis_mask(n0.x, ox, lx, g.nx, true) && axis_mask(n0.y - 3, oy, ly, g.ny, !g.walls) &&
                        axis_mask(n0.z, oz, lz, g.nz, true);
            }
            const unsigned long long m = __ballot(touch);
            if (touch) q[qn + __popcll(m & ((1ull << lane) - 1ull))] = v;
            qn += __popcll(m);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (qn >= 64) {
                spread_vertex<T>(rec[q[lane]], node0[q[lane]], g, ox, oy, oz, lx, ly, lz, scale, w64, acc);
                const int rest = qn - 64;
                const int mv = lane < rest ? q[64 + lane] : 0;
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                if (lane < rest) q[lane] = mv;
                qn = rest;
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
        }
    }
    if (lane < qn) spread_vertex<T>(rec[q[lane]], node0[q[lane]], g, ox, oy, oz, lx, ly, lz, scale, w64, acc);
    __syncthreads();
    const double inv_scale = 1.0 / scale;
    const size_t N = (size_t)g.nx * g.ny * g.nz;
    for (int k = threadIdx.x; k < tg.tx * TILE_Y * TILE_Z; k += blockDim.x) {
        const int la = k % tg.tx, lb = (k / tg.tx) % TILE_Y, lc = k / (tg.tx * TILE_Y);
        if (la >= lx || lb >= ly || lc >= lz) continue;
        const size_t nidx = (size_t)(ox + la) + (size_t)g.nx * ((size_t)(oy + lb) + (size_t)g.ny * (oz + lc));
        const int li = la + ACC_SX * lb + ACC_SXY * lc;
#pragma unroll
        for (int d = 0; d < 3; d++)
            F[d * N + nidx] = (T)((double)FixedPoint<T>::value(acc[d * ACC_N + li]) * inv_scale);
    }
}

// Spreading, form 1.  One work group per tile takes its home vertices only
// and adds their whole 4x4x4 stencils into an LDS box of the tile plus the 3
// nodes above it on each axis (its stencils cannot leave that box); the box is
// then written to a staging array, and k_spread_gather sums for each lattice
// node the box entries that map to it.
//
// Vertices whose stencils start at the same node ("a cell") add to the same
// 64 nodes, F[(ky,kz), (kx,d)] = sum_v (wy_ky wz_kz)(v) (wx_kx f_d)(v): a 16 x 12
// product over the cell's vertices, which the FP64 matrix instruction takes
// four vertices at a time.  The work group sorts its vertices by cell in LDS
// (within a cell by vertex id, so that the sums do not depend on the order in
// which the binning placed them), a wave multiplies one cell after another,
// and each cell's 192 sums then go into the box as 64-bit fixed point with
// integer LDS atomics.  That rate of the atomics is what bounded the form that
// issued them per vertex (about 12 cycles per wave and CU): a mesh of 2562
// vertices on a radius of 4 has 13 vertices per cell, the uneven suspension of
// 1024 cells 4.8.  Per launch, before and after: 64 cells of 2562 vertices
// (FP32) 90 -> 34 us, that suspension 250 -> 205 us, 384 such cells in FP64
// 144 -> 122 us; with 8x8x8 tiles, 16x8x8 before.  What bounds it now is the
// latency of its phases (loads, scan, sort, products) at the three work groups
// that the box's LDS admits per CU.
// The weights are formed in T, their products and sums in FP64.
constexpr int SB_X = TILE_X + 3, SB_Y = TILE_Y + 3, SB_Z = TILE_Z + 3, SB_N = SB_X * SB_Y * SB_Z;
constexpr int SPREAD_BOX_WG = 512;
constexpr int SB_MAXC = 4;  // box entries per lattice coordinate and axis (k_spread_gather)
constexpr int SB_KEYS = TILE_X * SB_Y * TILE_Z;  // cells of a tile; y from -3 (below the wall in the first tile row)
// A tile of more than SB_CHUNK vertices is shared out by its cells between
// several work groups, each with a box of its own, which k_spread_combine adds
// up: 64 cells of radius 4 fill 159 of 1024 tiles with up to 2490 vertices, and
// the launch would end with the fullest.  Those boxes stay in fixed point (ChunkBox),
// so that the tile's sum is rounded to T once, as that of a tile of one chunk.
// SPAN: sorted vertices per wave and batch; with these three work groups fit a
// CU's LDS.
constexpr int SB_VPT = 2, SB_CAP = SB_VPT * SPREAD_BOX_WG;
template <typename T> constexpr int SB_SPAN = sizeof(T) == 4 ? 32 : 16;
static_assert(SB_CAP > SB_CHUNK, "the sort takes a chunk and a spread about it");
typedef double double_x4 __attribute__((ext_vector_type(4)));

// The fixed-point sums of one chunk of a tile that is shared out.  Their scales
// follow behind the boxes: a power of two, or infinity where the chunk's forces are all 0 (and 0
// where one is infinite, which gives a tile without finite sums).  The boxes of the
// extra chunks first, at the number of the chunk; behind them those of the
// first chunks, at the number of the tile's first extra chunk.
struct ChunkBox {
    long long v[3 * SB_N];
};
__device__ __forceinline__ double *chunk_scales(ChunkBox *chunks, int maxextra) {
    return (double *)(chunks + 2 * (size_t)maxextra);
}

template <typename T>
__global__ __launch_bounds__(SPREAD_BOX_WG, sizeof(T) == 4 ? 6 : 4) void k_spread_box(const SpreadRec<T> *__restrict__ rec,
                                                              const short4 *__restrict__ node0,
                                                              const int *__restrict__ home_list,
                                                              const int *__restrict__ tile_count,
                                                              const int *__restrict__ tile_off, T *__restrict__ S,
                                                              IbmGeom g, TileGeom tg, const int *__restrict__ order,
                                                              const int2 *__restrict__ extra, int maxextra,
                                                              const int *__restrict__ tile_ex,
                                                              ChunkBox *__restrict__ chunks) {
    constexpr int WG_ = SPREAD_BOX_WG, NW = WG_ / 64, SPAN = SB_SPAN<T>, BATCH = NW * SPAN;
    constexpr int KPT = (SB_KEYS + WG_) / WG_;  // keys per thread of the scan, and the total
    // REC values per sorted vertex: sin and cos of the x, y and z fractions, the
    // force and a 0 (for the result columns that no component has); the record
    // behind the last one is all 0: what a block's missing vertices read
    constexpr int REC = 10;
    union Work {
        int id[SB_CAP + 4];  // the selected vertices, then vertex ids by unordered position
        T b[REC * (BATCH + 1)];
    };
    __shared__ unsigned long long acc[3 * SB_N];
    __shared__ Work wk;
    __shared__ int start[SB_KEYS + 1];  // counts of the keys, then their first sorted positions
    __shared__ unsigned short okey[SB_CAP];
    __shared__ int wsum[NW], nsel;
    __shared__ float wmax[NW];
    // the extra chunks of full tiles first, then every tile's first chunk
    int tile, chunk = 0;
    if ((int)blockIdx.x < maxextra) {
        const int2 ex = extra[blockIdx.x];
        if (ex.x < 0) return;  // not so many chunks
        tile = ex.x;
        chunk = ex.y;
    } else {
        tile = order[blockIdx.x - maxextra];
    }
    const int cnt = tile_count[tile], off = tile_off[tile], ex0 = tile_ex[tile];
    if (cnt == 0) return;  // whole work group leaves together; the gather skips empty tiles
    const int nch = spread_chunks(cnt);
    const int tx = tile % tg.ntx, ty = (tile / tg.ntx) % tg.nty, tz = tile / (tg.ntx * tg.nty);
    const int ox = tx * TILE_X, oy = ty * TILE_Y, oz = tz * TILE_Z;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // the cell of a vertex's first stencil node (x, z wrapped at binning; y
    // raw: with walls it may lie below the lattice in the first tile row), -1
    // when this tile is not a valid home
    auto key_of = [&](short4 n0) {
        int y1 = n0.y - 3;
        if (!g.walls) wrap_index(y1, g.ny);
        const int bx = n0.x - ox, by = y1 - oy + 3, bz = n0.z - oz;
        if (bx < 0 || bx >= TILE_X || bz < 0 || bz >= TILE_Z || by < 0 || by >= SB_Y) return -1;
        return bx + TILE_X * (by + SB_Y * bz);
    };
    for (int k = tid; k < 3 * SB_N; k += WG_) acc[k] = 0ull;
    for (int k = tid; k <= SB_KEYS; k += WG_) start[k] = 0;
    if (tid == 0) nsel = 0;
    __syncthreads();
    // exclusive scan of the key counts, KPT consecutive keys per thread, the total behind the last
    auto scan_keys = [&] {
        int own[KPT], before = 0;
#pragma unroll
        for (int k = 0; k < KPT; k++) {
            own[k] = KPT * tid + k < SB_KEYS ? start[KPT * tid + k] : 0;
            before += own[k];
        }
        int incl = before;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int t = __shfl_up(incl, o);
            if (lane >= o) incl += t;
        }
        if (lane == 63) wsum[wave] = incl;
        __syncthreads();
        int base = incl - before;
#pragma unroll
        for (int w = 0; w < NW; w++)
            if (w < wave) base += wsum[w];
#pragma unroll
        for (int k = 0; k < KPT; k++) {
            if (KPT * tid + k <= SB_KEYS) start[KPT * tid + k] = base;
            base += own[k];
        }
    };
    int n = cnt, lo = 0, hi = cnt;
    if (nch > 1) {
        // this chunk's cells: a stretch of the tile's vertices in the order of
        // their cells (a share by the cells' numbers alone gave a flat membrane
        // that runs diagonally through the tile to one chunk whole)
        for (int i = tid; i < cnt; i += WG_) {
            const int k = key_of(node0[off + i]);
            if (k >= 0) atomicAdd(&start[k], 1);
        }
        __syncthreads();
        scan_keys();
        __syncthreads();
        const int all = __builtin_amdgcn_readfirstlane(start[SB_KEYS]);
        lo = (int)((long long)all * chunk / nch);
        hi = (int)((long long)all * (chunk + 1) / nch);
#pragma unroll 2
        for (int i0 = 0; i0 < cnt; i0 += WG_) {  // whole waves: one counter update per wave
            const int i = i0 + tid;
            const int k = key_of(node0[off + min(i, cnt - 1)]);
            const bool take = i < cnt && k >= 0 && start[max(k, 0)] >= lo && start[max(k, 0)] < hi;
            const unsigned long long m = __ballot(take);
            int at = 0;
            if (lane == 0) at = atomicAdd(&nsel, __popcll(m));
            at = __builtin_amdgcn_readfirstlane(at) + __popcll(m & ((1ull << lane) - 1ull));
            if (take && at < SB_CAP) wk.id[at] = i;
        }
        __syncthreads();
        n = __builtin_amdgcn_readfirstlane(nsel);
    }
    const bool sorted = n <= SB_CAP;
    if (nch > 1 && sorted) {
        for (int k = tid; k <= SB_KEYS; k += WG_) start[k] = 0;
        __syncthreads();
    }
    // this thread's vertices, all loads first
    int key[SB_VPT], id[SB_VPT], r[SB_VPT];
    SpreadRec<T> sr[SB_VPT];
    float fm = 0.0f;
    if (sorted) {
        int i[SB_VPT];
        short4 n0[SB_VPT];
#pragma unroll
        for (int j = 0; j < SB_VPT; j++) {
            const int at = tid + j * WG_;
            i[j] = off + (at < n ? (nch > 1 ? wk.id[at] : at) : 0);
        }
#pragma unroll
        for (int j = 0; j < SB_VPT; j++) {
            key[j] = -1;
            if (tid + j * WG_ < n) {
                n0[j] = node0[i[j]];
                id[j] = home_list[i[j]];
                sr[j] = rec[i[j]];
            }
        }
#pragma unroll
        for (int j = 0; j < SB_VPT; j++)
            if (tid + j * WG_ < n) {
                key[j] = key_of(n0[j]);
                r[j] = key[j] >= 0 ? atomicAdd(&start[key[j]], 1) : 0;
                fm = fmaxf(fm, fmaxf(fabsf((float)sr[j].f[0]), fmaxf(fabsf((float)sr[j].f[1]), fabsf((float)sr[j].f[2]))));
            }
    } else {
        for (int i = tid; i < cnt; i += WG_) {
            const SpreadRec<T> s = rec[off + i];
            fm = fmaxf(fm, fmaxf(fabsf((float)s.f[0]), fmaxf(fabsf((float)s.f[1]), fabsf((float)s.f[2]))));
        }
    }
    // a box node takes at most one term per vertex, each at most |f|max /
    // (8 dx^3) with |f|max over the chunk's own vertices (a maximum, so
    // independent of the order of the records): the power of two keeps the
    // sums below 2^kBits
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) fm = fmaxf(fm, __shfl_xor(fm, o));
    if (lane == 0) wmax[wave] = fm;
    __syncthreads();
    if (sorted) scan_keys();  // otherwise the tile's own scan stays, for the bounds
    fm = wmax[0];
#pragma unroll
    for (int w = 1; w < NW; w++) fm = fmaxf(fm, wmax[w]);
    // the float rounding of a double |f| may round down
    const double fmax = (double)fm * (1.0 + 0x1p-20);
    double scale = 1.0;
    if (fmax > 0.0) {
        const double bound = (double)cnt * fmax / (8.0 * g.dx * g.dx * g.dx);
        scale = ldexp(1.0, FixedPoint<T>::kBits - 1 - ilogb(bound));
    }
    const double w64 = scale / (64.0 * g.dx * g.dx * g.dx);
    __syncthreads();
    if (sorted) {
        // unordered positions, then ordered by vertex id within each cell
#pragma unroll
        for (int j = 0; j < SB_VPT; j++)
            if (key[j] >= 0) wk.id[start[key[j]] + r[j]] = id[j];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < SB_VPT; j++) {
            if (key[j] < 0) continue;
            const int a = start[key[j]], b = start[key[j] + 1];
            int at = a;
            for (int t = a; t < b; t += 4) {  // four reads at a time
                const int i0 = wk.id[t], i1 = wk.id[t + 1], i2 = wk.id[t + 2], i3 = wk.id[t + 3];
                at += i0 < id[j];
                at += t + 1 < b && i1 < id[j];
                at += t + 2 < b && i2 < id[j];
                at += t + 3 < b && i3 < id[j];
            }
            r[j] = at;
            okey[at] = (unsigned short)key[j];
        }
        n = start[SB_KEYS];
        // operand lane j = lane & 15 of vertex lane >> 4: wy_(j&3) wz_(j>>2) and
        // wx_(j&3) f_(j>>2); result lane: kx = lane & 3, d = (lane >> 2) & 3,
        // ky = lane >> 4, register i: kz = i
        const int jx = lane & 3, jz = (lane >> 2) & 3;
        const T sgx = jx == 0 || jx == 3 ? T(-1) : T(1), sgz = jz == 0 || jz == 3 ? T(-1) : T(1);
        const int vrec = REC * (lane >> 4);
        unsigned long long *const out = acc + jz * SB_N + jx + SB_X * ((lane >> 4) - 3);
        const bool edge = g.walls && ty == 0;
        __syncthreads();
        // batches of equal size, spans of equal size per wave
        const int nb = (n + BATCH - 1) / BATCH, span = nb ? ((n + nb - 1) / nb + NW - 1) / NW : 0;
        for (int s0 = 0; s0 < n; s0 += NW * span) {
#pragma unroll
            for (int j = 0; j < SB_VPT; j++) {
                if (key[j] < 0 || r[j] < s0 || r[j] >= s0 + NW * span) continue;
                T *o = wk.b + REC * (r[j] - s0);
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    T sn, cs;
                    sincos_quarter(sr[j].t[d], &sn, &cs);
                    o[2 * d] = sn;
                    o[2 * d + 1] = cs;
                    o[6 + d] = sr[j].f[d];
                }
                o[9] = T(0);
            }
            if (tid < REC) wk.b[REC * NW * span + tid] = T(0);
            __syncthreads();
            const int sA = s0 + wave * span;
            const int m = __builtin_amdgcn_readfirstlane(min(span, n - sA));
            if (m > 0) {
                // the span's blocks of up to four vertices of one cell, listed
                // one per lane: first slot, end of the cell's slots, key
                const int kk = lane < m ? (int)okey[sA + lane] : -1;
                const int prev = __shfl_up(kk, 1);
                const unsigned long long starts = __ballot(lane < m && (lane == 0 || kk != prev));
                const unsigned long long upto = (2ull << lane) - 1ull, later = starts & ~upto;
                const int first = 63 - __clzll((long long)(starts & upto));  // slot 0 is a start
                const int last = later ? __ffsll((long long)later) - 1 : m;
                const bool blk = lane < m && ((lane - first) & 3) == 0;
                const unsigned long long blocks = __ballot(blk);
                const int nblk = __popcll(blocks);
                const unsigned long long below = blk ? blocks : ~blocks;
                // the cell's place in the box: x + SB_X (y + 3) + SB_X SB_Y z, y from -3
                const int box = kk % TILE_X + SB_X * (kk / TILE_X % SB_Y + SB_Y * (kk / (TILE_X * SB_Y)));
                // every lane takes part, those without a block behind the list
                const int list = __builtin_amdgcn_ds_permute(
                    4 * ((blk ? 0 : nblk) + __popcll(below & (upto >> 1))), lane | (last << 6) | (box << 12));
                auto operands = [&](int d, double &A, double &B) {
                    const int p = d & 63, e = (d >> 6) & 63;
                    const int at = (lane >> 4) < e - p ? REC * (wave * span + p) + vrec : REC * NW * span;
                    const T *qx = wk.b + at + (jx & 1), *qz = wk.b + at + 4 + (jz & 1);
                    const T wx = fma(sgx, qx[0], T(1)), wy = fma(sgx, qx[2], T(1)), wz = fma(sgz, qz[0], T(1));
                    A = (double)wy * (double)wz;
                    B = (double)wx * (double)wk.b[at + 6 + jz];
                };
                // a cell's sums into the box: result column d = 3 is none
                auto flush = [&](int d, const double_x4 &c) {
                    const int at = d >> 12;
                    // below the wall only in the first tile row (the box has no such rows)
                    const bool low = edge && at % (SB_X * SB_Y) / SB_X + (lane >> 4) < 3;
                    unsigned long long *o = out + at;
                    if (jz < 3 && !low) {
#pragma unroll
                        for (int i = 0; i < 4; i++) atomicAdd(o + i * SB_X * SB_Y, FixedPoint<T>::fixed(c[i], w64));
                    }
                };
                // two halves of the list at once: their chains of loads,
                // product and addition do not wait for each other
                const int h = (nblk + 1) >> 1;
                const double_x4 zero = {0.0, 0.0, 0.0, 0.0};
                double_x4 c0 = zero, c1 = zero;
                double A0, B0, A1, B1;
                int d0 = __builtin_amdgcn_readlane(list, 0), d1 = __builtin_amdgcn_readlane(list, min(h, nblk - 1));
                operands(d0, A0, B0);
                operands(d1, A1, B1);
                bool new0 = true, new1 = true;
                for (int i = 0; i < h; i++) {
                    if (new0) c0 = __builtin_amdgcn_mfma_f64_16x16x4f64(A0, B0, zero, 0, 0, 0);
                    else c0 = __builtin_amdgcn_mfma_f64_16x16x4f64(A0, B0, c0, 0, 0, 0);
                    if (new1) c1 = __builtin_amdgcn_mfma_f64_16x16x4f64(A1, B1, zero, 0, 0, 0);
                    else c1 = __builtin_amdgcn_mfma_f64_16x16x4f64(A1, B1, c1, 0, 0, 0);
                    const int e0 = d0, e1 = d1;
                    if (i + 1 < h) {  // the next blocks' operands while these are multiplied
                        d0 = __builtin_amdgcn_readlane(list, i + 1);
                        d1 = __builtin_amdgcn_readlane(list, min(h + i + 1, nblk - 1));
                        operands(d0, A0, B0);
                        operands(d1, A1, B1);
                    }
                    new0 = i + 1 == h || (e0 & 63) + 4 >= ((e0 >> 6) & 63);
                    new1 = h + i + 1 >= nblk || (e1 & 63) + 4 >= ((e1 >> 6) & 63);
                    if (new0) flush(e0, c0);
                    if (new1 && h + i < nblk) flush(e1, c1);
                }
            }
            __syncthreads();
        }
    } else {
        // more vertices than the sort holds: a stretch ends with a whole cell, so
        // one of SB_CAP - SB_CHUNK vertices or more at its end may be too many.
        // Their terms one by one
        const T w1 = (T)(1.0 / (64.0 * g.dx * g.dx * g.dx));
        for (int i = tid; i < cnt; i += WG_) {
            const int kc = key_of(node0[off + i]);
            if (kc < 0 || start[kc] < lo || start[kc] >= hi) continue;
            const SpreadRec<T> s = rec[off + i];
            T wx[4], wy[4], wz[4];
            stencil_weights<T>(s.t[0], wx);
            stencil_weights<T>(s.t[1], wy);
            stencil_weights<T>(s.t[2], wz);
            const FixedPoint<T> fp(s.f[0], s.f[1], s.f[2], scale);
            const int bx = kc % TILE_X, by = (kc / TILE_X) % SB_Y - 3, bz = kc / (TILE_X * SB_Y);
#pragma unroll 1
            for (int c = 0; c < 64; c++) {
                const int kx = c & 3, ky = (c >> 2) & 3, kz = c >> 4;
                if (by + ky < 0) continue;
                fp.add(acc, bx + kx + SB_X * ((by + ky) + SB_Y * (bz + kz)),
                       sel4(wx, kx) * (sel4(wy, ky) * sel4(wz, kz) * w1), SB_N);
            }
        }
        __syncthreads();
    }
    const double inv_scale = 1.0 / scale;
    T *St = S + (size_t)tile * 3 * SB_N;
    const int slot = chunk > 0 ? (int)blockIdx.x : maxextra + ex0;
    ChunkBox *box = chunks + (nch == 1 ? 0 : slot);
    for (int k0 = tid; k0 < 3 * SB_N; k0 += 4 * WG_) {  // four reads, then four stores
        unsigned long long a[4];
#pragma unroll
        for (int j = 0; j < 4; j++) a[j] = acc[min(k0 + j * WG_, 3 * SB_N - 1)];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int k = k0 + j * WG_;
            if (k >= 3 * SB_N) continue;
            if (nch > 1) box->v[k] = FixedPoint<T>::value(a[j]);
            else St[k] = (T)FixedPoint<T>::real(a[j], inv_scale);
        }
    }
    if (nch > 1 && tid == 0) chunk_scales(chunks, maxextra)[slot] = fmax > 0.0 ? scale : HUGE_VAL;
}

// Adds the chunks' boxes of each tile that was shared out into the tile's box:
// work groups (e, .) take the tile whose first extra chunk is e, the others
// leave at once.  The sum is formed in fixed point at the coarsest of the chunks'
// scales, which is the one that all of the tile's vertices in one work group would
// have had, and rounded to T at the end; boxes rounded to FP32 and added in FP32
// lost up to 2.8 times as much where the chunks' sums cancel.  That costs twice
// the bytes: 64 cells 33.4 -> 34.1 us in k_spread_box (and 5.2 here), the 1024-cell
// suspension 199 -> 206 (and 15.8 here).  What bounds this is the chain of loads: the
// first two boxes' beside that of their number, then four boxes at a time; one
// after another took 7.9 and 20.5, and 78 instead of 19 where 82000 vertices lie in a
// few tiles.  The boxes are read once: past the caches, or they would drive out
// those that the gather reads next (62 instead of 55 us).  The gather adding the chunks itself took 64 instead of 44 us: the
// loop over them keeps its loads from being issued together.
constexpr int COMBINE_WG = 256, COMBINE_PER = 4;  // threads and values of each; blockIdx.y: stretch of the box
constexpr int COMBINE_PARTS = (3 * SB_N + COMBINE_WG * COMBINE_PER - 1) / (COMBINE_WG * COMBINE_PER);
template <typename T>
__global__ __launch_bounds__(COMBINE_WG) void k_spread_combine(T *__restrict__ S, ChunkBox *__restrict__ chunks,
                                                         const int2 *__restrict__ extra,
                                                         const int *__restrict__ tile_count, int maxextra) {
    const int2 ex = extra[blockIdx.x];
    if (ex.x < 0 || ex.y != 1) return;
    const ChunkBox *first = chunks + maxextra + blockIdx.x, *more = chunks + blockIdx.x;
    // every load that does not need the number of chunks, beside that of the number
    constexpr int PER = COMBINE_PER;
    const int k0 = (int)blockIdx.y * COMBINE_WG * PER + (int)threadIdx.x;
    int k[PER];
    long long v[PER], next[PER], sum[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) {
        k[j] = min(k0 + COMBINE_WG * j, 3 * SB_N - 1);
        v[j] = __builtin_nontemporal_load(&first->v[k[j]]);
        next[j] = __builtin_nontemporal_load(&more[0].v[k[j]]);
        sum[j] = 0;
    }
    const int nx = spread_chunks(tile_count[ex.x]) - 1;
    const double *scales = chunk_scales(chunks, maxextra), *ms = scales + blockIdx.x;
    const double s0 = scales[maxextra + blockIdx.x];
    double scale = fmin(s0, ms[0]);  // the coarsest
    for (int c = 1; c < nx; c++) scale = fmin(scale, ms[c]);
    const int e = ilogb(scale);
    auto add = [&](const long long (&w)[PER], double t) {
        // at most 62: a chunk without forces, at infinity, holds zeros
        const int sh = scale > 0.0 ? (int)min((long long)ilogb(t) - e, 62ll) : 0;
        const long long half = sh > 0 ? 1ll << (sh - 1) : 0;
#pragma unroll
        for (int j = 0; j < PER; j++) sum[j] += (w[j] + half) >> sh;
    };
    add(v, s0);
    add(next, ms[0]);
    constexpr int AHEAD = 4;  // boxes read at a time
    for (int c0 = 1; c0 < nx; c0 += AHEAD) {
        long long w[AHEAD][PER];
#pragma unroll
        for (int a = 0; a < AHEAD; a++)
#pragma unroll
            for (int j = 0; j < PER; j++) w[a][j] = __builtin_nontemporal_load(&more[min(c0 + a, nx - 1)].v[k[j]]);
#pragma unroll
        for (int a = 0; a < AHEAD; a++)
            if (c0 + a < nx) add(w[a], ms[c0 + a]);
    }
    const double inv = 1.0 / scale;
    T *own = S + (size_t)ex.x * 3 * SB_N;
#pragma unroll
    for (int j = 0; j < PER; j++)
        if (k0 + COMBINE_WG * j < 3 * SB_N) own[k[j]] = (T)((double)sum[j] * inv);
}

// Spreading, form 1, point by point (lbmibm_ctx::pointwise): every vertex adds
// its 64 products, formed in FP32, to the box of its tile, at the rate of the
// LDS atomics: 29 us on 77x46x51 nodes with 3204 vertices, as before, of
// about 330 us of kernels per step.  Lane l of wave w takes column
// NW l + w of the bin read as WG columns, so that the lanes of a wave hold
// vertices far apart.
constexpr int SP_X = TILE_XW + 3, SP_N = SP_X * SB_Y * SB_Z;
__global__ __launch_bounds__(SPREAD_BOX_WG) void k_spread_points(const SpreadRec<float> *__restrict__ rec,
                                                                 const short4 *__restrict__ node0,
                                                                 const int *__restrict__ tile_count,
                                                                 const int *__restrict__ tile_off,
                                                                 float *__restrict__ S, IbmGeom g, TileGeom tg,
                                                                 const int *__restrict__ order) {
    __shared__ unsigned long long acc[3 * SP_N];
    __shared__ float wmax[SPREAD_BOX_WG / 64];
    const int tile = order[blockIdx.x];
    const int cnt = tile_count[tile], off = tile_off[tile];
    if (cnt == 0) return;  // whole work group leaves together; the gather skips empty tiles
    const int tx = tile % tg.ntx, ty = (tile / tg.ntx) % tg.nty, tz = tile / (tg.ntx * tg.nty);
    const int ox = tx * TILE_XW, oy = ty * TILE_Y, oz = tz * TILE_Z;
    for (int k = threadIdx.x; k < 3 * SP_N; k += SPREAD_BOX_WG) acc[k] = 0ull;
    constexpr int NW = SPREAD_BOX_WG / 64;
    const int R = (cnt + SPREAD_BOX_WG - 1) / SPREAD_BOX_WG;
    const int first = (NW * (threadIdx.x & 63) + (threadIdx.x >> 6)) * R, last = min(first + R, cnt);
    float fm = 0.0f;
    for (int i = first; i < last; i++) {
        const SpreadRec<float> sr = rec[off + i];
        fm = fmaxf(fm, fmaxf(fabsf(sr.f[0]), fmaxf(fabsf(sr.f[1]), fabsf(sr.f[2]))));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) fm = fmaxf(fm, __shfl_xor(fm, o));
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = fm;
    __syncthreads();
    fm = wmax[0];
#pragma unroll
    for (int w = 1; w < NW; w++) fm = fmaxf(fm, wmax[w]);
    const double fmax = (double)fm * (1.0 + 0x1p-20);  // scale as in k_spread_box
    double scale = 1.0;
    if (fmax > 0.0) {
        const double bound = (double)cnt * fmax / (8.0 * g.dx * g.dx * g.dx);
        scale = ldexp(1.0, FixedPoint<float>::kBits - 1 - ilogb(bound));
    }
    const float w64 = (float)(1.0 / (64.0 * g.dx * g.dx * g.dx));
    for (int i = first; i < last; i++) {
        const short4 n0 = node0[off + i];
        const SpreadRec<float> sr = rec[off + i];
        const int bx = n0.x - ox, bz = n0.z - oz;
        int y1 = n0.y - 3;
        if (!g.walls) wrap_index(y1, g.ny);
        const int by = y1 - oy;
        if (bx < 0 || bx >= TILE_XW || bz < 0 || bz >= TILE_Z || by < -3 || by >= TILE_Y) continue;  // not a valid home
        float wx[4], wy[4], wz[4];
        stencil_weights<float>(sr.t[0], wx);
        stencil_weights<float>(sr.t[1], wy);
        stencil_weights<float>(sr.t[2], wz);
        const FixedPoint<float> fp(sr.f[0], sr.f[1], sr.f[2], scale);
#pragma unroll
        for (int kz = 0; kz < 4; kz++) {
#pragma unroll
            for (int ky = 0; ky < 4; ky++) {
                if (by + ky < 0) continue;  // below the wall
                const float wyz = wy[ky] * wz[kz] * w64;
                const int row = bx + SP_X * ((by + ky) + SB_Y * (bz + kz));
#pragma unroll
                for (int kx = 0; kx < 4; kx++) fp.add(acc, row + kx, wx[kx] * wyz, SP_N);
            }
        }
    }
    __syncthreads();
    const double inv_scale = 1.0 / scale;
    float *St = S + (size_t)tile * 3 * SP_N;
    for (int k = threadIdx.x; k < 3 * SP_N; k += SPREAD_BOX_WG)
        St[k] = (float)FixedPoint<float>::real(acc[k], inv_scale);
}

// Sums, per lattice node, the box entries of k_spread_box that map to it, in
// a fixed order (deterministic).  cx/cy/cz list for each coordinate of an axis
// up to SB_MAXC entries (tile index along the axis) * 32 + box coordinate,
// padded with -1 (built once on the host).  The boxes are added in FP64 and the sum
// is rounded to T once: tiles of 8 nodes put more of them into a node than those of
// 16 did.  Boxes of 16x8x8 tiles (lbmibm_ctx::pointwise) are added in T, as they
// always were.
template <typename T, int TX>
__global__ __launch_bounds__(256) void k_spread_gather(const T *__restrict__ S, const int *__restrict__ tile_count,
                                                       const int *__restrict__ cx, const int *__restrict__ cy,
                                                       const int *__restrict__ cz, T *__restrict__ F, IbmGeom g,
                                                       TileGeom tg) {
    constexpr int BX = TX + 3, BN = BX * SB_Y * SB_Z;
    const size_t N = (size_t)g.nx * g.ny * g.nz;
    // each XCD gathers one contiguous eighth of the lattice: the box rows
    // of neighbouring y rows share cache lines, which are then fetched into
    // one L2 instead of into the L2s of the XCDs the rows' work groups land on
    const int nblocks = (int)((N + 255) / 256);
    const int lb = xcd_block(nblocks);
    if (lb >= nblocks) return;
    const size_t n = (size_t)lb * 256 + threadIdx.x;
    if (n >= N) return;
    const int x = (int)(n % g.nx), y = (int)((n / g.nx) % g.ny), z = (int)(n / ((size_t)g.nx * g.ny));
    // all table entries first, then per (z, y) entry the tile counts and box
    // values of every x entry, so that independent loads are in flight
    // together; the sums keep the order (z, y, x entry)
    int ex[SB_MAXC], ey[SB_MAXC], ez[SB_MAXC];
#pragma unroll
    for (int i = 0; i < SB_MAXC; i++) {
        ex[i] = cx[SB_MAXC * x + i];
        ey[i] = cy[SB_MAXC * y + i];
        ez[i] = cz[SB_MAXC * z + i];
    }
    using Sum = std::conditional_t<TX == TILE_X, double, T>;
    Sum a0 = Sum(0), a1 = Sum(0), a2 = Sum(0);
#pragma unroll
    for (int iz = 0; iz < SB_MAXC; iz++) {
        if (ez[iz] < 0) break;
#pragma unroll
        for (int iy = 0; iy < SB_MAXC; iy++) {
            if (ey[iy] < 0) break;
            const int tyz = tg.ntx * ((ey[iy] >> 5) + tg.nty * (ez[iz] >> 5));
            const int byz = BX * ((ey[iy] & 31) + SB_Y * (ez[iz] & 31));
            int cnt[SB_MAXC];
#pragma unroll
            for (int ix = 0; ix < SB_MAXC; ix++) cnt[ix] = ex[ix] >= 0 ? tile_count[(ex[ix] >> 5) + tyz] : 0;
            T v0[SB_MAXC], v1[SB_MAXC], v2[SB_MAXC];
#pragma unroll
            for (int ix = 0; ix < SB_MAXC; ix++) {
                v0[ix] = v1[ix] = v2[ix] = T(0);
                if (cnt[ix] > 0) {
                    const size_t b = (size_t)((ex[ix] >> 5) + tyz) * 3 * BN + (ex[ix] & 31) + byz;
                    v0[ix] = S[b];
                    v1[ix] = S[b + BN];
                    v2[ix] = S[b + 2 * BN];
                }
            }
#pragma unroll
            for (int ix = 0; ix < SB_MAXC; ix++)
                if (cnt[ix] > 0) { a0 += v0[ix]; a1 += v1[ix]; a2 += v2[ix]; }
        }
    }
    F[n] = (T)a0;
    F[N + n] = (T)a1;
    F[2 * N + n] = (T)a2;
}

// ---- interpolation + advection ------------------------------------------------

// The part of a tile's bin that work group b takes: the tiles that
// k_spread_box shares out are shared out here too, their vertices in equal
// parts, the extra parts first.  False (for the whole group) without any.
__device__ __forceinline__ bool tile_part(int b, const int *__restrict__ order, const int2 *__restrict__ extra,
                                          int maxextra, const int *__restrict__ tile_count,
                                          const int *__restrict__ tile_off, int &tile, int &cnt, int &off) {
    int chunk = 0;
    if (b < maxextra) {
        const int2 ex = extra[b];
        if (ex.x < 0) return false;
        tile = ex.x;
        chunk = ex.y;
    } else {
        tile = order[b - maxextra];
    }
    const int all = tile_count[tile];
    if (all == 0) return false;
    const int nch = spread_chunks(all), first = (int)((long long)all * chunk / nch);
    cnt = (int)((long long)all * (chunk + 1) / nch) - first;
    off = tile_off[tile] + first;
    return true;
}

// Velocity box staged per tile: the tile plus 1 node below and 4 above on
// every axis.  The first stencil node of a home vertex lies in the tile, an
// RK stage moves it by less than one node in practice (|u| M dt << dx), and
// the stencil spans 4 nodes; stages that leave the box read global memory.
constexpr int RX = TILE_X + 5, RY = TILE_Y + 5, RZ = TILE_Z + 5, RN = RX * RY * RZ;
constexpr int RLO = 1;  // nodes of the box below the tile
constexpr int INTERP_WG = 256;  // work-group size of k_interp_tiles (a tile of the suspension holds 300 vertices)

// Out-of-line and not unrolled: it is the rare path, and inlining it into
// every RK stage would multiply the kernel's code size.
template <typename T>
__device__ __forceinline__ void interp_global(const T *__restrict__ U, size_t N, const IbmGeom &g, double x,
                                           double y, double z, bool unit, T &ur, T &vr, T &wr) {
    int x1, y1, z1;
    T wx[4], wy[4], wz[4];
    stencil3<T>(g, x, y, z, unit, x1, y1, z1, wx, wy, wz);
    ur = vr = wr = T(0);
#pragma unroll 1
    for (int kz = 0; kz < 4; kz++) {
        int iz = z1 + kz;
        if (!wrap_index(iz, g.nz)) continue;
#pragma unroll 1
        for (int ky = 0; ky < 4; ky++) {
            int iy = y1 + ky;
            if (g.walls) {
                if (iy < 0 || iy >= g.ny) continue;
            } else if (!wrap_index(iy, g.ny)) continue;
#pragma unroll 1
            for (int kx = 0; kx < 4; kx++) {
                int ix = x1 + kx;
                if (!wrap_index(ix, g.nx)) continue;
                const T dlt = wx[kx] * wy[ky] * wz[kz] * T(1.0 / 64.0);
                const size_t n = (size_t)ix + (size_t)g.nx * ((size_t)iy + (size_t)g.ny * iz);
                ur += dlt * U[n];
                vr += dlt * U[N + n];
                wr += dlt * U[2 * N + n];
            }
        }
    }
}

struct AdvectArgs {
    double dt, M;
    double lx, ly, lz;
    int rk;
    int periodic_y;
};

// Four consecutive values of one stencil row, read with one (unaligned)
// wide load.
template <typename T> struct Row4 {
    T v[4];
} __attribute__((aligned(sizeof(T))));

// The interpolated velocity inside one lattice cell.  With t = frac(X/h) the
// four weights of an axis are 1 - s, 1 + c, 1 + s, 1 - c (s, c = sin, cos of
// pi t / 2), so a row contributes (u0+u1+u2+u3) + s (u2-u0) + c (u1-u3), and the
// 64 stencil nodes reduce to 27 coefficients per component of the products of
// (1, s, c) along the axes.  They depend on the cell alone: the RK stages move a
// vertex by a small part of a cell, so one reading of the 192 node values
// serves all four stages almost always, and a stage takes 78 FMAs instead of
// 272.  What bounded both forms was the VALU (2700 instructions per vertex, now
// 2100) and the reads (768 LDS values per vertex, or 48 rows per stage).  Per
// launch before and after, the form that each size takes: 64 cells of 2562
// vertices (FP32) 65 -> 29.6 us, 32 such cells 46 -> 27, 384 uneven cells in
// FP64 245 -> 147, the 1024-cell suspension (FP32) 212 -> 214: there the VALU
// is busy for two thirds of the launch either way, and reading the velocity
// from one XCD's L2 (872 -> 244 MB fetched, tile rows kept on one XCD) gained
// nothing against the heavy-first order.
template <typename T> struct CellField {
    int x1, y1, z1;  // first stencil node of the cell (unpadded)
    T a[3][27];      // [component][z][y][x], over (1, s, c) each
    // fetch(kx-row of 4 values, ky, kz, component)
    template <typename Fetch> __device__ __forceinline__ void load(Fetch fetch) {
#pragma unroll
        for (int d = 0; d < 3; d++) {
            T *o = a[d];
#pragma unroll
            for (int kz = 0; kz < 4; kz++) {
                T r[4][3];
#pragma unroll
                for (int ky = 0; ky < 4; ky++) {
                    T u[4];
                    fetch(u, ky, kz, d);
                    r[ky][0] = (u[0] + u[2]) + (u[1] + u[3]);
                    r[ky][1] = u[2] - u[0];
                    r[ky][2] = u[1] - u[3];
                }
#pragma unroll
                for (int m = 0; m < 3; m++) {
                    const T y[3] = {(r[0][m] + r[2][m]) + (r[1][m] + r[3][m]), r[2][m] - r[0][m], r[1][m] - r[3][m]};
#pragma unroll
                    for (int l = 0; l < 3; l++) {
                        const int k = 3 * l + m;
                        if (kz == 0) { o[k] = y[l]; o[9 + k] = -y[l]; }
                        if (kz == 1) { o[k] += y[l]; o[18 + k] = y[l]; }
                        if (kz == 2) { o[k] += y[l]; o[9 + k] += y[l]; }
                        if (kz == 3) { o[k] += y[l]; o[18 + k] -= y[l]; }
                    }
                }
                // one slice's loads at a time: all 192 in flight would take
                // the registers of two more waves
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    __device__ __forceinline__ void at(const T sn[3], const T cs[3], T &ur, T &vr, T &wr) const {
        T v[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            T z[3];
#pragma unroll
            for (int k = 0; k < 3; k++) {
                T y[3];
#pragma unroll
                for (int l = 0; l < 3; l++) {
                    const T *q = a[d] + 9 * k + 3 * l;
                    y[l] = fma(cs[0], q[2], fma(sn[0], q[1], q[0]));
                }
                z[k] = fma(cs[1], y[2], fma(sn[1], y[1], y[0]));
            }
            v[d] = fma(cs[2], z[2], fma(sn[2], z[1], z[0])) * T(1.0 / 64.0);
        }
        ur = v[0]; vr = v[1]; wr = v[2];
    }
    // sum_d k_d times the gradient of component d; kf = pi / (2 h) turns the
    // derivatives (0, c, -s) of (1, s, c) into those along the position
    __device__ __forceinline__ void grad(const T k[3], const T sn[3], const T cs[3], T kf, T out[3]) const {
        T V[3], DX[3], DY[3];
#pragma unroll
        for (int z = 0; z < 3; z++) {
            T vx[3], dx[3];
#pragma unroll
            for (int l = 0; l < 3; l++) {
                T b[3];
#pragma unroll
                for (int m = 0; m < 3; m++) {
                    const int q = 9 * z + 3 * l + m;
                    b[m] = fma(k[2], a[2][q], fma(k[1], a[1][q], k[0] * a[0][q]));
                }
                vx[l] = fma(cs[0], b[2], fma(sn[0], b[1], b[0]));
                dx[l] = fma(cs[0], b[1], -(sn[0] * b[2]));
            }
            V[z] = fma(cs[1], vx[2], fma(sn[1], vx[1], vx[0]));
            DX[z] = fma(cs[1], dx[2], fma(sn[1], dx[1], dx[0]));
            DY[z] = fma(cs[1], vx[1], -(sn[1] * vx[2]));
        }
        const T q = kf * T(1.0 / 64.0);
        out[0] = q * fma(cs[2], DX[2], fma(sn[2], DX[1], DX[0]));
        out[1] = q * fma(cs[2], DY[2], fma(sn[2], DY[1], DY[0]));
        out[2] = q * fma(cs[2], V[1], -(sn[2] * V[2]));
    }
    // load() from a field [3][N] in memory; every active lane of the wave calls it
    __device__ __forceinline__ void load_field(const T *__restrict__ U, size_t N, const IbmGeom &g, const int f[3]) {
        x1 = f[0]; y1 = f[1]; z1 = f[2];
        const bool whole = __all(f[0] >= 0 && f[0] + 3 < g.nx);
        int ixw[4];
        bool okx[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            ixw[k] = f[0] + k;
            okx[k] = wrap_index(ixw[k], g.nx);
        }
        load([&](T *o, int ky, int kz, int d) {
            int iy = f[1] + ky, iz = f[2] + kz;
            const bool ok = wrap_index(iz, g.nz) && (g.walls ? (iy >= 0 && iy < g.ny) : wrap_index(iy, g.ny));
            // a row outside the lattice holds 0
            const size_t row = ok ? d * N + (size_t)g.nx * ((size_t)iy + (size_t)g.ny * iz) : 0;
            if (whole) {  // one (unaligned) wide load
                const Row4<T> r = *(const Row4<T> *)(U + row + f[0]);
#pragma unroll
                for (int kx = 0; kx < 4; kx++) o[kx] = ok ? r.v[kx] : T(0);
            } else {  // a row of the wave wraps in x
#pragma unroll
                for (int kx = 0; kx < 4; kx++) o[kx] = ok && okx[kx] ? U[row + (okx[kx] ? ixw[kx] : 0)] : T(0);
            }
        });
    }
    // whether a lane of the wave is in another cell than the one loaded
    __device__ __forceinline__ bool left(const int f[3]) const { return __any(f[0] != x1 || f[1] != y1 || f[2] != z1); }
};

// First stencil node (unpadded, unwrapped) and sine and cosine of the
// fractions of a position (as stencil3).
template <typename W>
__device__ __forceinline__ void cell_of(const IbmGeom &g, double x, double y, double z, bool unit, int f[3], W sn[3],
                                        W cs[3]) {
    const double X[3] = {x, y, z};
    const int np[3] = {g.nxp, g.nyp, g.nzp};
#pragma unroll
    for (int d = 0; d < 3; d++) {
        // RK2 / Euler branches use unit spacing (ibm.cu:524-551, 581-608)
        const double q = unit ? X[d] + (double)(np[d] - 1) / 2.0 : over_h(X[d] + (double)(np[d] - 1) * g.dx / 2.0, g.dx);
        const double fl = floor(q);
        f[d] = (int)fl - 3;
        sincos_quarter((W)(q - fl), &sn[d], &cs[d]);
    }
}

// The RK stages of vertex j (ibm.cu:430-517, 524-551, 581-608) with the
// interpolation ip(stage, x, y, z, unit, u, v, w), then the periodic wrap of the new
// position (ibm.cu:616-632) and its stores.  (xn, yn, zn) is the vertex's
// position; xo may be the array that it was read from (each vertex is read
// before it is written, by the same thread).
template <typename T, typename Interp>
__device__ __forceinline__ void advect_vertex(int j, double xn, double yn, double zn, double *xo, T *__restrict__ uvw,
                                              double *__restrict__ xd, int nv, const AdvectArgs &a, Interp ip) {
    const double M = a.M, dt = a.dt;
    const bool unit = a.rk != 4;
    // stage s is taken at X + k_{s-1} (M dt/2, M dt/2, M dt) for RK4 and
    // X + k_1 M for RK2, each offset evaluated as (k M) dt / 2 in that order;
    // the stage sum is (k1 + 2 k2 + 2 k3 + k4)/6, (k1 + k2)/2, k1.  One loop
    // keeps a single inlined copy of the interpolation.
    const int ns = a.rk == 4 ? 4 : (a.rk == 2 ? 2 : 1);
    T ku = T(0), kv = T(0), kw = T(0), su = T(0), sv = T(0), sw = T(0);
#pragma unroll 1
    for (int s = 0; s < ns; s++) {
        double ox = 0.0, oy = 0.0, oz = 0.0;
        if (s > 0) {
            ox = (double)ku * M; oy = (double)kv * M; oz = (double)kw * M;
            if (a.rk == 4) {
                ox *= dt; oy *= dt; oz *= dt;
                if (s < 3) { ox /= 2.0; oy /= 2.0; oz /= 2.0; }
            }
        }
        ip(s, xn + ox, yn + oy, zn + oz, unit, ku, kv, kw);
        const T wt = (a.rk == 4 && (s == 1 || s == 2)) ? T(2) : T(1);
        su += wt * ku; sv += wt * kv; sw += wt * kw;
    }
    const T den = a.rk == 4 ? T(6) : (a.rk == 2 ? T(2) : T(1));
    const T um = su / den, vm = sv / den, wm = sw / den;
    double xr = xn + (double)um * M * dt, yr = yn + (double)vm * M * dt, zr = zn + (double)wm * M * dt;
    if (xr < -a.lx / 2.0) xr += a.lx;
    if (xr > a.lx / 2.0) xr -= a.lx;
    if (zr < -a.lz / 2.0) zr += a.lz;
    if (zr > a.lz / 2.0) zr -= a.lz;
    if (a.periodic_y) {
        if (yr < -a.ly / 2.0) yr += a.ly;
        if (yr > a.ly / 2.0) yr -= a.ly;
    }
    if (uvw) { uvw[j] = um; uvw[nv + j] = vm; uvw[2 * (size_t)nv + j] = wm; }
    xo[j] = xr; xo[nv + j] = yr; xo[2 * (size_t)nv + j] = zr;
    xd[3 * (size_t)j] = xr; xd[3 * (size_t)j + 1] = yr; xd[3 * (size_t)j + 2] = zr;
}

// Interpolation form 0: one work group per tile stages the tile's velocity
// plus halo in LDS once and runs its home vertices from there.
template <typename T>
__global__ __launch_bounds__(INTERP_WG, sizeof(T) == 4 ? 3 : 2) void k_interp_tiles(const T *__restrict__ U, const double *xin, double *xo,
                                                      T *__restrict__ uvw, double *__restrict__ xd,
                                                      const int *__restrict__ tile_count,
                                                      const int *__restrict__ tile_off,
                                                      const int *__restrict__ home_list, int nv, IbmGeom g,
                                                      TileGeom tg, AdvectArgs a, const int *__restrict__ order,
                                                      const int2 *__restrict__ extra, int maxextra) {
    extern __shared__ double dyn[];
    T *Us = (T *)dyn;  // [3][RZ][RY][RX]
    int tile, cnt, off;
    if (!tile_part((int)blockIdx.x, order, extra, maxextra, tile_count, tile_off, tile, cnt, off)) return;
    const int tx = tile % tg.ntx, ty = (tile / tg.ntx) % tg.nty, tz = tile / (tg.ntx * tg.nty);
    const int bx = tx * TILE_X - RLO, by = ty * TILE_Y - RLO, bz = tz * TILE_Z - RLO;
    const size_t N = (size_t)g.nx * g.ny * g.nz;
    // the first vertex's position, read while the box is staged
    int id = 0;
    double x[3] = {0.0, 0.0, 0.0};
    if ((int)threadIdx.x < cnt) {
        id = home_list[off + threadIdx.x];
#pragma unroll
        for (int d = 0; d < 3; d++) x[d] = xin[d * (size_t)nv + id];
    }
    // 16 lanes per box row of 13 nodes, four rows at a time so that their
    // loads are in flight together
    static_assert(RX <= 16, "a row per 16 lanes");
    const bool small = min(min(g.nx, g.nz), g.walls ? RY : g.ny) < RX;  // the box may span an axis more than once
    const int rx = threadIdx.x & 15;
    int ix = bx + rx;
    if (small) ix = pmod(ix, g.nx);
    else wrap_index(ix, g.nx);
    constexpr int ROWS = INTERP_WG / 16, AHEAD = 4;
    for (int row0 = threadIdx.x >> 4; row0 < RY * RZ; row0 += AHEAD * ROWS) {
        T v[AHEAD][3];
#pragma unroll
        for (int j = 0; j < AHEAD; j++) {
            const int row = row0 + j * ROWS;
            int iy = by + row % RY, iz = bz + row / RY;
            bool ok = row < RY * RZ && rx < RX;
            if (small) iz = pmod(iz, g.nz);
            else wrap_index(iz, g.nz);
            if (g.walls) ok = ok && iy >= 0 && iy < g.ny;
            else if (small) iy = pmod(iy, g.ny);
            else wrap_index(iy, g.ny);
            const size_t n = ok ? (size_t)ix + (size_t)g.nx * ((size_t)iy + (size_t)g.ny * iz) : 0;
#pragma unroll
            for (int d = 0; d < 3; d++) v[j][d] = ok ? U[d * N + n] : T(0);
        }
#pragma unroll
        for (int j = 0; j < AHEAD; j++) {
            const int row = row0 + j * ROWS;
            if (row < RY * RZ && rx < RX)
#pragma unroll
                for (int d = 0; d < 3; d++) Us[d * RN + rx + RX * row] = v[j][d];
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < cnt; i += INTERP_WG) {
        // FP32: the next vertex's position while this one moves (FP64 has no
        // registers for it)
        const bool ahead = sizeof(T) == 4;
        if (!ahead && i >= INTERP_WG) {
            id = home_list[off + i];
#pragma unroll
            for (int d = 0; d < 3; d++) x[d] = xin[d * (size_t)nv + id];
        }
        const int j = id;
        const double xn = x[0], yn = x[1], zn = x[2];
        if (ahead && i + INTERP_WG < cnt) {
            id = home_list[off + i + INTERP_WG];
#pragma unroll
            for (int d = 0; d < 3; d++) x[d] = xin[d * (size_t)nv + id];
        }
        CellField<T> cf;
        bool out = false;
        advect_vertex<T>(j, xn, yn, zn, xo, uvw, xd, nv, a,
                         [&](int stage, double x, double y, double z, bool unit, T &u, T &v, T &w) {
                             int f[3];
                             T sn[3], cs[3];
                             cell_of<T>(g, x, y, z, unit, f, sn, cs);
                             // the whole wave reads again when one of its lanes left its cell
                             // (a lane's own branch would keep both sets of coefficients)
                             if (__any(stage == 0 || f[0] != cf.x1 || f[1] != cf.y1 || f[2] != cf.z1)) {
                                 cf.x1 = f[0]; cf.y1 = f[1]; cf.z1 = f[2];
                                 int rx = f[0] - bx, ry = f[1] - by, rz = f[2] - bz;
                                 if (rx < 0) rx += g.nx; else if (rx >= g.nx) rx -= g.nx;
                                 if (rz < 0) rz += g.nz; else if (rz >= g.nz) rz -= g.nz;
                                 if (!g.walls) { if (ry < 0) ry += g.ny; else if (ry >= g.ny) ry -= g.ny; }
                                 out = rx < 0 || rx + 3 >= RX || ry < 0 || ry + 3 >= RY || rz < 0 || rz + 3 >= RZ;
                                 const T *row = Us + (out ? 0 : rx + RX * (ry + RY * rz));
                                 cf.load([&](T *o, int ky, int kz, int d) {
#pragma unroll
                                     for (int kx = 0; kx < 4; kx++) o[kx] = row[d * RN + RX * (ky + RY * kz) + kx];
                                 });
                             }
                             if (out) {  // not in the box: from memory
                                 interp_global<T>(U, N, g, x, y, z, unit, u, v, w);
                                 return;
                             }
                             cf.at(sn, cs, u, v, w);
                         });
    }
}

// Interpolation form 1: one thread per vertex in bin order (neighbouring
// lanes read neighbouring rows), rows read from the field through the caches.
template <typename T>
__global__ __launch_bounds__(256) void k_interp_vert(const T *__restrict__ U, const double *xin, double *xo,
                                                     T *__restrict__ uvw, double *__restrict__ xd,
                                                     const int *__restrict__ home_list, int nv, IbmGeom g,
                                                     AdvectArgs a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nv) return;
    const size_t N = (size_t)g.nx * g.ny * g.nz;
    const int j = home_list[i];
    CellField<T> cf;
    advect_vertex<T>(j, xin[j], xin[nv + j], xin[2 * (size_t)nv + j], xo, uvw, xd, nv, a,
                     [&](int stage, double x, double y, double z, bool unit, T &u, T &v, T &w) {
                         int f[3];
                         T sn[3], cs[3];
                         cell_of<T>(g, x, y, z, unit, f, sn, cs);
                         if (stage == 0 || cf.left(f)) cf.load_field(U, N, g, f);
                         cf.at(sn, cs, u, v, w);
                     });
}

// Interpolation point by point (lbmibm_ctx::pointwise): FP32 products summed in
// the order of the stencil, from row(kz, ky, component, kx).
template <typename Row>
__device__ __forceinline__ void point_sum(const float wx[4], const float wy[4], const float wz[4], float &ur,
                                          float &vr, float &wr, Row row) {
    ur = vr = wr = 0.0f;
#pragma unroll
    for (int kz = 0; kz < 4; kz++) {
        const float wz64 = wz[kz] * (1.0f / 64.0f);
#pragma unroll
        for (int ky = 0; ky < 4; ky++) {
            const float wyz = wy[ky] * wz64;
#pragma unroll
            for (int kx = 0; kx < 4; kx++) {
                const float dlt = wx[kx] * wyz;
                ur = fmaf(dlt, row(kz, ky, 0, kx), ur);
                vr = fmaf(dlt, row(kz, ky, 1, kx), vr);
                wr = fmaf(dlt, row(kz, ky, 2, kx), wr);
            }
        }
    }
}

// Form 0: one work group per tile of TILE_XW nodes stages its velocity box in
// LDS, and every stage reads its 64 nodes from there.  Form 1 (k_interp_points)
// takes less on a few thousand vertices, which fill few tiles (64 cells of 2562: 43
// instead of 88 us), this one on many (the 1024-cell suspension: 221 instead of
// 410 us); both are timed at creation.  Stencils that leave the box read memory,
// with the same products in the same order: the two forms give the same bits.
constexpr int PX = TILE_XW + 5, PN = PX * RY * RZ;
constexpr int POINT_WG = 512;
__global__ __launch_bounds__(POINT_WG) void k_interp_point_tiles(
    const float *__restrict__ U, const double *xin, double *xo, float *__restrict__ uvw, double *__restrict__ xd,
    const int *__restrict__ tile_count, const int *__restrict__ tile_off, const int *__restrict__ home_list, int nv,
    IbmGeom g, TileGeom tg, AdvectArgs a, const int *__restrict__ order) {
    __shared__ float Us[3 * PN];  // [3][RZ][RY][PX]
    const int tile = order[blockIdx.x];
    const int cnt = tile_count[tile], off = tile_off[tile];
    if (cnt == 0) return;  // whole work group leaves together
    const int tx = tile % tg.ntx, ty = (tile / tg.ntx) % tg.nty, tz = tile / (tg.ntx * tg.nty);
    const int bx = tx * TILE_XW - RLO, by = ty * TILE_Y - RLO, bz = tz * TILE_Z - RLO;
    const size_t N = (size_t)g.nx * g.ny * g.nz;
    for (int k = threadIdx.x; k < PN; k += POINT_WG) {
        const int rx = k % PX, ry = (k / PX) % RY, rz = k / (PX * RY);
        // the box may span an axis more than once on small lattices
        const int ix = pmod(bx + rx, g.nx), iz = pmod(bz + rz, g.nz);
        int iy = by + ry;
        const bool ok = !g.walls || (iy >= 0 && iy < g.ny);
        if (!g.walls) iy = pmod(iy, g.ny);
        const size_t n = ok ? (size_t)ix + (size_t)g.nx * ((size_t)iy + (size_t)g.ny * iz) : 0;
#pragma unroll
        for (int d = 0; d < 3; d++) Us[d * PN + k] = ok ? U[d * N + n] : 0.0f;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < cnt; i += POINT_WG) {
        const int j = home_list[off + i];
        advect_vertex<float>(
            j, xin[j], xin[nv + j], xin[2 * (size_t)nv + j], xo, uvw, xd, nv, a,
            [&](int, double x, double y, double z, bool unit, float &ur, float &vr, float &wr) {
                int x1, y1, z1;
                float wx[4], wy[4], wz[4];
                stencil3<float>(g, x, y, z, unit, x1, y1, z1, wx, wy, wz);
                int rx = x1 - bx, ry = y1 - by, rz = z1 - bz;
                if (rx < 0) rx += g.nx; else if (rx >= g.nx) rx -= g.nx;
                if (rz < 0) rz += g.nz; else if (rz >= g.nz) rz -= g.nz;
                if (!g.walls) { if (ry < 0) ry += g.ny; else if (ry >= g.ny) ry -= g.ny; }
                if (rx >= 0 && rx <= PX - 4 && ry >= 0 && ry <= RY - 4 && rz >= 0 && rz <= RZ - 4) {
                    const float *box = Us + rx + PX * (ry + RY * rz);
                    point_sum(wx, wy, wz, ur, vr, wr,
                              [&](int kz, int ky, int d, int kx) { return box[d * PN + PX * (ky + RY * kz) + kx]; });
                    return;
                }
                ur = vr = wr = 0.0f;
#pragma unroll 1
                for (int kz = 0; kz < 4; kz++) {
                    int iz = z1 + kz;
                    if (!wrap_index(iz, g.nz)) continue;
                    const float wz64 = sel4(wz, kz) * (1.0f / 64.0f);
#pragma unroll 1
                    for (int ky = 0; ky < 4; ky++) {
                        int iy = y1 + ky;
                        if (!(g.walls ? iy >= 0 && iy < g.ny : wrap_index(iy, g.ny))) continue;
                        const float wyz = sel4(wy, ky) * wz64;
                        const float *u = U + (size_t)g.nx * ((size_t)iy + (size_t)g.ny * iz);
#pragma unroll 1
                        for (int kx = 0; kx < 4; kx++) {
                            int ix = x1 + kx;
                            if (!wrap_index(ix, g.nx)) continue;
                            const float dlt = sel4(wx, kx) * wyz;
                            ur = fmaf(dlt, u[ix], ur);
                            vr = fmaf(dlt, u[N + ix], vr);
                            wr = fmaf(dlt, u[2 * N + ix], wr);
                        }
                    }
                }
            });
    }
}

// Form 1: a lane keeps the 192 values of its cell, which the stages nearly
// always share, and work groups of one wave spread a few vertices over the chip
// (3204 of them: 25 us, 33 from tiles in LDS, 47 with the rows of a z plane read
// again by every stage).
__global__ __launch_bounds__(64) void k_interp_points(const float *__restrict__ U, const double *xin, double *xo,
                                                      float *__restrict__ uvw, double *__restrict__ xd,
                                                      const int *__restrict__ home_list, int nv, IbmGeom g,
                                                      AdvectArgs a) {
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i >= nv) return;
    const size_t N = (size_t)g.nx * g.ny * g.nz;
    const int j = home_list[i];
    float r[4][4][3][4];  // kz, ky, component, kx; 0 beyond the lattice
    int xl = 0, yl = 0, zl = 0;
    advect_vertex<float>(
        j, xin[j], xin[nv + j], xin[2 * (size_t)nv + j], xo, uvw, xd, nv, a,
        [&](int stage, double x, double y, double z, bool unit, float &ur, float &vr, float &wr) {
            int x1, y1, z1;
            float wx[4], wy[4], wz[4];
            stencil3<float>(g, x, y, z, unit, x1, y1, z1, wx, wy, wz);
            if (__any(stage == 0 || x1 != xl || y1 != yl || z1 != zl)) {
                xl = x1; yl = y1; zl = z1;
                const bool whole = __all(x1 >= 0 && x1 + 3 < g.nx);
                int ix[4];
                bool okx[4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    ix[k] = x1 + k;
                    okx[k] = wrap_index(ix[k], g.nx);
                }
#pragma unroll
                for (int kz = 0; kz < 4; kz++) {
                    int iz = z1 + kz;
                    const bool okz = wrap_index(iz, g.nz);
#pragma unroll
                    for (int ky = 0; ky < 4; ky++) {
                        int iy = y1 + ky;
                        const bool ok = okz && (g.walls ? iy >= 0 && iy < g.ny : wrap_index(iy, g.ny));
                        const float *u = U + (ok ? (size_t)g.nx * ((size_t)iy + (size_t)g.ny * iz) : 0);
#pragma unroll
                        for (int d = 0; d < 3; d++) {
                            if (whole) {  // one (unaligned) wide load
                                const Row4<float> q = *(const Row4<float> *)(u + d * N + x1);
#pragma unroll
                                for (int kx = 0; kx < 4; kx++) r[kz][ky][d][kx] = ok ? q.v[kx] : 0.0f;
                            } else {
#pragma unroll
                                for (int kx = 0; kx < 4; kx++)
                                    r[kz][ky][d][kx] = ok && okx[kx] ? u[d * N + (okx[kx] ? ix[kx] : 0)] : 0.0f;
                            }
                        }
                    }
                }
            }
            point_sum(wx, wy, wz, ur, vr, wr, [&](int kz, int ky, int d, int kx) { return r[kz][ky][d][kx]; });
        });
}

// ---- adjoints (vector-Jacobian products) ------------------------------------
//
// The delta weights are C^1 in the position: with t = frac(xtr/h) the four
// weights are (1 - sin, 1 + cos, 1 + sin, 1 - cos)(pi t/2), and their
// derivatives (pi/2h) (-cos, -sin, cos, sin)(pi t/2) agree at t = 0 and 1
// with those of the neighbouring stencil, so the stencil switch adds no term.
// The spread adjoint is a gather over each vertex's 4x4x4 stencil in global
// memory (one thread per vertex).  The advection adjoint gathers for the
// position terms the same way, and adds the velocity adjoint to the nodes
// per tile in LDS (k_advect_adj_scatter).

// Adjoint of ibm_st1 at the current positions and nodal forces: given Fa (the
// adjoint of the lattice force), cfa = sum D Fa is the adjoint of the nodal
// force and xa += sum (Fa . f) grad D that of the position, D = phi^3/dx^3.
template <typename T>
__global__ __launch_bounds__(256) void k_spread_adj(const double *__restrict__ xs, const T *__restrict__ cf,
                                                    const T *__restrict__ Fa, T *__restrict__ cfa,
                                                    double *__restrict__ xa, int nv, IbmGeom g) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nv) return;
    const size_t N = (size_t)g.nx * g.ny * g.nz;
    const T f0[3] = {cf[j], cf[nv + j], cf[2 * (size_t)nv + j]};
    CellField<T> field;
    int f[3];
    T sn[3], cs[3], b[3], x[3];
    cell_of<T>(g, xs[j], xs[nv + j], xs[2 * (size_t)nv + j], false, f, sn, cs);
    field.load_field(Fa, N, g, f);
    field.at(sn, cs, b[0], b[1], b[2]);
    field.grad(f0, sn, cs, (T)(M_PI / (2.0 * g.dx)), x);
    const T w = (T)(1.0 / (g.dx * g.dx * g.dx));  // both carry the 1/64
#pragma unroll
    for (int d = 0; d < 3; d++) {
        cfa[(size_t)d * nv + j] = b[d] * w;
        xa[(size_t)d * nv + j] += (double)(x[d] * w);
    }
}

// Adjoint of ibm_st2 with RK4 at the current positions and velocity field:
// xa holds the adjoint of the advected positions on entry and that of the
// current positions on exit; the adjoint of the velocity field is added to
// ua.  The stage positions are recomputed; stage s contributes
// ua += phi^3(X_s) kb_s and X_s-bar = sum (u . kb_s) grad phi^3, which feeds
// the stage before it (ibm.cu:430-517: X2 = X + h/2 k1, X3 = X + h/2 k2,
// X4 = X + h k3, X' = X + h (k1 + 2 k2 + 2 k3 + k4)/6, h = M dt).
// Two kernels.  k_advect_adj_vert, one lane per vertex in bin order, does
// the gathers (the stage positions, X-bar) and writes each stage's position
// and kb_s to a record; k_advect_adj_scatter, one work group per tile over
// its home vertices, adds the velocity adjoint of the records.

template <typename T> struct AdvRec {
    double p[3];  // stage position
    T k[3];       // kb_s
};

// One lane per vertex (bin order), the velocity and its gradient from the
// coefficients of its cell (CellField), which the four stages nearly always
// share.  Four lanes per vertex with a z-slice each, which read the 64 nodes
// for every stage's velocity and again for its gradient, took 108 us on 32
// cells of 2562 vertices; this takes 57.
template <typename T>
__global__ __launch_bounds__(256) void k_advect_adj_vert(const double *__restrict__ xs, const T *__restrict__ U,
                                                         double *__restrict__ xa, const int *__restrict__ home_list,
                                                         int nv, IbmGeom g, double h, AdvRec<T> *__restrict__ rec,
                                                         unsigned *__restrict__ kbmax) {
    __shared__ float shm[4];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;  // vertex in bin order
    float km = 0.0f;
    if (i < nv) {
        const int j = home_list[i];
        const size_t N = (size_t)g.nx * g.ny * g.nz;
        const double X[3] = {xs[j], xs[nv + j], xs[2 * (size_t)nv + j]};
        CellField<T> cf;
        int f[3];
        T sn[3], cs[3];
        double P[4][3], back[4] = {0.0, h / 2.0, h / 2.0, h};  // X_s = X + back[s] k_{s-1}
#pragma unroll
        for (int d = 0; d < 3; d++) P[0][d] = X[d];
#pragma unroll
        for (int s = 0; s < 3; s++) {
            cell_of<T>(g, P[s][0], P[s][1], P[s][2], false, f, sn, cs);
            if (s == 0 || cf.left(f)) cf.load_field(U, N, g, f);
            T k[3];
            cf.at(sn, cs, k[0], k[1], k[2]);
#pragma unroll
            for (int d = 0; d < 3; d++) P[s + 1][d] = X[d] + (s < 2 ? (double)k[d] * h / 2.0 : (double)k[d] * h);
        }
        const double xb[3] = {xa[j], xa[nv + j], xa[2 * (size_t)nv + j]};
        double acc[3] = {xb[0], xb[1], xb[2]}, next[3] = {0.0, 0.0, 0.0};
        const double cw[4] = {h / 6.0, h / 3.0, h / 3.0, h / 6.0};
        const T kf = (T)(M_PI / (2.0 * g.dx));
#pragma unroll
        for (int s = 3; s >= 0; s--) {  // kb_s = cw[s] xb + back[s + 1] X_{s+1}-bar
            AdvRec<T> r;
#pragma unroll
            for (int d = 0; d < 3; d++) {
                r.p[d] = P[s][d];
                r.k[d] = (T)(cw[s] * xb[d] + next[d]);
            }
            rec[4 * (size_t)i + s] = r;
            km += fmaxf(fabsf((float)r.k[0]), fmaxf(fabsf((float)r.k[1]), fabsf((float)r.k[2])));
            cell_of<T>(g, P[s][0], P[s][1], P[s][2], false, f, sn, cs);
            if (cf.left(f)) cf.load_field(U, N, g, f);
            T gr[3];
            cf.grad(r.k, sn, cs, kf, gr);
#pragma unroll
            for (int d = 0; d < 3; d++) {
                acc[d] += (double)gr[d];
                next[d] = back[s] * (double)gr[d];
            }
        }
        xa[j] = acc[0];
        xa[nv + j] = acc[1];
        xa[2 * (size_t)nv + j] = acc[2];
        km *= 1.0001f;  // margin for the float rounding
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) km = fmaxf(km, __shfl_xor(km, o));
    if ((threadIdx.x & 63) == 0) shm[threadIdx.x >> 6] = km;
    __syncthreads();
    // non-negative floats order as their bit patterns: an integer maximum
    if (threadIdx.x == 0) atomicMax(kbmax, __float_as_uint(fmaxf(fmaxf(shm[0], shm[1]), fmaxf(shm[2], shm[3]))));
}

// One work group per tile takes its home vertices (the bins of the
// interpolation) and adds ua += sum_s phi^3(X_s) kb_s / 64 into an LDS box
// of the tile plus its halo (the staging box of k_interp_tiles), then adds
// the box to ua with one global atomic per node; stencils that leave the box
// add to ua directly.  The four stage stencils of a vertex nearly always
// start at the same node (the stages move it by h |u| << 1): then the four
// terms are summed per node and added once.  Lane l of wave w takes column
// 8l + w of the part read as 512 columns, so the lanes of a wave hold vertices
// far apart, whose nodes rarely coincide (LDS atomics to one address
// serialise).  FP32 accumulates in 64-bit fixed point, as the spreading
// (raw bits of fma(v, scale, 1.5 2^52), whose low 48 bits sum exactly), with
// the scale from the bound cnt max_v sum_s |kb_s| / 8 of a node's sum (a
// weight product is at most 8/64); FP64 uses FP64 LDS atomics.  On 32 cells
// of 2562 vertices: 130 us with 16x8x8 tiles and a work group per tile, 54 us
// with 8x8x8 tiles and full ones shared out.
constexpr int ADV_WG = 512;  // work-group size of k_advect_adj_scatter

template <typename T>
__global__ __launch_bounds__(ADV_WG) void k_advect_adj_scatter(const AdvRec<T> *__restrict__ rec, T *__restrict__ ua,
                                                            const int *__restrict__ tile_count,
                                                            const int *__restrict__ tile_off, IbmGeom g,
                                                            TileGeom tg, const unsigned *__restrict__ kbmax,
                                                            const int *__restrict__ order,
                                                            const int2 *__restrict__ extra, int maxextra) {
    extern __shared__ double dyn[];
    constexpr bool FIX = sizeof(T) == 4;
    unsigned long long *Ub = (unsigned long long *)dyn;  // [3][RZ][RY][RX]
    double *Ud = dyn;
    int tile, cnt, off;
    if (!tile_part((int)blockIdx.x, order, extra, maxextra, tile_count, tile_off, tile, cnt, off)) return;
    const int tx = tile % tg.ntx, ty = (tile / tg.ntx) % tg.nty, tz = tile / (tg.ntx * tg.nty);
    const int bx = tx * TILE_X - RLO, by = ty * TILE_Y - RLO, bz = tz * TILE_Z - RLO;
    const size_t N = (size_t)g.nx * g.ny * g.nz;
    double scale = 1.0;
    if (FIX) {
        const double km = (double)__uint_as_float(*kbmax);
        if (km > 0.0) scale = ldexp(1.0, 46 - ilogb((double)cnt * km / 8.0));
    }
    for (int k = threadIdx.x; k < 3 * RN; k += blockDim.x) Ub[k] = 0ull;
    __syncthreads();
    const T q64 = T(1.0 / 64.0);
    constexpr int NW = ADV_WG / 64;
    const int R = (cnt + ADV_WG - 1) / ADV_WG;
    const int col = NW * (threadIdx.x & 63) + (threadIdx.x >> 6);
    for (int r = 0; r < R; r++) {
        const int i = col * R + r;
        if (i >= cnt) break;
        int x1[4], y1[4], z1[4];
        T wx[4][4], wy[4][4], wz[4][4], kk[4][3];
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const AdvRec<T> rr = rec[4 * (size_t)(off + i) + s];
            stencil3<T>(g, rr.p[0], rr.p[1], rr.p[2], false, x1[s], y1[s], z1[s], wx[s], wy[s], wz[s]);
            kk[s][0] = rr.k[0] * q64; kk[s][1] = rr.k[1] * q64; kk[s][2] = rr.k[2] * q64;
        }
        bool same = true;
#pragma unroll
        for (int s = 1; s < 4; s++) same = same && x1[s] == x1[0] && y1[s] == y1[0] && z1[s] == z1[0];
        // one walk of the common stencil with all four stages, or one walk per
        // stage with the other stages masked out
        const int ns = same ? 1 : 4;
        for (int it = 0; it < ns; it++) {
            T m[4];
            int sx = x1[0], sy = y1[0], sz = z1[0];
#pragma unroll
            for (int s = 0; s < 4; s++) {
                m[s] = (same || s == it) ? T(1) : T(0);
                if (!same && s == it) { sx = x1[s]; sy = y1[s]; sz = z1[s]; }
            }
            // box coordinates of the first stencil node (as interp_tile)
            int rx = sx - bx, ry = sy - by, rz = sz - bz;
            if (rx < 0) rx += g.nx; else if (rx >= g.nx) rx -= g.nx;
            if (rz < 0) rz += g.nz; else if (rz >= g.nz) rz -= g.nz;
            if (!g.walls) { if (ry < 0) ry += g.ny; else if (ry >= g.ny) ry -= g.ny; }
            const bool inbox = rx >= 0 && rx + 3 < RX && ry >= 0 && ry + 3 < RY && rz >= 0 && rz + 3 < RZ;
#pragma unroll 1
            for (int kz = 0; kz < 4; kz++) {
                int iz = sz + kz;
                if (!wrap_index(iz, g.nz)) continue;
                T cz[4][3];  // mask * kb_s/64 * wz_s
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    const T w = m[s] * sel4(wz[s], kz);
                    cz[s][0] = w * kk[s][0]; cz[s][1] = w * kk[s][1]; cz[s][2] = w * kk[s][2];
                }
#pragma unroll
                for (int ky = 0; ky < 4; ky++) {
                    int iy = sy + ky;
                    if (g.walls) {
                        if (iy < 0 || iy >= g.ny) continue;
                    } else if (!wrap_index(iy, g.ny)) continue;
                    T cy[4][3];
#pragma unroll
                    for (int s = 0; s < 4; s++)
#pragma unroll
                        for (int d = 0; d < 3; d++) cy[s][d] = wy[s][ky] * cz[s][d];
#pragma unroll
                    for (int kx = 0; kx < 4; kx++) {
                        int ix = sx + kx;
                        if (!wrap_index(ix, g.nx)) continue;
                        const size_t n = (size_t)ix + (size_t)g.nx * ((size_t)iy + (size_t)g.ny * iz);
                        const int bi = (rx + kx) + RX * ((ry + ky) + RY * (rz + kz));
                        T v0 = T(0), v1 = T(0), v2 = T(0);
#pragma unroll
                        for (int s = 0; s < 4; s++) {
                            v0 += wx[s][kx] * cy[s][0]; v1 += wx[s][kx] * cy[s][1]; v2 += wx[s][kx] * cy[s][2];
                        }
                        // into the box when the stencil lies in it, else into ua (written
                        // out here: the LDS atomics must see the LDS pointer itself)
                        if (inbox) {
                            if (FIX) {
                                const double big = 6755399441055744.0;  // 1.5 2^52
                                atomicAdd(Ub + bi,
                                          (unsigned long long)__double_as_longlong(fma((double)v0, scale, big)));
                                atomicAdd(Ub + RN + bi,
                                          (unsigned long long)__double_as_longlong(fma((double)v1, scale, big)));
                                atomicAdd(Ub + 2 * RN + bi,
                                          (unsigned long long)__double_as_longlong(fma((double)v2, scale, big)));
                            } else {
                                atomicAdd(Ud + bi, (double)v0);
                                atomicAdd(Ud + RN + bi, (double)v1);
                                atomicAdd(Ud + 2 * RN + bi, (double)v2);
                            }
                        } else {
                            atomicAdd(&ua[n], v0);
                            atomicAdd(&ua[N + n], v1);
                            atomicAdd(&ua[2 * N + n], v2);
                        }
                    }
                }
            }
        }
    }
    __syncthreads();
    // the box into ua (the box may wrap onto itself on small lattices: atomics)
    const double inv_scale = 1.0 / scale;
    for (int k = threadIdx.x; k < RN; k += blockDim.x) {
        auto val = [&](int i) {
            return FIX ? (T)((double)((long long)(Ub[i] << 16) >> 16) * inv_scale) : (T)Ud[i];
        };
        const T a0 = val(k), a1 = val(RN + k), a2 = val(2 * RN + k);
        if (a0 == T(0) && a1 == T(0) && a2 == T(0)) continue;
        const int rx = k % RX, ry = (k / RX) % RY, rz = k / (RX * RY);
        const int ix = pmod(bx + rx, g.nx), iz = pmod(bz + rz, g.nz);
        int iy = by + ry;
        if (g.walls) {
            if (iy < 0 || iy >= g.ny) continue;
        } else {
            iy = pmod(iy, g.ny);
        }
        const size_t n = (size_t)ix + (size_t)g.nx * ((size_t)iy + (size_t)g.ny * iz);
        atomicAdd(&ua[n], a0);
        atomicAdd(&ua[N + n], a1);
        atomicAdd(&ua[2 * N + n], a2);
    }
}

IbmGeom geom_of(const lbmibm_ctx *ctx) {
    IbmGeom g;
    g.nx = ctx->nx; g.ny = ctx->ny; g.nz = ctx->nz;
    g.nxp = ctx->nxp; g.nyp = ctx->nyp; g.nzp = ctx->nzp;
    g.walls = ctx->p.periodic_y == 0;
    g.dx = ctx->p.dx;
    return g;
}

static TileGeom tiles_of(const lbmibm_ctx *ctx) { return {ctx->ntx, ctx->nty, ctx->ntz, ctx->ntiles, ctx->tile_x}; }

BinGeom bin_geom(const lbmibm_ctx *ctx) {
    BinGeom b;
    b.nx = ctx->nx; b.ny = ctx->ny; b.nz = ctx->nz;
    b.nxp = ctx->nxp; b.nyp = ctx->nyp; b.nzp = ctx->nzp;
    b.walls = ctx->p.periodic_y == 0;
    b.ntx = ctx->ntx; b.nty = ctx->nty;
    b.tx = ctx->tile_x;
    b.dx = ctx->p.dx;
    return b;
}

// The offsets and orders of the tiles from their counts (k_tile_scan with no
// force maxima).
lbmibm_status tile_offsets(lbmibm_ctx *ctx, hipStream_t stream, int nblk_fmax) {
    const IbmGeom g = geom_of(ctx);
    const TileGeom tg = tiles_of(ctx);
    hipLaunchKernelGGL((ctx->spread_form == 0 ? k_tile_scan<true> : k_tile_scan<false>), dim3(1), dim3(1024), 0, stream, ctx->tile_count, ctx->tile_off, ctx->tile_cur,
                       ctx->ntiles, ctx->blk_fmax, nblk_fmax, ctx->absmax, ctx->tile_ex, ctx->sb_extra,
                       ctx->sb_maxextra, g, tg, ctx->tile_cand, ctx->order_spread, ctx->order_interp,
                       ctx->order_calls);
    LBMIBM_LAUNCHED(ctx, "k_tile_scan");
    return LBMIBM_OK;
}

// The scatter of the binning: home list, first stencil nodes and spreading
// records (fractions, current forces) in bin order.
template <typename T> lbmibm_status bin_scatter(lbmibm_ctx *ctx, hipStream_t stream) {
    hipLaunchKernelGGL(k_bin_scatter<T>, dim3(ctx->nblk_bin), dim3(BIN_WG), 0, stream, (const double *)ctx->xs,
                       (const T *)spread_force(ctx), ctx->home, ctx->nv, geom_of(ctx), ctx->tile_off, ctx->tile_cur,
                       ctx->home_list, ctx->node0, (SpreadRec<T> *)ctx->srec);
    LBMIBM_LAUNCHED(ctx, "k_bin_scatter");
    return LBMIBM_OK;
}

// Binning of the vertices by the tile of their first stencil node, with the
// spreading records of the current nodal forces and max |f|.
template <typename T> lbmibm_status bin_impl(lbmibm_ctx *ctx) {
    hipStream_t stream = ctx->stream;
    const int nv = ctx->nv;
    const hipEvent_t kt = kt_begin(ctx, stream);
    hipLaunchKernelGGL(k_zero_int, dim3((ctx->ntiles + 255) / 256), dim3(256), 0, stream, ctx->tile_count,
                       ctx->ntiles);
    LBMIBM_LAUNCHED(ctx, "k_zero_int");
    hipLaunchKernelGGL(k_bin_count<T>, dim3(ctx->nblk_bin), dim3(BIN_WG), 0, stream, (const double *)ctx->xs,
                       (const T *)spread_force(ctx), nv, bin_geom(ctx), ctx->home, ctx->tile_count, ctx->blk_fmax);
    LBMIBM_LAUNCHED(ctx, "k_bin_count");
    lbmibm_status s = tile_offsets(ctx, stream, ctx->nblk_bin);
    if (s == LBMIBM_OK) s = bin_scatter<T>(ctx, stream);
    if (s != LBMIBM_OK) return s;
    kt_end(ctx, stream, "binning", kt);
    ctx->bins_valid = true;
    ctx->counts_ready = false;
    return LBMIBM_OK;
}

// The spreading of the binned records into F with the given form.
template <typename T> lbmibm_status spread_launch(lbmibm_ctx *ctx, int form) {
    const TileGeom tg = tiles_of(ctx);
    const IbmGeom g = geom_of(ctx);
    if (form == 1) {
        if (ctx->pointwise) {
            LBMIBM_KT(ctx, ctx->stream, "k_spread_points",
                      hipLaunchKernelGGL(k_spread_points, dim3(ctx->ntiles), dim3(SPREAD_BOX_WG), 0, ctx->stream,
                                         (const SpreadRec<float> *)ctx->srec, ctx->node0, ctx->tile_count,
                                         ctx->tile_off, (float *)ctx->sbox, g, tg, ctx->order_interp));
            LBMIBM_LAUNCHED(ctx, "k_spread_points");
        } else {
            LBMIBM_KT(ctx, ctx->stream, "k_spread_box",
                      hipLaunchKernelGGL(k_spread_box<T>, dim3(ctx->sb_maxextra + ctx->ntiles), dim3(SPREAD_BOX_WG), 0,
                                         ctx->stream,
                                         (const SpreadRec<T> *)ctx->srec, ctx->node0, ctx->home_list, ctx->tile_count,
                                         ctx->tile_off, (T *)ctx->sbox, g, tg, ctx->order_interp, ctx->sb_extra,
                                         ctx->sb_maxextra, ctx->tile_ex, (ChunkBox *)ctx->sb_chunks));
            LBMIBM_LAUNCHED(ctx, "k_spread_box");
            if (ctx->sb_maxextra > 0) {
                LBMIBM_KT(ctx, ctx->stream, "k_spread_combine",
                          hipLaunchKernelGGL(k_spread_combine<T>, dim3(ctx->sb_maxextra, COMBINE_PARTS),
                                             dim3(COMBINE_WG), 0, ctx->stream, (T *)ctx->sbox,
                                             (ChunkBox *)ctx->sb_chunks, ctx->sb_extra, ctx->tile_count,
                                             ctx->sb_maxextra));
                LBMIBM_LAUNCHED(ctx, "k_spread_combine");
            }
        }
        constexpr int XW = sizeof(T) == 4 ? TILE_XW : TILE_X;
        LBMIBM_KT(ctx, ctx->stream, "k_spread_gather",
                  hipLaunchKernelGGL((ctx->pointwise ? k_spread_gather<T, XW> : k_spread_gather<T, TILE_X>),
                                     dim3((unsigned)xcd_grid((int)((ctx->N + 255) / 256))), dim3(256), 0,
                                     ctx->stream, (const T *)ctx->sbox, ctx->tile_count, ctx->sb_cand,
                                     ctx->sb_cand + SB_MAXC * ctx->nx, ctx->sb_cand + SB_MAXC * (ctx->nx + ctx->ny),
                                     (T *)ctx->F, g, tg));
        LBMIBM_LAUNCHED(ctx, "k_spread_gather");
        return LBMIBM_OK;
    }
    LBMIBM_KT(ctx, ctx->stream, "k_spread_tiles",
              hipLaunchKernelGGL(k_spread_tiles<T>, dim3(ctx->ntiles), dim3(256), 0, ctx->stream,
                                 (const SpreadRec<T> *)ctx->srec, ctx->node0, ctx->tile_count, ctx->tile_off,
                                 (T *)ctx->F, g, tg, ctx->absmax, ctx->order_spread));
    LBMIBM_LAUNCHED(ctx, "k_spread_tiles");
    return LBMIBM_OK;
}

template <typename T> lbmibm_status spread_impl(lbmibm_ctx *ctx) {
    if (ctx->nv == 0) return lattice_fill(ctx, ctx->F, 3 * (size_t)ctx->N, 0.0, false);
    if (!ctx->bins_valid && ctx->counts_ready && ctx->spread_form == 1) {
        // counted with the volume correction: only the scatter is left (form 1
        // scales each tile by its own max |f| and needs no global maximum)
        const hipEvent_t kt = kt_begin(ctx, ctx->stream);
        lbmibm_status s = bin_scatter<T>(ctx, ctx->stream);
        if (s != LBMIBM_OK) return s;
        kt_end(ctx, ctx->stream, "binning", kt);
        ctx->bins_valid = true;
        ctx->counts_ready = false;
    } else if (!ctx->bins_valid) {
        lbmibm_status s = bin_impl<T>(ctx);
        if (s != LBMIBM_OK) return s;
    } else {  // same positions, new forces: refresh the force part of the records
        hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(64), 0, ctx->stream, (int *)ctx->absmax, 1);
        LBMIBM_LAUNCHED(ctx, "k_zero_int");
        hipLaunchKernelGGL(k_bin_forces<T>, dim3((ctx->nv + 255) / 256), dim3(256), 0, ctx->stream, ctx->home_list,
                           (const T *)spread_force(ctx), ctx->nv, (SpreadRec<T> *)ctx->srec, ctx->absmax);
        LBMIBM_LAUNCHED(ctx, "k_bin_forces");
    }
    return spread_launch<T>(ctx, ctx->spread_form);
}

// One interpolation + advection of all vertices with the given form, from
// xin into xo / xd (uvw may be null).
template <typename T>
lbmibm_status interp_launch(lbmibm_ctx *ctx, int form, const double *xin, double *xo, T *uvw, double *xd) {
    AdvectArgs a;
    a.dt = ctx->p.dt; a.M = ctx->p.m;
    a.lx = ctx->nx * ctx->p.dx; a.ly = ctx->ny * ctx->p.dx; a.lz = ctx->nz * ctx->p.dx;
    a.rk = ctx->p.runge_kutta;
    a.periodic_y = ctx->p.periodic_y;
    if (ctx->pointwise && form == 0) {
        LBMIBM_KT(ctx, ctx->stream, "k_interp_point_tiles",
                  hipLaunchKernelGGL(k_interp_point_tiles, dim3(ctx->ntiles), dim3(POINT_WG), 0, ctx->stream,
                                     (const float *)ctx->U, xin, xo, (float *)uvw, xd, ctx->tile_count, ctx->tile_off,
                                     ctx->home_list, ctx->nv, geom_of(ctx), tiles_of(ctx), a, ctx->order_interp));
        LBMIBM_LAUNCHED(ctx, "k_interp_point_tiles");
        return LBMIBM_OK;
    }
    if (ctx->pointwise) {
        LBMIBM_KT(ctx, ctx->stream, "k_interp_points",
                  hipLaunchKernelGGL(k_interp_points, dim3((ctx->nv + 63) / 64), dim3(64), 0, ctx->stream,
                                     (const float *)ctx->U, xin, xo, (float *)uvw, xd, ctx->home_list, ctx->nv,
                                     geom_of(ctx), a));
        LBMIBM_LAUNCHED(ctx, "k_interp_points");
        return LBMIBM_OK;
    }
    if (form == 1) {
        LBMIBM_KT(ctx, ctx->stream, "k_interp_vert",
                  hipLaunchKernelGGL(k_interp_vert<T>, dim3((ctx->nv + 255) / 256), dim3(256), 0, ctx->stream,
                                     (const T *)ctx->U, xin, xo, uvw, xd, ctx->home_list, ctx->nv, geom_of(ctx), a));
        LBMIBM_LAUNCHED(ctx, "k_interp_vert");
        return LBMIBM_OK;
    }
    const TileGeom tg = tiles_of(ctx);
    const size_t lds = 3 * (size_t)RN * sizeof(T);
    LBMIBM_KT(ctx, ctx->stream, "k_interp_tiles",
              hipLaunchKernelGGL(k_interp_tiles<T>, dim3(ctx->sb_maxextra + ctx->ntiles), dim3(INTERP_WG), lds, ctx->stream,
                                 (const T *)ctx->U, xin, xo, uvw, xd, ctx->tile_count, ctx->tile_off, ctx->home_list,
                                 ctx->nv, geom_of(ctx), tg, a, ctx->order_interp, ctx->sb_extra, ctx->sb_maxextra));
    LBMIBM_LAUNCHED(ctx, "k_interp_tiles");
    return LBMIBM_OK;
}

template <typename T> lbmibm_status interp_impl(lbmibm_ctx *ctx) {
    if (ctx->nv == 0) return LBMIBM_OK;
    if (!ctx->bins_valid) {
        lbmibm_status s = bin_impl<T>(ctx);
        if (s != LBMIBM_OK) return s;
    }
    double *xo = ctx->xs_out ? ctx->xs_out : (double *)ctx->xs;
    lbmibm_status s = interp_launch<T>(ctx, ctx->interp_form, (const double *)ctx->xs, xo,
                                       ctx->p.store_macros ? (T *)ctx->uvw : (T *)nullptr, (double *)ctx->xd);
    invalidate_bins(ctx);  // the positions moved
    return s;
}

// Times the interpolation forms on the current positions and velocity field,
// writing to scratch arrays (the vertices do not move), and keeps the faster.
template <typename T> lbmibm_status interp_autotune_impl(lbmibm_ctx *ctx) {
    if (!ctx->bins_valid) {
        lbmibm_status s = bin_impl<T>(ctx);
        if (s != LBMIBM_OK) return s;
    }
    double *xo = nullptr, *xd = nullptr;
    const size_t bytes = 3 * (size_t)ctx->nv * sizeof(double);
    LBMIBM_HIP(ctx, hipMalloc((void **)&xo, bytes));
    if (hipMalloc((void **)&xd, bytes) != hipSuccess) {
        (void)hipFree(xo);
        return LBMIBM_ERR_HIP;
    }
    hipEvent_t e0 = nullptr, e1 = nullptr;
    lbmibm_status s = LBMIBM_OK;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) s = LBMIBM_ERR_HIP;
    static const char *names[2] = {"tiles in LDS", "rows from memory"};
    char line[160];
    float best = 0.0f;
    for (int f = 0; f < 2 && s == LBMIBM_OK; f++) {
        s = interp_launch<T>(ctx, f, (const double *)ctx->xs, xo, (T *)nullptr, xd);  // warm-up
        if (s != LBMIBM_OK) break;
        if (hipEventRecord(e0, ctx->stream) != hipSuccess) { s = LBMIBM_ERR_HIP; break; }
        for (int r = 0; r < 3 && s == LBMIBM_OK; r++)
            s = interp_launch<T>(ctx, f, (const double *)ctx->xs, xo, (T *)nullptr, xd);
        float ms = 0.0f;
        if (s == LBMIBM_OK && (hipEventRecord(e1, ctx->stream) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
                               hipEventElapsedTime(&ms, e0, e1) != hipSuccess))
            s = LBMIBM_ERR_HIP;
        if (s != LBMIBM_OK) break;
        ms /= 3.0f;
        snprintf(line, sizeof line, "interp form %s: %.4f ms\n", names[f], ms);
        ctx->tune_report += line;
        if (f == 0 || ms < best) { best = ms; ctx->interp_form = f; }
    }
    if (s == LBMIBM_OK) {
        snprintf(line, sizeof line, "interp: using %s\n", names[ctx->interp_form]);
        ctx->tune_report += line;
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipFree(xo);
    (void)hipFree(xd);
    return s;
}

template <typename T> lbmibm_status spread_adj_impl(lbmibm_ctx *ctx) {
    if (ctx->nv == 0) return LBMIBM_OK;
    hipLaunchKernelGGL(k_spread_adj<T>, dim3((ctx->nv + 255) / 256), dim3(256), 0, ctx->stream,
                       (const double *)ctx->xs, (const T *)ctx->cf, (const T *)ctx->adj_F, (T *)ctx->adj_cf,
                       ctx->adj_x, ctx->nv, geom_of(ctx));
    LBMIBM_LAUNCHED(ctx, "k_spread_adj");
    return LBMIBM_OK;
}

template <typename T> lbmibm_status advect_adj_impl(lbmibm_ctx *ctx) {
    if (ctx->nv == 0) return LBMIBM_OK;
    if (!ctx->bins_valid) {
        lbmibm_status s = bin_impl<T>(ctx);
        if (s != LBMIBM_OK) return s;
    }
    hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(64), 0, ctx->stream, (int *)ctx->adj_xmax, 1);
    LBMIBM_LAUNCHED(ctx, "k_zero_int");
    const IbmGeom g = geom_of(ctx);
    hipLaunchKernelGGL(k_advect_adj_vert<T>, dim3((ctx->nv + 255) / 256), dim3(256), 0,
                       ctx->stream,
                       (const double *)ctx->xs, (const T *)ctx->U, ctx->adj_x, ctx->home_list, ctx->nv, g,
                       ctx->p.m * ctx->p.dt, (AdvRec<T> *)ctx->adj_rec, ctx->adj_xmax);
    LBMIBM_LAUNCHED(ctx, "k_advect_adj_vert");
    const TileGeom tg = tiles_of(ctx);
    const size_t lds = 3 * (size_t)RN * sizeof(unsigned long long);
    hipLaunchKernelGGL(k_advect_adj_scatter<T>, dim3(ctx->sb_maxextra + ctx->ntiles), dim3(ADV_WG), lds, ctx->stream,
                       (const AdvRec<T> *)ctx->adj_rec, (T *)ctx->adj_u, ctx->tile_count, ctx->tile_off, g, tg,
                       ctx->adj_xmax, ctx->order_interp, ctx->sb_extra, ctx->sb_maxextra);
    LBMIBM_LAUNCHED(ctx, "k_advect_adj_scatter");
    return LBMIBM_OK;
}

}  // namespace

lbmibm_status ibm_spread_adjoint(lbmibm_ctx *ctx) {
    return ctx->prec == LBMIBM_F64 ? spread_adj_impl<double>(ctx) : spread_adj_impl<float>(ctx);
}

lbmibm_status ibm_interp_adjoint(lbmibm_ctx *ctx) {
    if (ctx->p.runge_kutta != 4) {
        ctx->err = "adjoint: the advection adjoint supports RUNGE_KUTTA = 4";
        return LBMIBM_ERR_STATE;
    }
    return ctx->prec == LBMIBM_F64 ? advect_adj_impl<double>(ctx) : advect_adj_impl<float>(ctx);
}

lbmibm_status ibm_setup(lbmibm_ctx *ctx) {
    // extra chunks: at most nv / SB_CHUNK over all tiles
    ctx->sb_maxextra = ctx->pointwise ? 0 : xcd_grid(ctx->nv / SB_CHUNK);  // whole rounds of the XCDs
    lbmibm_status s = dev_alloc(ctx, (void **)&ctx->tile_ex, (size_t)ctx->ntiles * sizeof(int));
    if (s == LBMIBM_OK) s = dev_alloc(ctx, (void **)&ctx->sb_extra, (size_t)ctx->sb_maxextra * sizeof(int2));
    if (s != LBMIBM_OK) return s;
    const int lds64 = (int)(3 * (size_t)RN * sizeof(double));
    const int lds32 = (int)(3 * (size_t)RN * sizeof(float));
    LBMIBM_HIP(ctx, hipFuncSetAttribute((const void *)k_interp_tiles<double>,
                                        hipFuncAttributeMaxDynamicSharedMemorySize, lds64));
    LBMIBM_HIP(ctx, hipFuncSetAttribute((const void *)k_interp_tiles<float>,
                                        hipFuncAttributeMaxDynamicSharedMemorySize, lds32));
    LBMIBM_HIP(ctx, hipFuncSetAttribute((const void *)k_advect_adj_scatter<double>,
                                        hipFuncAttributeMaxDynamicSharedMemorySize, lds64));
    LBMIBM_HIP(ctx, hipFuncSetAttribute((const void *)k_advect_adj_scatter<float>,
                                        hipFuncAttributeMaxDynamicSharedMemorySize, lds64));
    return LBMIBM_OK;
}

lbmibm_status ibm_count_end(lbmibm_ctx *ctx, hipStream_t stream) { return tile_offsets(ctx, stream, 0); }

lbmibm_status ibm_spread(lbmibm_ctx *ctx) {
    lbmibm_status s = ctx->prec == LBMIBM_F64 ? spread_impl<double>(ctx) : spread_impl<float>(ctx);
    if (s == LBMIBM_OK) ctx->force_zero = (ctx->nv == 0);
    return s;
}

// Host tables of spread form 1: for each coordinate of each axis, the
// (tile along the axis, box coordinate) pairs whose box node lands on it,
// tiles ascending; false when a coordinate has more than SB_MAXC (lattices
// much smaller than a box) or the tile counts do not fit the packing.
static bool spread_box_tables(const lbmibm_ctx *ctx, std::vector<int> &out) {
    const int n[3] = {ctx->nx, ctx->ny, ctx->nz}, nt[3] = {ctx->ntx, ctx->nty, ctx->ntz};
    const int tile[3] = {ctx->tile_x, TILE_Y, TILE_Z}, R[3] = {ctx->tile_x + 3, SB_Y, SB_Z};
    const bool wrap[3] = {true, ctx->p.periodic_y != 0, true};
    // boxes of TILE_XW + 3 nodes meet rows of four more than SB_MAXC times; with
    // those of TILE_X + 3 such lattices stay without the form, which they never had
    if (n[0] < 5) return false;
    out.assign((size_t)SB_MAXC * (n[0] + n[1] + n[2]), -1);
    size_t base = 0;
    for (int a = 0; a < 3; a++) {
        if (nt[a] >= (1 << 25)) return false;
        for (int t = 0; t < nt[a]; t++)
            for (int k = 0; k < R[a]; k++) {
                int cc = t * tile[a] + k;
                if (cc >= n[a]) {
                    if (!wrap[a]) continue;
                    cc %= n[a];
                }
                int *e = &out[base + (size_t)SB_MAXC * cc];
                int slot = 0;
                while (slot < SB_MAXC && e[slot] >= 0) slot++;
                if (slot == SB_MAXC) return false;
                e[slot] = t * 32 + k;
            }
        base += (size_t)SB_MAXC * n[a];
    }
    return true;
}

// Allocates the staging boxes and uploads the tables of spread form 1;
// *ok = false where the form does not apply.
static lbmibm_status spread_box_setup(lbmibm_ctx *ctx, bool *ok) {
    *ok = false;
    std::vector<int> tab;
    if (!spread_box_tables(ctx, tab)) return LBMIBM_OK;
    if (!ctx->sb_cand) {
        lbmibm_status s = dev_alloc(ctx, (void **)&ctx->sb_cand, tab.size() * sizeof(int));
        if (s != LBMIBM_OK) return s;
        LBMIBM_HIP(ctx, hipMemcpy(ctx->sb_cand, tab.data(), tab.size() * sizeof(int), hipMemcpyHostToDevice));
    }
    if (!ctx->sbox) {
        lbmibm_status s = dev_alloc(ctx, &ctx->sbox, (size_t)ctx->ntiles * 3 * (ctx->pointwise ? SP_N : SB_N) * ctx->szT);
        if (s == LBMIBM_OK && ctx->sb_maxextra > 0)
            s = dev_alloc(ctx, &ctx->sb_chunks, 2 * (size_t)ctx->sb_maxextra * (sizeof(ChunkBox) + sizeof(double)));
        if (s != LBMIBM_OK) return s;
    }
    *ok = true;
    return LBMIBM_OK;
}

// Times the spreading forms on the binned initial positions (the force
// field they write is overwritten by the first step) and keeps the faster.
template <typename T> lbmibm_status spread_autotune_impl(lbmibm_ctx *ctx) {
    if (!ctx->bins_valid) {
        lbmibm_status s = bin_impl<T>(ctx);
        if (s != LBMIBM_OK) return s;
    }
    hipEvent_t e0 = nullptr, e1 = nullptr;
    lbmibm_status s = LBMIBM_OK;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) s = LBMIBM_ERR_HIP;
    static const char *names[2] = {"source bins per tile", "home boxes + gather"};
    char line[160];
    float best = 0.0f;
    for (int f = 0; f < 2 && s == LBMIBM_OK; f++) {
        s = spread_launch<T>(ctx, f);  // warm-up
        if (s != LBMIBM_OK) break;
        if (hipEventRecord(e0, ctx->stream) != hipSuccess) { s = LBMIBM_ERR_HIP; break; }
        for (int r = 0; r < 3 && s == LBMIBM_OK; r++) s = spread_launch<T>(ctx, f);
        float ms = 0.0f;
        if (s == LBMIBM_OK && (hipEventRecord(e1, ctx->stream) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
                               hipEventElapsedTime(&ms, e0, e1) != hipSuccess))
            s = LBMIBM_ERR_HIP;
        if (s != LBMIBM_OK) break;
        ms /= 3.0f;
        snprintf(line, sizeof line, "spread form %s: %.4f ms\n", names[f], ms);
        ctx->tune_report += line;
        if (f == 0 || ms < best) { best = ms; ctx->spread_form = f; }
    }
    if (s == LBMIBM_OK) {
        snprintf(line, sizeof line, "spread: using %s\n", names[ctx->spread_form]);
        ctx->tune_report += line;
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    return s;
}

// a form fixed in the environment: "0" .. last into *form, -1 when unset
static lbmibm_status env_form(const char *name, int *form, char last = '1') {
    *form = -1;
    const char *v = getenv(name);
    if (!v || !v[0]) return LBMIBM_OK;
    if (v[0] < '0' || v[0] > last || v[1]) return LBMIBM_ERR_ARG;
    *form = v[0] - '0';
    return LBMIBM_OK;
}

lbmibm_status ibm_autotune(lbmibm_ctx *ctx) {
    ctx->interp_form = 0;
    ctx->spread_form = 0;
    if (ctx->nv == 0) return LBMIBM_OK;
    // LBMIBM_INTERP_FORM / LBMIBM_SPREAD_FORM = 0|1 fix a form;
    // LBMIBM_AUTOTUNE=0 keeps forms 0
    int fi = -1, fs = -1;
    lbmibm_status s = env_form("LBMIBM_INTERP_FORM", &fi);
    if (s == LBMIBM_OK) s = env_form("LBMIBM_SPREAD_FORM", &fs);
    if (s != LBMIBM_OK) return s;
    bool box_ok = false;
    s = spread_box_setup(ctx, &box_ok);
    if (s != LBMIBM_OK) return s;
    if (fs == 1 && !box_ok) return LBMIBM_ERR_ARG;  // the lattice is too small for the boxes
    const char *env = getenv("LBMIBM_AUTOTUNE");
    const bool tune = !(env && env[0] == '0');
    if (fi >= 0) {
        ctx->interp_form = fi;
        ctx->tune_report += "interp form fixed by LBMIBM_INTERP_FORM\n";
    } else if (tune) {
        s = ctx->prec == LBMIBM_F64 ? interp_autotune_impl<double>(ctx) : interp_autotune_impl<float>(ctx);
        if (s != LBMIBM_OK) return s;
    }
    if (fs >= 0) {
        ctx->spread_form = fs;
        ctx->tune_report += "spread form fixed by LBMIBM_SPREAD_FORM\n";
    } else if (tune && box_ok) {
        s = ctx->prec == LBMIBM_F64 ? spread_autotune_impl<double>(ctx) : spread_autotune_impl<float>(ctx);
        if (s != LBMIBM_OK) return s;
    }
    return LBMIBM_OK;
}

lbmibm_status ibm_interp(lbmibm_ctx *ctx) {
    return ctx->prec == LBMIBM_F64 ? interp_impl<double>(ctx) : interp_impl<float>(ctx);
}

}  // namespace lbmibm
