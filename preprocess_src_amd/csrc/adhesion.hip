// Cytoadhesion of cell knobs to wall receptors (adhesion.cu), for the slab
// (CapsuleSHEARFLOW) with the linear spring or WLC law: receptors on the wall
// y = -LY/2 on an nxw x nzw grid (wall_init, adhesion.cu:441-458), knobs
// with springs_per_knob springs, Bell-model attach / detach
// (adhesion.cu:513-615) and the spring force that the spreading adds to the
// membrane force (ibm_st1bb, ibm.cu:133-212).
//
// The reference leaves two things to the hardware; both are fixed here:
//   - random numbers: splitmix64 of (seed, iteration, spring id), one draw
//     per spring per call, mapped to (0, 1] (curand seeded from clock() in
//     the reference);
//   - a receptor wanted by several springs in one call goes to the lowest
//     spring id (vertex * springs_per_knob + spring), the others trying
//     their next candidate, in rounds (an atomicOr race in the reference);
//     the bids are 64-bit keys stamped with the call and round.
// Detachments go first; a spring that detaches does not re-attach in the
// same call (one draw decides either branch in the reference).
#include <algorithm>
#include <climits>
#include <vector>

#include "common.hpp"

namespace lbmibm {
namespace {

constexpr int AWG = 256;

struct AdhDev {
    double rc, k_ad, l0, k_on0, k_off0, chi_beta, kbt, shear_rate, gs;
    int limit, maxn, ns, nxw, nzw;
    double dxw, dzw, lx, ly, lz, dx, dtm;  // dtm = dt M
    unsigned long long seed;
    int nv;
    int wlc;                                      // 0 LINEAR_SPRING, 1 WLC
    double lcont, f_wlc, ra, alpha1, alpha2;
    int ring;                                     // the tube's receptor ring
    double radius;
    const double *ring_xy;                        // [nxw][2]: R cos, R sin of each column (host libm)
    double reach;                                 // angular half-width of the columns within LIMIT dx
};

// Extension measure and force of the Bell rates: LINEAR_SPRING
// (adhesion.cu:562-563) or WLC with LL = Lcont dx (adhesion.cu:564-566).
__device__ __forceinline__ double bell_extension(const AdhDev &a, double r) {
#pragma clang fp contract(off)
    if (a.wlc) {
        const double LL = a.lcont * a.dx;
        return fmax(0.0, 0.25 / ((1.0 - r / LL) * (1.0 - r / LL)) + r / LL - 0.25);
    }
    return fmax(0.0, (r - a.l0 * a.dx) * a.rc);
}
__device__ __forceinline__ double bell_force(const AdhDev &a, double dr) {
    return a.wlc ? fabs(a.f_wlc * dr) : fabs(a.k_ad * dr);
}

__host__ __device__ __forceinline__ double adh_uniform(unsigned long long seed, long long iter, long long sid) {
    // splitmix64 (Steele, Lea, Flood 2014) of the key, mapped to (0, 1]
    unsigned long long z = seed ^ ((unsigned long long)iter * 0x9E3779B97F4A7C15ull) ^
                           ((unsigned long long)sid * 0xD1B54A32D192ED03ull);
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z = z ^ (z >> 31);
    return (double)((z >> 11) + 1) * (1.0 / 9007199254740992.0);
}

// A bid of spring sid in round `round` of the call numbered `call` (a
// device counter that every call advances): later rounds and calls outrank
// every older bid, so claims need no clearing, and within a round the
// lowest spring id is the largest key.
__device__ __forceinline__ unsigned long long bid_key(unsigned long long call, int round, int maxn, int sid) {
    const unsigned long long stamp = call * (unsigned long long)(maxn + 2) + (unsigned)round + 1u;
    return (stamp << 32) | (unsigned long long)(0xFFFFFFFFu - (unsigned)sid);
}

// Advances the call counter (one work group). Stamps must stay below 2^32 (the key keeps 32
// bits of stamp): when the next call's largest stamp would not, every claim
// is cleared and the counter restarts at 0, whose stamps outrank a cleared
// claim. With MAXN = 100 that happens once in about 42 million calls.
__device__ __forceinline__ void advance_calls(unsigned long long *__restrict__ calls,
                                              unsigned long long *__restrict__ claim, long long nrec, int maxn) {
    const unsigned long long next = calls[0] + 1ull;
    const bool wrap = (next + 1ull) * (unsigned long long)(maxn + 2) > 0xFFFFFFFFull;
    if (wrap)
        for (long long i = threadIdx.x; i < nrec; i += blockDim.x) claim[i] = 0ull;
    __syncthreads();
    if (threadIdx.x == 0) calls[0] = wrap ? 0ull : next;
}

// Receptor id = iz * nxw + ix on the slab's wall y = -LY/2 (adhesion.cu:
// 452-457) or on the tube's ring at angle ix * dxw (adhesion.cu:475-490).
__device__ __forceinline__ void receptor(const AdhDev &a, int id, double &x, double &y, double &z) {
    const int iz = id / a.nxw, ix = id - iz * a.nxw;
    if (a.ring) {
        x = a.ring_xy[2 * ix];
        y = a.ring_xy[2 * ix + 1];
    } else {
        x = (ix - a.nxw / 2) * a.dxw;
        y = -0.5 * a.ly;
    }
    z = (iz - a.nzw / 2) * a.dzw;
}

__device__ __forceinline__ double image_shift(double d, double L, double xi, double xj) {
    if (fabs(d) > L / 2.0) {  // adhesion.cu:656-668
        if (xi > xj) d += L;
        else if (xi < xj) d -= L;
    }
    return d;
}

__device__ __forceinline__ double p_on(const AdhDev &a, double r, double &dr) {
#pragma clang fp contract(off)
    dr = bell_extension(a, r);  // adhesion.cu:562-573
    const double f_ad = bell_force(a, dr);
    const double k_on = a.k_on0 / a.shear_rate * exp(f_ad * (a.chi_beta - 0.5 * dr) / a.kbt);
    return 1.0 - exp(-k_on * a.dtm);
}

// AdhesiveSpringForce_GPU (adhesion.cu:617-706) and the spreading force
// cf + f_adh of ibm_st1bb.
template <typename T>
__global__ __launch_bounds__(AWG) void k_adh_force(AdhDev a, const double *__restrict__ xs,
                                                   const T *__restrict__ cf, const unsigned char *__restrict__ knob,
                                                   const int *__restrict__ attach, double *__restrict__ f_adh,
                                                   T *__restrict__ fsum) {
#pragma clang fp contract(off)
    const int v = blockIdx.x * AWG + threadIdx.x;
    if (v >= a.nv) return;
    double f[3] = {0.0, 0.0, 0.0};
    if (knob[v]) {
        const double xi = xs[v], yi = xs[a.nv + v], zi = xs[2 * (size_t)a.nv + v];
        // WLC: the repulsive term keeps the previous spring's value where
        // |dy| >= L0 dx, as the reference's variable does (adhesion.cu:677-690)
        double repulf = 0.0;
        for (int s = 0; s < a.ns; s++) {
            const int id = attach[v * a.ns + s];
            if (id == -1) continue;
            double xj, yj, zj;
            receptor(a, id, xj, yj, zj);
            const double dx = a.ring ? xj - xi : image_shift(xj - xi, a.lx, xi, xj), dy = yj - yi;
            const double dz = image_shift(zj - zi, a.lz, zi, zj);
            const double r = sqrt(dx * dx + dy * dy + dz * dz);
            if (a.wlc) {
                const double LL = a.lcont * a.dx;
                const double dr = 0.25 / ((1.0 - r / LL) * (1.0 - r / LL)) + r / LL - 0.25;
                if (fabs(dy) < a.l0 * a.dx) {
                    const double ex = exp(-a.alpha2 * fabs(dy));
                    repulf = a.alpha1 / (a.gs * a.ra) * a.alpha2 * ex / (1.0 - ex) * dy / fabs(dy);
                }
                f[0] += a.f_wlc / (a.gs * a.ra) * dr * dx / r;
                f[1] += a.f_wlc / (a.gs * a.ra) * dr * dy / r + repulf;
                f[2] += a.f_wlc / (a.gs * a.ra) * dr * dz / r;
                continue;
            }
            const double dr = r - a.l0 * a.dx;
            f[0] += a.k_ad / a.gs * dr * dx / r;
            f[1] += a.k_ad / a.gs * dr * dy / r;
            f[2] += a.k_ad / a.gs * dr * dz / r;
        }
    }
    for (int c = 0; c < 3; c++) {
        f_adh[3 * (size_t)v + c] = f[c];
        fsum[c * (size_t)a.nv + v] = (T)((double)cf[c * (size_t)a.nv + v] + f[c]);
    }
}

// StoreNeighWall_CUBE_GPU (adhesion.cu:109-206): receptors within LIMIT dx
// of a knob near the wall, nearest first, ties in scan order, at most MAXN.
// One wave per knob: its lanes test the candidates 64 at a time and list those in
// range in scan order in LDS.  When the list is full it is ranked (for each one, how
// many come before it) and cut to the MAXN nearest, and from then on only
// candidates nearer than the last of them are listed.  One lane per vertex,
// inserting into a sorted list in memory, was a chain of dependent reads for each
// candidate: 63 us for 64 cells with 20 to 40 knobs each, 5 us now.  With 64
// receptors per unit area (more than 256 in range) the lane's insertion took 0.75 ms of
// a step with MAXN = 16 and 4.3 ms with 100; this takes 0.04 and 0.12.
constexpr int SEARCH_CAP = 256;  // entries in LDS per knob; lists that fill them (MAXN > 192) take the insertion by one lane
__global__ __launch_bounds__(AWG) void k_adh_search(AdhDev a, const double *__restrict__ xs,
                                                    const int *__restrict__ klist, int nk, int *__restrict__ id_wall,
                                                    double *__restrict__ r_wall) {
#pragma clang fp contract(off)
    __shared__ double lr[AWG / 64][SEARCH_CAP];
    __shared__ int lid[AWG / 64][SEARCH_CAP];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int t = blockIdx.x * (AWG / 64) + wave;
    if (t >= nk) return;  // whole waves leave; nothing here waits for another wave
    const int v = klist[t];
    int *ids = id_wall + (size_t)v * a.maxn;
    double *rs = r_wall + (size_t)v * a.maxn;
    const double xi = xs[v], yi = xs[a.nv + v], zi = xs[2 * (size_t)a.nv + v];
    const bool away = a.ring ? sqrt(xi * xi + yi * yi) < a.radius - a.limit * a.dx  // adhesion.cu:248-249
                             : sqrt(yi * yi) < 0.5 * a.ly - a.limit * a.dx;
    const int iz = (int)((zi - (-a.lz / 2.0)) / a.dzw);
    const int span = a.limit * (int)(a.dx / a.dzw);
    // Only columns within LIMIT dx can pass the range test: an x window on
    // the slab, an angular window around the knob on the ring (two ranges
    // when it wraps past angle 0). Scanning them in increasing column order,
    // as a scan of every column does, keeps the list and its ties.
    int ra0, ra1, rb0 = 0, rb1 = -1;
    if (a.ring) {
        double t = atan2(yi, xi);
        if (t < 0.0) t += 2.0 * M_PI;
        const int j0 = (int)floor((t - a.reach) / a.dxw) - 1, j1 = (int)ceil((t + a.reach) / a.dxw) + 1;
        if (j1 - j0 + 1 >= a.nxw) { ra0 = 0; ra1 = a.nxw - 1; }
        else if (j0 < 0) { ra0 = 0; ra1 = j1; rb0 = j0 + a.nxw; rb1 = a.nxw - 1; }
        else if (j1 >= a.nxw) { ra0 = 0; ra1 = j1 - a.nxw; rb0 = j0; rb1 = a.nxw - 1; }
        else { ra0 = j0; ra1 = j1; }
    } else {
        ra0 = max(0, (int)floor((xi - a.limit * a.dx) / a.dxw) + a.nxw / 2 - 1);
        ra1 = min(a.nxw - 1, (int)ceil((xi + a.limit * a.dx) / a.dxw) + a.nxw / 2 + 1);
    }
    const int ncol = ra1 - ra0 + 1 + (rb1 - rb0 + 1);
    const int nrow = away || ncol <= 0 ? 0 : 2 * span;
    // candidate (row, col) in scan order; false out of range
    auto candidate = [&](int row, int col, int &id, double &r) {
        int jz = iz + row - (span - 1);
        double zj = (jz - a.nzw / 2) * a.dzw;
        if (jz < 0) { jz += a.nzw; zj += a.lz; }
        else if (jz >= a.nzw) { jz -= a.nzw; zj -= a.lz; }
        if (jz < 0 || jz >= a.nzw) return false;  // more than a period away: LIMIT dx beyond the box
        const int k = ra0 + col, jx = k <= ra1 ? k : rb0 + (k - ra1 - 1);
        id = jz * a.nxw + jx;
        double xj, yj, zr;
        receptor(a, id, xj, yj, zr);
        r = sqrt((xj - xi) * (xj - xi) + (yj - yi) * (yj - yi) + (zj - zi) * (zj - zi));
        return !(r > a.limit * a.dx);
    };
    auto in_step = [] {  // the wave's LDS accesses before, and those after
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    int have = 0;
    auto rank_of = [&](int i) {
        const double r = lr[wave][i];
        int rank = 0;
        for (int j = 0; j < have; j++) rank += j < i ? !(lr[wave][j] > r) : r > lr[wave][j];
        return rank;
    };
    bool full = false, serial = false;
    double worst = 0.0;  // distance of the last of MAXN, where there are so many
    const int nc = max(ncol, 1);
    int row = lane / nc, col = lane % nc;
    while (__any(row < nrow)) {
        int id = 0;
        double r = 0.0;
        const bool in = row < nrow && candidate(row, col, id, r) && !(full && !(worst > r));
        row += 64 / nc;
        col += 64 % nc;
        if (col >= nc) { col -= nc; row++; }
        const unsigned long long m = __ballot(in);
        const int at = have + __popcll(m & ((1ull << lane) - 1ull));
        if (in) { lr[wave][at] = r; lid[wave][at] = id; }
        have += __popcll(m);
        if (have <= SEARCH_CAP - 64) continue;
        if (a.maxn > SEARCH_CAP - 64) {
            serial = true;
            break;
        }
        in_step();
        int to[SEARCH_CAP / 64], ids_[SEARCH_CAP / 64];
        double rs_[SEARCH_CAP / 64];
#pragma unroll
        for (int j = 0; j < SEARCH_CAP / 64; j++) {
            const int i = lane + 64 * j;
            to[j] = a.maxn;
            if (i < have) {
                to[j] = rank_of(i);
                rs_[j] = lr[wave][i];
                ids_[j] = lid[wave][i];
            }
        }
        in_step();
#pragma unroll
        for (int j = 0; j < SEARCH_CAP / 64; j++)
            if (to[j] < a.maxn) { lr[wave][to[j]] = rs_[j]; lid[wave][to[j]] = ids_[j]; }
        in_step();
        have = a.maxn;
        full = true;
        worst = lr[wave][a.maxn - 1];
    }
    if (!serial) {
        in_step();
        for (int k = min(have, a.maxn) + lane; k < a.maxn; k += 64) { ids[k] = -1; rs[k] = 1.0e15; }
        for (int i = lane; i < have; i += 64) {
            const int rank = rank_of(i);
            if (rank < a.maxn) { ids[rank] = lid[wave][i]; rs[rank] = lr[wave][i]; }
        }
    } else if (lane == 0) {
        int cnt = 0;
        for (row = 0; row < nrow; row++)
            for (col = 0; col < ncol; col++) {
                int id;
                double r;
                if (!candidate(row, col, id, r)) continue;
                int pos = cnt;
                while (pos > 0 && rs[pos - 1] > r) pos--;
                if (pos >= a.maxn) continue;
                for (int k = cnt < a.maxn ? cnt : a.maxn - 1; k > pos; k--) { ids[k] = ids[k - 1]; rs[k] = rs[k - 1]; }
                ids[pos] = id;
                rs[pos] = r;
                if (cnt < a.maxn) cnt++;
            }
        for (int k = cnt; k < a.maxn; k++) { ids[k] = -1; rs[k] = 1.0e15; }
    }
}

// Detachment of attached springs (adhesion.cu:584-612, z image only); the
// free springs become the candidates of the attachment rounds.
__global__ __launch_bounds__(AWG) void k_adh_detach(AdhDev a, const double *__restrict__ xs,
                                                    const unsigned char *__restrict__ knob, int *__restrict__ attach,
                                                    double *__restrict__ r_ij, int *__restrict__ is_attached,
                                                    int *__restrict__ pos, int *__restrict__ active,
                                                    const DevStep *__restrict__ st, int init,
                                                    const int *__restrict__ klist, int nk,
                                                    unsigned long long *__restrict__ calls,
                                                    unsigned long long *__restrict__ claim, long long nrec,
                                                    int *__restrict__ more, int *__restrict__ made) {
#pragma clang fp contract(off)
    if (blockIdx.x == 0) {
        advance_calls(calls, claim, nrec, a.maxn);
        if (threadIdx.x < 2) more[threadIdx.x] = 0;
        for (int r = threadIdx.x; r <= a.maxn; r += AWG) made[r] = 0;
    }
    const int t = blockIdx.x * AWG + threadIdx.x;
    if (t >= nk * a.ns) return;
    const int v = klist[t / a.ns], sid = v * a.ns + t % a.ns;
    pos[sid] = 0;
    active[sid] = 0;
    if (!knob[v]) return;
    const int id = attach[sid];
    if (id == -1) {
        active[sid] = 1;
        return;
    }
    if (init) return;
    double xj, yj, zj;
    receptor(a, id, xj, yj, zj);
    const double xi = xs[v], yi = xs[a.nv + v], zi = xs[2 * (size_t)a.nv + v];
    const double dx = xj - xi, dy = yj - yi, dz = image_shift(zj - zi, a.lz, zi, zj);
    const double r = sqrt(dx * dx + dy * dy + dz * dz);
    const double dr = bell_extension(a, r);
    const double f_ad = bell_force(a, dr);
    const double k_off = a.k_off0 / a.shear_rate * exp(f_ad * a.chi_beta / a.kbt);
    const double p_off = 1.0 - exp(-k_off * a.dtm);
    if (p_off <= adh_uniform(a.seed, st->iter, sid)) return;
    is_attached[id] = 0;
    attach[sid] = -1;
    r_ij[sid] = dr;
}

// One attachment round, in two halves.  Each active spring proposes its next
// acceptable free candidate (returned; -1: none) and bids for it with its id.
struct AdhRound {
    const int *id_wall, *klist;
    const double *r_wall;
    int *is_attached, *attach, *pos, *active, *prop;
    double *r_ij;
    unsigned long long *claim;
    const unsigned long long *calls;
    const DevStep *st;
    int init, nk;
    int *more, *list[2];  // [2] springs that go on after round 0, and after the rounds of k_adh_round: numbers, ids
    int *made;            // [maxn + 1] whether a round of k_adh_round had proposals
};
// whether a receptor has a winner already; since_call: it may have one by a bid
// of an earlier round of this call, which nobody has entered yet
__device__ __forceinline__ bool adh_taken(const AdhDev &a, const AdhRound &q, int round, unsigned long long call,
                                          bool since_call, int id) {
    if (q.is_attached[id]) return true;
    if (!since_call) return false;
    const unsigned long long bid = q.claim[id];
    // the smallest keys of round 0 and of this one: those of a spring above all ids
    return bid >= bid_key(call, 0, a.maxn, -1) && bid < bid_key(call, round, a.maxn, -1);
}
__device__ __forceinline__ int adh_propose(const AdhDev &a, const AdhRound &q, int round, unsigned long long call,
                                           int sid, bool since_call = false) {
    const int v = sid / a.ns;
    const double u = q.init ? 0.0 : adh_uniform(a.seed, q.st->iter, sid);
    int c = q.pos[sid], id = -1;
    for (; c < a.maxn; c++) {
        id = q.id_wall[(size_t)v * a.maxn + c];
        if (id == -1) continue;
        if (!q.init) {
            double dr;
            if (p_on(a, q.r_wall[(size_t)v * a.maxn + c], dr) <= u) continue;
        }
        if (adh_taken(a, q, round, call, since_call, id)) continue;
        break;
    }
    if (c >= a.maxn) {
        q.active[sid] = 0;
        return -1;
    }
    q.pos[sid] = c;
    atomicMax(q.claim + id, bid_key(call, round, a.maxn, sid));
    return id;
}
// The highest bid takes the receptor (true), the others go on to their next candidate.
__device__ __forceinline__ bool adh_resolve(const AdhDev &a, const AdhRound &q, int round, unsigned long long call,
                                            int sid, int id) {
    // bids are made in L2: read there
    if (__hip_atomic_load(q.claim + id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
        bid_key(call, round, a.maxn, sid)) {
        q.attach[sid] = id;
        q.is_attached[id] = 1;
        if (!q.init) {
            double dr;
            (void)p_on(a, q.r_wall[(size_t)(sid / a.ns) * a.maxn + q.pos[sid]], dr);
            q.r_ij[sid] = dr;
        }
        q.active[sid] = 0;
        return true;
    }
    q.pos[sid] = q.pos[sid] + 1;
    return false;
}

// Round 0, which meets every free spring: a launch per half.  The losers are
// listed (in any order: the bids decide) for the other rounds.
__global__ __launch_bounds__(AWG) void k_adh_propose(AdhDev a, AdhRound q) {
    const int t = blockIdx.x * AWG + threadIdx.x;
    if (t >= q.nk * a.ns) return;
    const int sid = q.klist[t / a.ns] * a.ns + t % a.ns;
    q.prop[sid] = q.active[sid] ? adh_propose(a, q, 0, *q.calls, sid) : -1;
}
// The lanes' springs that are `on` behind those listed already; whole waves.
__device__ __forceinline__ void adh_append(int *__restrict__ more, int *__restrict__ list, bool on, int sid) {
    const int lane = threadIdx.x & 63;
    const unsigned long long m = __ballot(on);
    if (!m) return;
    int at = 0;
    if (lane == 0) at = atomicAdd(more, __popcll(m));
    at = __shfl(at, 0) + __popcll(m & ((1ull << lane) - 1ull));
    if (on) list[at] = sid;
}
__global__ __launch_bounds__(AWG) void k_adh_resolve(AdhDev a, AdhRound q) {
    const int t = blockIdx.x * AWG + threadIdx.x;
    int sid = 0;
    bool lost = false;
    if (t < q.nk * a.ns) {
        sid = q.klist[t / a.ns] * a.ns + t % a.ns;
        const int id = q.prop[sid];
        lost = id >= 0 && !adh_resolve(a, q, 0, *q.calls, sid, id);
        if (lost) q.prop[sid] = -1;
    }
    adh_append(q.more, q.list[0], lost, sid);
}

// The other rounds, which only the losers of the one before take part in.
// Every spring advances or retires in every round, so MAXN more rounds are
// enough.  Here they run in one work group, which stops after a round without
// proposals: `first` and the later ones of a list (0: the losers of round 0, where
// they are at most `most`; 1: those of the rounds of k_adh_round).
//
// A pair of launches for each of the MAXN + 1 rounds, most of them empty, took 34
// launches and 95 us per step for 64 cells with 40 knobs of 2 springs and
// MAXN = 16 (27 now, 12 of them here).  But a thousand losers are what one CU
// takes in the time of a launch: all rounds in one group took 2.45 ms of a step
// with 363 000 springs and 34.7 ms with 1.8 million (MAXN = 100), 0.50 and 2.2
// in pairs of launches, 0.24 and 1.2 now.  ROUNDS_SPRINGS: with 8100 springs of 16
// per knob, half of them near the wall, and MAXN = 100 the group alone takes 0.17 ms,
// the pairs took 1.5; below, the launches that find nothing to do would cost 20 us
// and more of every step.  Springs of one knob contend for the same receptors round
// after round, so with more of them per knob (ROUNDS_PER_KNOB) the launches are made.
constexpr int ROUNDS_GROUP = 1024;
constexpr int ROUNDS_SPRINGS = 8192, ROUNDS_PER_KNOB = 16;  // springs up to which no other launches are made
constexpr int ROUNDS_MANY = 65536;                          // and above which every round has one
__global__ __launch_bounds__(1024) void k_adh_rounds(AdhDev a, AdhRound q, int which, int first, int most) {
    __shared__ int made;
    const int m = q.more[which];
    const int *list = q.list[which];
    if (m > most) return;
    const unsigned long long call = *q.calls;
    for (int round = first; round <= a.maxn; round++) {
        if (threadIdx.x == 0) made = 0;
        __syncthreads();
        for (int k = threadIdx.x; k < m; k += 1024) {
            const int sid = list[k];
            const int id = q.active[sid] ? adh_propose(a, q, round, call, sid) : -1;
            q.prop[sid] = id;
            if (id >= 0) made = 1;
        }
        __threadfence();  // the bids, before they are read
        __syncthreads();
        if (!made) return;
        for (int k = threadIdx.x; k < m; k += 1024) {
            const int sid = list[k], id = q.prop[sid];
            if (id >= 0) (void)adh_resolve(a, q, round, call, sid, id);
        }
        __syncthreads();
    }
}
// More losers: a launch per round, over the whole chip, for the first few of
// them.  A spring first learns how its bid of the round before ended, then makes
// the next; receptors that somebody won in that round are told by the bids on them,
// whether the winner has entered itself yet or not.  The `last` launch only
// enters the winners, and lists the losers.  Every round up to MAXN has its launch at
// the set-up, where all springs lose at once, and for more than ROUNDS_MANY
// springs (a launch that finds nothing to do costs 2.3 us); otherwise 4 rounds per
// spring of a knob have one, at least 8, and k_adh_rounds takes what is left.  With 8
// rounds always, 1.8 million springs at 400 per knob took 69 ms (10 in pairs of
// launches, 3.0 now), and the set-up of those at 40 per knob 57 ms (9 and 7).
constexpr int ROUND_GROUPS = 512;
__global__ __launch_bounds__(AWG) void k_adh_round(AdhDev a, AdhRound q, int round, bool last, int most) {
    const int m = q.more[0];
    if (m <= most || (round > 1 && q.made[round - 1] == 0)) return;
    const unsigned long long call = *q.calls;
    bool any = false;
    for (int k0 = blockIdx.x * AWG; k0 < m; k0 += ROUND_GROUPS * AWG) {  // whole waves
        const int k = k0 + threadIdx.x;
        const int sid = k < m ? q.list[0][k] : 0;
        bool on = k < m && q.active[sid];
        int id = on ? q.prop[sid] : -1;
        if (id >= 0) on = !adh_resolve(a, q, round - 1, call, sid, id);
        if (last) {
            adh_append(q.more + 1, q.list[1], on, sid);
        } else if (on) {
            id = adh_propose(a, q, round, call, sid, true);
            q.prop[sid] = id;
            any = any || id >= 0;
        }
    }
    if (__any(any) && (threadIdx.x & 63) == 0) q.made[round] = 1;
}

template <typename V> __global__ void k_afill(V *__restrict__ p, size_t n, V v) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

AdhDev adh_dev(const lbmibm_ctx *ctx) {
    const lbmibm_adhesion_params &h = ctx->adh;
    AdhDev a;
    a.rc = h.rc; a.k_ad = h.k_ad; a.l0 = h.l0; a.k_on0 = h.k_on0; a.k_off0 = h.k_off0;
    a.chi_beta = h.chi_beta; a.kbt = h.kbt; a.shear_rate = h.shear_rate; a.gs = h.gs;
    a.limit = h.limit; a.maxn = h.max_neighwall; a.ns = h.springs_per_knob;
    a.nxw = ctx->adh_nxw; a.nzw = ctx->adh_nzw; a.dxw = ctx->adh_dxw; a.dzw = ctx->adh_dzw;
    a.dx = ctx->p.dx;
    a.lx = ctx->p.lx * a.dx; a.ly = ctx->p.ly * a.dx; a.lz = ctx->p.lz * a.dx;
    a.dtm = ctx->p.dt * (double)ctx->p.m;
    a.seed = h.seed;
    a.nv = ctx->nv;
    a.wlc = h.wlc;
    a.lcont = h.lcont; a.f_wlc = h.f_wlc; a.ra = h.ra; a.alpha1 = h.alpha1; a.alpha2 = h.alpha2;
    a.ring = ctx->p.tube_radius > 0.0;
    a.radius = ctx->p.tube_radius;
    a.ring_xy = ctx->adh_ring;
    a.reach = 0.0;
    if (a.ring) {  // chord >= 2 sqrt(R rho) |sin(dtheta / 2)| with rho >= R - LIMIT dx for a searching knob
        const double L = h.limit * a.dx, R = a.radius, rho = std::max(R - L, 1.0e-300);
        const double arg = L / (2.0 * std::sqrt(R * rho));
        a.reach = arg >= 1.0 ? M_PI : 2.0 * std::asin(arg);
    }
    return a;
}

inline unsigned ablocks(long long n) { return n > 0 ? (unsigned)((n + AWG - 1) / AWG) : 1u; }

// Search, detachment and the attachment rounds (init: the nearest free
// receptors with no draw, AttachmentPointAtWall_GPU, adhesion.cu:278-314).
lbmibm_status adh_bell(lbmibm_ctx *ctx, int init) {
    const AdhDev a = adh_dev(ctx);
    hipStream_t st = ctx->stream;
    const long long nsp = (long long)ctx->adh_nk * a.ns;  // springs of the knobs
    const int *kl = ctx->adh_klist;
    const int nk = ctx->adh_nk;
    const AdhRound q{ctx->adh_idw, kl, ctx->adh_rw, ctx->adh_isatt, ctx->adh_attach, ctx->adh_pos, ctx->adh_active,
                     ctx->adh_prop, ctx->adh_rij, ctx->adh_claim, ctx->adh_calls, (const DevStep *)ctx->step, init, nk,
                     ctx->adh_list, {ctx->adh_list + 2, ctx->adh_list + 2 + nsp}, ctx->adh_made};
    hipLaunchKernelGGL(k_adh_search, dim3(ablocks(64LL * nk)), dim3(AWG), 0, st, a, (const double *)ctx->xs, kl, nk,
                       ctx->adh_idw, ctx->adh_rw);
    hipLaunchKernelGGL(k_adh_detach, dim3(ablocks(nsp)), dim3(AWG), 0, st, a, (const double *)ctx->xs,
                       (const unsigned char *)ctx->adh_knob, ctx->adh_attach, ctx->adh_rij, ctx->adh_isatt,
                       ctx->adh_pos, ctx->adh_active, (const DevStep *)ctx->step, init, kl, nk, ctx->adh_calls,
                       ctx->adh_claim, (long long)a.nxw * a.nzw, q.more, q.made);
    hipLaunchKernelGGL(k_adh_propose, dim3(ablocks(nsp)), dim3(AWG), 0, st, a, q);
    hipLaunchKernelGGL(k_adh_resolve, dim3(ablocks(nsp)), dim3(AWG), 0, st, a, q);
    const bool few = nsp <= ROUNDS_GROUP || (nsp <= ROUNDS_SPRINGS && a.ns <= ROUNDS_PER_KNOB);
    const int most = few ? INT_MAX : ROUNDS_GROUP;
    hipLaunchKernelGGL(k_adh_rounds, dim3(1), dim3(1024), 0, st, a, q, 0, 1, most);
    if (!few) {
        const int n = init || nsp > ROUNDS_MANY ? a.maxn : std::min(std::max(8LL, 4LL * a.ns), (long long)a.maxn);
        for (int r = 1; r <= n + 1; r++)
            hipLaunchKernelGGL(k_adh_round, dim3(ROUND_GROUPS), dim3(AWG), 0, st, a, q, r, r > n, most);
        if (n < a.maxn) hipLaunchKernelGGL(k_adh_rounds, dim3(1), dim3(1024), 0, st, a, q, 1, n + 1, INT_MAX);
    }
    LBMIBM_LAUNCHED(ctx, "k_adh_*");
    return LBMIBM_OK;
}

}  // namespace

// Adhesion() (adhesion.cu:772-790): the spring force of the current
// attachments (and the spreading force cf + f_adh), then the Bell update.
lbmibm_status adhesion_step(lbmibm_ctx *ctx) {
    const AdhDev a = adh_dev(ctx);
    if (ctx->prec == LBMIBM_F64)
        hipLaunchKernelGGL(k_adh_force<double>, dim3(ablocks(a.nv)), dim3(AWG), 0, ctx->stream, a,
                           (const double *)ctx->xs, (const double *)ctx->cf, (const unsigned char *)ctx->adh_knob,
                           (const int *)ctx->adh_attach, ctx->adh_fadh, (double *)ctx->adh_fsum);
    else
        hipLaunchKernelGGL(k_adh_force<float>, dim3(ablocks(a.nv)), dim3(AWG), 0, ctx->stream, a,
                           (const double *)ctx->xs, (const float *)ctx->cf, (const unsigned char *)ctx->adh_knob,
                           (const int *)ctx->adh_attach, ctx->adh_fadh, (float *)ctx->adh_fsum);
    LBMIBM_LAUNCHED(ctx, "k_adh_force");
    return adh_bell(ctx, 0);
}

lbmibm_status adhesion_setup(lbmibm_ctx *ctx, const lbmibm_adhesion_params *h, const unsigned char *is_knob) {
    ctx->adh = *h;
    // wall_init (adhesion.cu:441-458 slab, 467-480 tube ring)
    const double dx = ctx->p.dx, LX = ctx->p.lx * dx, LZ = ctx->p.lz * dx;
    const double dz = std::sqrt(1.0 / h->receptor_density) / h->rc;
    ctx->adh_nzw = (int)(LZ / dz + 1.0e-03);
    if (ctx->adh_nzw < 1) {
        ctx->err = "adhesion: receptor spacing larger than the box";
        return LBMIBM_ERR_ARG;
    }
    ctx->adh_dzw = LZ / (double)ctx->adh_nzw;
    if (ctx->p.tube_radius > 0.0) {
        ctx->adh_dxw = ctx->adh_dzw / ctx->p.tube_radius;  // dtheta
        ctx->adh_nxw = (int)(2.0 * M_PI / ctx->adh_dxw);   // ntheta
    } else {
        ctx->adh_nxw = (int)(LX / dz + 1.0e-03);
        ctx->adh_dxw = ctx->adh_nxw > 0 ? LX / (double)ctx->adh_nxw : 0.0;
    }
    if (ctx->adh_nxw < 1) {
        ctx->err = "adhesion: receptor spacing larger than the box";
        return LBMIBM_ERR_ARG;
    }
    const long long nrec = (long long)ctx->adh_nxw * ctx->adh_nzw, nv = ctx->nv;
    const long long nsp = nv * h->springs_per_knob, nn = nv * h->max_neighwall;
    // knobs: the caller's flags (the reference's ./input/icosa file) or
    // drawn with probability KNOB / (vertices of the cell)
    std::vector<int> voff(ctx->nc + 1);
    LBMIBM_HIP(ctx, hipMemcpy(voff.data(), ctx->voff, voff.size() * sizeof(int), hipMemcpyDeviceToHost));
    std::vector<unsigned char> knob((size_t)nv, 0);
    for (int c = 0; c < ctx->nc; c++)
        for (int v = voff[c]; v < voff[c + 1]; v++) {
            if (is_knob) {
                knob[v] = is_knob[v] ? 1 : 0;
            } else {  // iteration -1 is the knob draw's stream
                knob[v] = adh_uniform(h->seed, -1, v) < h->knob / (double)(voff[c + 1] - voff[c]) ? 1 : 0;
            }
        }
    std::vector<int> klist;
    for (long long v = 0; v < nv; v++)
        if (knob[v]) klist.push_back((int)v);
    ctx->adh_nk = (int)klist.size();
    // A second set-up may change every size (receptor count, MAXN, springs
    // per knob, knobs): the previous buffers, and the step graph recorded with
    // their addresses, are released once the device is done with them.
    lbmibm_status s = LBMIBM_OK;
    if (ctx->adh_knob) {
        LBMIBM_HIP(ctx, hipStreamSynchronize(ctx->stream));
        if (ctx->graph) (void)hipGraphExecDestroy(ctx->graph);
        ctx->graph = nullptr;
        ctx->graph_ready = false;
        ctx->adh_on = false;
        void **bufs[] = {&ctx->adh_knob, (void **)&ctx->adh_idw, (void **)&ctx->adh_rw, (void **)&ctx->adh_attach,
                         (void **)&ctx->adh_rij, (void **)&ctx->adh_pos, (void **)&ctx->adh_active,
                         (void **)&ctx->adh_prop, (void **)&ctx->adh_isatt, (void **)&ctx->adh_claim,
                         (void **)&ctx->adh_calls, (void **)&ctx->adh_fadh, (void **)&ctx->adh_list, (void **)&ctx->adh_made,
                         (void **)&ctx->adh_klist, &ctx->adh_fsum, (void **)&ctx->adh_ring};
        for (void **p : bufs) {
            if (*p) (void)hipFree(*p);
            *p = nullptr;
        }
    }
    auto al = [&](void **p, size_t bytes) {
        if (s == LBMIBM_OK) s = dev_alloc(ctx, p, bytes);
    };
    al(&ctx->adh_knob, nv);
    al((void **)&ctx->adh_idw, nn * sizeof(int));
    al((void **)&ctx->adh_rw, nn * sizeof(double));
    al((void **)&ctx->adh_attach, nsp * sizeof(int));
    al((void **)&ctx->adh_rij, nsp * sizeof(double));
    al((void **)&ctx->adh_pos, nsp * sizeof(int));
    al((void **)&ctx->adh_active, nsp * sizeof(int));
    al((void **)&ctx->adh_prop, nsp * sizeof(int));
    al((void **)&ctx->adh_isatt, nrec * sizeof(int));
    al((void **)&ctx->adh_claim, nrec * sizeof(unsigned long long));
    al((void **)&ctx->adh_calls, sizeof(unsigned long long));
    al((void **)&ctx->adh_fadh, 3 * nv * sizeof(double));
    al((void **)&ctx->adh_list, (2 + 2 * klist.size() * h->springs_per_knob) * sizeof(int));
    al((void **)&ctx->adh_made, (size_t)(h->max_neighwall + 2) * sizeof(int));
    al((void **)&ctx->adh_klist, std::max<size_t>(klist.size(), 1) * sizeof(int));
    al(&ctx->adh_fsum, 3 * nv * ctx->szT);
    std::vector<double> ring;
    if (ctx->p.tube_radius > 0.0) {  // the columns' coordinates with the host's libm, as wall_init computes them
        ring.resize(2 * (size_t)ctx->adh_nxw);
        for (int ix = 0; ix < ctx->adh_nxw; ix++) {
            ring[2 * ix] = ctx->p.tube_radius * std::cos(ix * ctx->adh_dxw);
            ring[2 * ix + 1] = ctx->p.tube_radius * std::sin(ix * ctx->adh_dxw);
        }
        al((void **)&ctx->adh_ring, ring.size() * sizeof(double));
    }
    if (s != LBMIBM_OK) return s;
    if (!ring.empty())
        LBMIBM_HIP(ctx, hipMemcpy(ctx->adh_ring, ring.data(), ring.size() * sizeof(double), hipMemcpyHostToDevice));
    LBMIBM_HIP(ctx, hipMemcpy(ctx->adh_knob, knob.data(), nv, hipMemcpyHostToDevice));
    if (!klist.empty())
        LBMIBM_HIP(ctx, hipMemcpy(ctx->adh_klist, klist.data(), klist.size() * sizeof(int), hipMemcpyHostToDevice));
    hipStream_t st = ctx->stream;
    hipLaunchKernelGGL(k_afill<int>, dim3(ablocks(nsp)), dim3(AWG), 0, st, ctx->adh_attach, (size_t)nsp, -1);
    hipLaunchKernelGGL(k_afill<double>, dim3(ablocks(nsp)), dim3(AWG), 0, st, ctx->adh_rij, (size_t)nsp, -1.0e10);
    hipLaunchKernelGGL(k_afill<int>, dim3(ablocks(nrec)), dim3(AWG), 0, st, ctx->adh_isatt, (size_t)nrec, 0);
    hipLaunchKernelGGL(k_afill<unsigned long long>, dim3(ablocks(nrec)), dim3(AWG), 0, st, ctx->adh_claim,
                       (size_t)nrec, 0ull);
    hipLaunchKernelGGL(k_afill<unsigned long long>, dim3(1), dim3(64), 0, st, ctx->adh_calls, (size_t)1, 0ull);
    hipLaunchKernelGGL(k_afill<double>, dim3(ablocks(3 * nv)), dim3(AWG), 0, st, ctx->adh_fadh, (size_t)(3 * nv), 0.0);
    hipLaunchKernelGGL(k_afill<int>, dim3(ablocks(nn)), dim3(AWG), 0, st, ctx->adh_idw, (size_t)nn, -1);
    hipLaunchKernelGGL(k_afill<double>, dim3(ablocks(nn)), dim3(AWG), 0, st, ctx->adh_rw, (size_t)nn, 1.0e15);
    LBMIBM_LAUNCHED(ctx, "k_afill");
    ctx->adh_on = true;
    s = adh_bell(ctx, 1);
    if (s == LBMIBM_OK) LBMIBM_HIP(ctx, hipStreamSynchronize(st));
    return s;
}

}  // namespace lbmibm
