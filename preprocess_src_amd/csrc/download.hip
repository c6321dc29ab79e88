// Fields and vertex arrays handed over in the reference's host layouts (FP64,
// the lattice padded by two nodes on every side).
//
// The compact device array crosses the link in pieces through a ring of pinned
// buffers, in its own precision, and threads of the call's own widen each
// piece and write its padded rows while the next ones are on their way.
// Pageable copies of whole fields and one thread's loop over the padded nodes
// took, before: velocity of 160^3 FP32 nodes 50 to 53 ms, now 2.8 to 7; of the
// 1024-cell suspension 45 and now 3 to 5, with its vertices 17 and now 3 to 5;
// eight fields of 64x32x32 FP64 nodes 0.70 and 0.36; what bounds it now is the
// host's writing (fresh pages first of all).
#include <condition_variable>
#include <cstring>
#include <new>
#include <system_error>
#include <thread>

#include "common.hpp"

namespace lbmibm {

// Ring of a context: RING pieces of at most PIECE bytes (one lattice row where
// that is longer), allocated with the context (pinning costs 0.2 ms per MB)
// and freed with it.
constexpr size_t PIECE = 512 << 10;
constexpr int RING = 8;
// Threads besides the caller's: one for every 8 MB, at most 4.  On three fields
// of 160^3 FP32 values 2, 4 and 8 of them took 3.8, 2.5 and 2.0 ms into arrays
// in use, 10, 8 and 8 to 9 ms into fresh pages.  Below 8 MB none: the 6 MB of a
// 128x64x64 lattice take the caller 0.6 ms, and waiting for threads to be
// scheduled next to a program's own took up to 5.
constexpr size_t PER_THREAD = 8 << 20;
constexpr int MAX_THREADS = 4;

struct Staging {
    void *buf = nullptr;
    size_t piece = 0;
    hipEvent_t ev[RING] = {};
};

void staging_free(lbmibm_ctx *ctx) {
    Staging *st = ctx->staging;
    if (!st) return;
    for (auto &e : st->ev)
        if (e) (void)hipEventDestroy(e);
    if (st->buf) (void)hipHostFree(st->buf);
    delete st;
    ctx->staging = nullptr;
}

lbmibm_status staging_init(lbmibm_ctx *ctx) {
    ctx->staging = new (std::nothrow) Staging;
    if (!ctx->staging) return LBMIBM_ERR_HIP;
    for (auto &e : ctx->staging->ev) LBMIBM_HIP(ctx, hipEventCreateWithFlags(&e, hipEventDisableTiming));
    return LBMIBM_OK;
}

static lbmibm_status staging_room(lbmibm_ctx *ctx, size_t piece) {
    Staging *st = ctx->staging;
    if (st->piece >= piece) return LBMIBM_OK;
    // what the context's largest array takes, so that it need not grow
    piece = std::max(piece, std::min(PIECE, std::max((size_t)ctx->N, 3 * (size_t)ctx->nv) * sizeof(double)));
    if (st->buf) (void)hipHostFree(st->buf);
    st->buf = nullptr;
    st->piece = 0;
    LBMIBM_HIP(ctx, hipHostMalloc(&st->buf, RING * piece, hipHostMallocPortable));
    st->piece = piece;
    return LBMIBM_OK;
}

void staging_reserve(lbmibm_ctx *ctx) {
    if (staging_room(ctx, 1) != LBMIBM_OK) {  // the first download tries again
        (void)hipGetLastError();
        ctx->err.clear();
    }
}

// Whether two of the host arrays, of n values each, share memory.
static bool overlap(const std::vector<FieldOut> &out, size_t n) {
    for (size_t i = 0; i < out.size(); i++)
        for (size_t j = 0; j < i; j++) {
            const uintptr_t a = (uintptr_t)out[i].dst, b = (uintptr_t)out[j].dst;
            if ((a < b ? b - a : a - b) < n * sizeof(double)) return true;
        }
    return false;
}

// Copies pieces 0..n-1 (source(i, &bytes) names piece i) and hands each to
// take(i, data), in any order, on several threads; take writes disjoint memory.
// Or in their order, on the caller's alone: where arrays share memory (a caller may
// give one place for all that it does not want), what comes last remains.
template <typename Source, typename Take>
static lbmibm_status staged(lbmibm_ctx *ctx, size_t n, size_t piece, size_t total, bool in_order, Source source,
                            Take take) {
    if (n == 0) return LBMIBM_OK;
    const std::lock_guard<std::mutex> lock(ctx->staging_mutex);  // callers may share a context's ring
    lbmibm_status s = staging_room(ctx, piece);
    if (s != LBMIBM_OK) return s;
    char *const buf = (char *)ctx->staging->buf;
    const size_t stride = ctx->staging->piece;
    hipEvent_t *const ev = ctx->staging->ev;
    std::mutex m;
    std::condition_variable arrival, room;
    size_t next = 0, ready = 0, oldest = 0;  // pieces claimed and arrived; all below `oldest` are taken
    bool stop = false;
    std::vector<char> done(n, 0);
    // claims the next piece, waits for it if told to, and takes it; false when there is none
    auto work = [&](bool wait) {
        std::unique_lock<std::mutex> l(m);
        if (wait) arrival.wait(l, [&] { return next < ready || next >= n || stop; });
        if (next >= ready || stop) return false;
        const size_t i = next++;
        l.unlock();
        take(i, buf + stride * (i % RING));
        l.lock();
        done[i] = 1;
        while (oldest < n && done[oldest]) oldest++;
        l.unlock();
        room.notify_one();
        return true;
    };
    std::vector<std::thread> pool;
    const size_t want = in_order ? 0 : std::min({(size_t)MAX_THREADS, total / PER_THREAD, n - 1});
    try {
        pool.reserve(want);
        for (size_t t = 0; t < want; t++) pool.emplace_back([&] { while (work(true)) {} });
    } catch (const std::exception &) {  // no more threads to be had: the ones there are, and this one
    }
    hipError_t r = hipSuccess;
    auto arrived = [&](size_t upto) {  // publishes the pieces below `upto`
        for (size_t i = ready; i < upto && r == hipSuccess; i++) {  // only this thread changes `ready`
            r = hipEventSynchronize(ev[i % RING]);
            const std::lock_guard<std::mutex> l(m);
            if (r == hipSuccess) ready = i + 1;
        }
        arrival.notify_all();
    };
    for (size_t c = 0; c < n && r == hipSuccess; c++) {
        if (c >= RING) {
            arrived(c - RING + 1);
            if (r != hipSuccess) break;
            // its buffer is free once the piece before it there is taken: by this thread, or by one at work on it
            while (work(false)) {
                const std::lock_guard<std::mutex> l(m);
                if (oldest > c - RING) break;
            }
            std::unique_lock<std::mutex> l(m);
            room.wait(l, [&] { return oldest > c - RING; });
        }
        size_t bytes;
        const void *src = source(c, &bytes);
        r = hipMemcpyAsync(buf + stride * (c % RING), src, bytes, hipMemcpyDeviceToHost, ctx->stream);
        if (r == hipSuccess) r = hipEventRecord(ev[c % RING], ctx->stream);
        if (c >= RING / 2) arrived(c + 1 - RING / 2);
    }
    arrived(n);
    if (r == hipSuccess) {
        while (work(false)) {}
    } else {
        const std::lock_guard<std::mutex> l(m);
        stop = true;
    }
    arrival.notify_all();
    for (auto &t : pool) t.join();
    if (r != hipSuccess) {
        (void)hipStreamSynchronize(ctx->stream);  // nothing may write the ring any more
        LBMIBM_HIP(ctx, r);
    }
    return LBMIBM_OK;
}

// Geometry of the padded rows; the periodic images in the halo as in lbm.cu:1350-1353,
// 1410-1411.
struct Frame {
    int nx, ny, nz, nxp, nyp, nzp;
    bool images, zero, py;         // periodic images / zeros in place of wall nodes / y periodic
    std::vector<int> first, last;  // tube: the inside span of each fluid row (empty: whole rows)
};

// Row (y, z) of the lattice into every padded row that holds it.
template <typename T> static void put_rows(const Frame &f, const T *src, int y, int z, double *dst) {
    const int x0 = f.first.empty() ? 0 : f.first[y], x1 = f.first.empty() ? f.nx : f.last[y];
    const bool wrap = f.images && f.first.empty();
    int ys[3], zs[3], ny = 0, nz = 0;
    ys[ny++] = y + 2;
    zs[nz++] = z + 2;
    if (f.images) {
        if (f.py && y >= f.ny - 2) ys[ny++] = y + 2 - f.ny;
        if (f.py && y < 2) ys[ny++] = y + 2 + f.ny;
        if (z >= f.nz - 2) zs[nz++] = z + 2 - f.nz;
        if (z < 2) zs[nz++] = z + 2 + f.nz;
    }
    for (int k = 0; k < nz; k++)
        for (int j = 0; j < ny; j++) {
            double *d = dst + (size_t)f.nxp * (ys[j] + (size_t)f.nyp * zs[k]);
            for (int x = x0; x < x1; x++) d[2 + x] = (double)src[x];
            if (wrap) {
                d[0] = (double)src[f.nx - 2];
                d[1] = (double)src[f.nx - 1];
                d[f.nx + 2] = (double)src[0];
                d[f.nx + 3] = (double)src[1];
            } else if (f.zero) {
                std::fill(d, d + 2 + x0, 0.0);
                std::fill(d + 2 + x1, d + f.nxp, 0.0);
            }
        }
    if (!f.zero) return;
    // the padded rows that hold no lattice row: with the row next to them
    auto clear = [&](int a, int b, int k0, int k1) {  // rows a..b-1 of planes k0..k1-1
        for (int k = k0; k < k1; k++) std::fill_n(dst + (size_t)f.nxp * (a + (size_t)f.nyp * k), (size_t)f.nxp * (b - a), 0.0);
    };
    if (!(f.images && f.py))
        for (int k = 0; k < nz; k++) {
            if (y == 0) clear(0, 2, zs[k], zs[k] + 1);
            if (y == f.ny - 1) clear(f.nyp - 2, f.nyp, zs[k], zs[k] + 1);
        }
    if (!f.images && y == 0) {
        if (z == 0) clear(0, f.nyp, 0, 2);
        if (z == f.nz - 1) clear(0, f.nyp, f.nzp - 2, f.nzp);
    }
}

lbmibm_status download_fields(lbmibm_ctx *ctx, const FieldOut *all, int nall, size_t elem, bool images, bool zero) {
    std::vector<FieldOut> out;
    for (int i = 0; i < nall; i++)
        if (all[i].dst) out.push_back(all[i]);
    Frame f{ctx->nx, ctx->ny, ctx->nz, ctx->nxp, ctx->nyp, ctx->nzp, images, zero, ctx->p.periodic_y != 0, {}, {}};
    if (images && ctx->p.tube_radius > 0.0) {  // the disc's halo columns are wall
        f.first.assign(f.ny, 0);
        f.last.assign(f.ny, 0);
        for (int y = 0; y < f.ny; y++) {
            int a = 0, b = f.nx;
            while (a < b && !tube_inside(ctx, a, y)) a++;
            while (b > a && !tube_inside(ctx, b - 1, y)) b--;
            f.first[y] = a;
            f.last[y] = b;
        }
    }
    const size_t row = (size_t)f.nx * elem, rows = (size_t)f.ny * f.nz;
    const size_t per = std::min(std::max<size_t>(PIECE / row, 1), rows), pieces = (rows + per - 1) / per;
    return staged(
        ctx, out.size() * pieces, per * row, out.size() * rows * row, overlap(out, (size_t)ctx->np),
        [&](size_t i, size_t *bytes) {
            const size_t r0 = i % pieces * per;
            *bytes = (std::min(r0 + per, rows) - r0) * row;
            return (const char *)out[i / pieces].src + r0 * row;
        },
        [&](size_t i, const char *data) {
            const size_t r0 = i % pieces * per, r1 = std::min(r0 + per, rows);
            double *dst = out[i / pieces].dst;
            for (size_t r = r0; r < r1; r++, data += row) {
                const int y = (int)(r % f.ny), z = (int)(r / f.ny);
                if (elem == 8) put_rows(f, (const double *)data, y, z, dst);
                else put_rows(f, (const float *)data, y, z, dst);
            }
        });
}

lbmibm_status download_arrays(lbmibm_ctx *ctx, const FieldOut *all, int nall, size_t elem, size_t n) {
    std::vector<FieldOut> out;
    for (int i = 0; i < nall; i++)
        if (all[i].dst) out.push_back(all[i]);
    const size_t per = std::min(PIECE / elem, n), pieces = n ? (n + per - 1) / per : 0;
    return staged(
        ctx, out.size() * pieces, per * elem, out.size() * n * elem, overlap(out, n),
        [&](size_t i, size_t *bytes) {
            const size_t a = i % pieces * per;
            *bytes = (std::min(a + per, n) - a) * elem;
            return (const char *)out[i / pieces].src + a * elem;
        },
        [&](size_t i, const char *data) {
            const size_t a = i % pieces * per, m = std::min(a + per, n) - a;
            double *dst = out[i / pieces].dst + a;
            if (elem == 8) std::memcpy(dst, data, m * 8);
            else
                for (size_t k = 0; k < m; k++) dst[k] = (double)((const float *)data)[k];
        });
}

}  // namespace lbmibm
