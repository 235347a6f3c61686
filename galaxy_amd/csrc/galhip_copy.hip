// galhip_copy.hip -- particle arrays between the caller's pageable memory and
// the device.
//
// A large hipMemcpy to pageable memory runs at 10 GB/s into pages not yet
// touched (17 GB/s into touched ones): one thread zeroes the pages and copies.
// An unload of many bytes goes through pinned chunks (55 GB/s) while several
// threads move the chunks that have arrived, so that first touches and copies
// go on together: 200 MB in five arrays 20.8 -> 5.6 ms.  Chunks of 1 MiB: 7.9
// ms, of 8 MiB 5.2; 4 threads 6.4, 12 threads 5.5.
// Loads stay plain copies: their pages are there, staging took 1e7 particles
// from 7.9 to 5.9 ms only, and 24 MB loaded beside a busy host thread took 14
// ms staged and 1.5 plain.  (Their gain, 10.4 -> 7.9 ms, is the zone check on
// the device.)
#include "galhip_ctx.h"

#include <algorithm>
#include <climits>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace {

using namespace gh;

constexpr size_t CHUNK = 4u << 20;    // bytes of a pinned chunk
constexpr int NBUF = 4;               // chunks of a buffer
constexpr int MAX_THREADS = 8;
constexpr size_t STAGED_MIN = 16u << 20;
constexpr long long ZONES_DEVICE = 1 << 17;
constexpr int COPY_SEGMENTS = 8;      // arrays of a copy at most
constexpr size_t KEEP = 2;            // idle buffers kept (32 MiB of pinned memory)

// Idle pinned buffers of NBUF chunks, shared by the contexts of the process;
// the last context to go frees them.
std::mutex g_mu;
std::vector<void *> g_idle;
int g_contexts = 0;   // contexts of the process

void *take_buffer() {
    {
        std::lock_guard<std::mutex> lock(g_mu);
        if (!g_idle.empty()) {
            void *p = g_idle.back();
            g_idle.pop_back();
            return p;
        }
    }
    void *p = nullptr;
    if (hipHostMalloc(&p, NBUF * CHUNK, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    return p;
}

void give_buffer(void *p) {
    {
        std::lock_guard<std::mutex> lock(g_mu);
        if (g_contexts > 0 && g_idle.size() < KEEP) {
            g_idle.push_back(p);
            return;
        }
    }
    (void)hipHostFree(p);
}

struct Piece {
    char *host, *dev;
    size_t bytes;
};

// The pieces to the host through the pinned chunks of buf; false if it could
// not be set up (nothing has been copied then) or, with err set, if a copy
// failed.  Whoever waits sleeps: threads that yield instead keep the CPU, by
// slices of 4 ms, from a thread with work on it once the process is busy
// otherwise.
bool staged(const std::vector<Piece> &pieces, char *buf, hipStream_t s, hipError_t *err) {
    const int n = (int)pieces.size();
    const int nthr = (int)std::min<unsigned>(MAX_THREADS,
                                             std::max(1u, std::thread::hardware_concurrency()));
    hipEvent_t ev[NBUF];
    int nev = 0;
    while (nev < NBUF && hipEventCreateWithFlags(&ev[nev], hipEventDisableTiming) == hipSuccess)
        nev++;
    std::mutex mu;
    std::condition_variable go, moved;
    int ready = 0;                       // pieces the threads may move
    bool stop = false;
    std::vector<int> left(n, nthr);      // threads that have not moved their share
    auto move = [&](int w) {
        for (int i = 0; i < n; i++) {
            {
                std::unique_lock<std::mutex> lock(mu);
                go.wait(lock, [&] { return stop || ready > i; });
                if (ready <= i) return;
            }
            // page-aligned shares, so that two threads do not touch one page
            const size_t share = ((pieces[i].bytes + nthr - 1) / nthr + 4095) / 4096 * 4096;
            const size_t lo = std::min(pieces[i].bytes, w * share);
            const size_t hi = std::min(pieces[i].bytes, lo + share);
            memcpy(pieces[i].host + lo, buf + (size_t)(i % NBUF) * CHUNK + lo, hi - lo);
            std::lock_guard<std::mutex> lock(mu);
            if (--left[i] == 0) moved.notify_one();
        }
    };
    std::vector<std::thread> team;
    bool ok = nev == NBUF;
    if (ok) {
        try {
            team.reserve(nthr);
            for (int w = 0; w < nthr; w++) team.emplace_back(move, w);
        } catch (...) {
            ok = false;
        }
    }
    auto release = [&](int k) {
        {
            std::lock_guard<std::mutex> lock(mu);
            ready = k;
        }
        go.notify_all();
    };
    hipError_t e = hipSuccess;
    if (ok) {
        for (int i = 0; i < n && e == hipSuccess; i++) {
            if (i >= NBUF) {
                std::unique_lock<std::mutex> lock(mu);
                moved.wait(lock, [&] { return left[i - NBUF] == 0; });
            }
            e = hipMemcpyAsync(buf + (size_t)(i % NBUF) * CHUNK, pieces[i].dev, pieces[i].bytes,
                               hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipEventRecord(ev[i % NBUF], s);
            if (i > 0 && e == hipSuccess) {
                e = hipEventSynchronize(ev[(i - 1) % NBUF]);
                if (e == hipSuccess) release(i);
            }
        }
        if (e == hipSuccess) e = hipEventSynchronize(ev[(n - 1) % NBUF]);
        if (e == hipSuccess) release(n);
    }
    if (!ok || e != hipSuccess) {
        {
            std::lock_guard<std::mutex> lock(mu);
            stop = true;
        }
        go.notify_all();
    }
    for (auto &t : team) t.join();
    for (int k = 0; k < nev; k++) (void)hipEventDestroy(ev[k]);
    if (e != hipSuccess) {
        (void)hipStreamSynchronize(s);   // no copy into the chunks is left in flight
        *err = e;
    }
    return ok && e == hipSuccess;
}

// Is a pointer's memory known to the runtime (pinned, managed, on a device)?
// The pinned chunks would only add a second pass: 20 MB in five pinned arrays
// 0.46 ms plain and 0.66 staged, 200 MB 4.2 and 4.8.
bool known_memory(const void *p) {
    hipPointerAttribute_t a;
    memset(&a, 0, sizeof a);
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

// Zones of a load: z[i] from iz[i], the lowest index outside 1..nz+1 to chk[0],
// the off-grid counts (zone nz + 1) to chk[4 m + 4].  A block takes one entry
// of an ensemble's block list, which never straddles two members, else `per`
// particles of the one grid.
__global__ __launch_bounds__(GH_BLOCK) void zone_load_kernel(const int *__restrict__ iz,
                                                             uint8_t *__restrict__ z, int nz,
                                                             long long n, int per,
                                                             const int4 *__restrict__ blk,
                                                             long long *chk) {
    const long long i0 = blk ? blk[blockIdx.x].y : (long long)blockIdx.x * per;
    const long long i1 = blk ? i0 + blk[blockIdx.x].z : min(n, i0 + per);
    const int m = blk ? blk[blockIdx.x].x : 0;
    int off = 0;
    for (long long i = i0 + threadIdx.x; i < i1; i += GH_BLOCK) {
        const int v = iz[i];
        z[i] = (uint8_t)v;
        off += v == nz + 1;
        if (v < 1 || v > nz + 1) atomicMin(chk, i);
    }
    for (int w = 32; w; w >>= 1) off += __shfl_xor(off, w);
    if ((threadIdx.x & 63) == 0 && off)
        atomicAdd((unsigned long long *)&chk[4 * m + 4], (unsigned long long)off);
}

// the zones and counts of a load that passed the check
__global__ __launch_bounds__(GH_BLOCK) void zone_accept_kernel(const uint8_t *__restrict__ z2,
                                                               uint8_t *__restrict__ z, long long n,
                                                               const long long *__restrict__ chk,
                                                               long long *__restrict__ counters,
                                                               int ncnt) {
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < ncnt; i += GH_BLOCK) counters[i] = chk[4 + i];
    const long long i0 = ((long long)blockIdx.x * GH_BLOCK + threadIdx.x) * 16;
    if (i0 + 16 <= n) *(int4 *)(z + i0) = *(const int4 *)(z2 + i0);
    else
        for (long long i = i0; i < n; i++) z[i] = z2[i];
}

__global__ void zone_check_init(long long *chk, int n) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) chk[i] = i ? 0 : LLONG_MAX;
}

// low parts of the positions -> planar arrays in load order
__global__ __launch_bounds__(GH_BLOCK) void planar_lo_kernel(const float2 *__restrict__ lo,
                                                             const unsigned *__restrict__ id,
                                                             float *__restrict__ d, long long n) {
    const long long i = (long long)blockIdx.x * GH_BLOCK + threadIdx.x;
    if (i >= n) return;
    const long long p = id[i];
    const float2 v = lo[i];
    d[p] = v.x;
    d[n + p] = v.y;
}

}  // namespace

CopyUser::CopyUser() {
    std::lock_guard<std::mutex> lock(g_mu);
    g_contexts++;
}

CopyUser::~CopyUser() {
    std::vector<void *> gone;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        if (--g_contexts == 0) gone.swap(g_idle);
    }
    for (void *p : gone) (void)hipHostFree(p);
}

// Copies the segments (host, device, bytes) on the context's stream and waits
// for them.  To pageable memory staged from STAGED_MIN bytes in all, plain copies
// below it: starting the threads costs 0.1 ms, 4 MB in five arrays take 0.34 ms
// staged and 0.24 plain, 8 MB 0.42 and 0.50, 20 MB 0.7 and 1.2.
int copy_segments(const galhip_ctx *c, const CopySegment *seg, int nseg, bool to_host) {
    // (a plain copy that finds the stream busy takes 30 us longer)
    HIPCHK(hipStreamSynchronize(c->s));
    size_t total = 0;
    bool plain[COPY_SEGMENTS];
    if (nseg > COPY_SEGMENTS) return gh_fail(GALHIP_EINVAL, "particle copy: %d arrays", nseg);
    for (int k = 0; k < nseg; k++) {
        plain[k] = !to_host || !seg[k].host;
        if (!plain[k]) total += seg[k].bytes;
    }
    if (total >= STAGED_MIN)   // (a look costs 0.7 us: not for small copies)
        for (int k = 0; k < nseg; k++)
            if (!plain[k] && known_memory(seg[k].host)) {
                plain[k] = true;
                total -= seg[k].bytes;
            }
    bool done = false;         // the pageable ones
    if (total >= STAGED_MIN) {
        void *buf = take_buffer();
        if (buf) {
            bool ok = false;
            hipError_t e = hipSuccess;
            try {
                std::vector<Piece> pieces;
                for (int k = 0; k < nseg; k++)
                    for (size_t o = 0; !plain[k] && o < seg[k].bytes; o += CHUNK)
                        pieces.push_back({(char *)seg[k].host + o, (char *)seg[k].dev + o,
                                          std::min(CHUNK, seg[k].bytes - o)});
                ok = staged(pieces, (char *)buf, c->s, &e);
            } catch (...) {
                ok = false;
            }
            give_buffer(buf);
            done = ok;
            if (e != hipSuccess)
                return gh_fail(GALHIP_EHIP, "particle copy: %s", hipGetErrorString(e));
        }
    }
    for (int k = 0; k < nseg; k++) {
        if (!seg[k].host || seg[k].bytes == 0 || (done && !plain[k])) continue;
        if (to_host)
            HIPCHK(hipMemcpy(seg[k].host, seg[k].dev, seg[k].bytes, hipMemcpyDeviceToHost));
        else
            HIPCHK(hipMemcpy(seg[k].dev, seg[k].host, seg[k].bytes, hipMemcpyHostToDevice));
    }
    return 0;
}

// The zones of a load: the context's zones and off-grid counts stay as they
// were if one is outside 1..nz+1.  Checked on the device from ZONES_DEVICE
// particles on, where the host's loop begins to cost more than the round trip
// of the check (1.4e5: 0.30 ms a load both ways; 1e3: 0.12 ms on the host, 0.145
// on the device; 1e7: 14 ms less on the device).
int load_zones(galhip_ctx *c, long long n, const int32_t *iz) {
    if (n < ZONES_DEVICE) {
        std::vector<uint8_t> z(n);
        std::vector<long long> cnt(4 * (size_t)c->nmem, 0);
        int m = 0;
        for (long long i = 0; i < n; i++) {
            while (c->ens && i >= c->m_off[m + 1]) m++;
            const int v = iz[i];
            if (v < 1 || v > c->nz + 1)
                return gh_fail(GALHIP_EINVAL, "particle %lld has zone %d outside 1..%d", i, v, c->nz + 1);
            z[i] = (uint8_t)v;
            if (v == c->nz + 1) cnt[4 * m]++;    // /admin/ noff: the off-grid list
        }
        HIPCHK(hipMemcpy(c->counters, cnt.data(), sizeof(long long) * cnt.size(), hipMemcpyHostToDevice));
        if (n > 0) HIPCHK(hipMemcpy(c->zone, z.data(), n, hipMemcpyHostToDevice));
        return 0;
    }
    const int nchk = 4 * (c->nmem + 1);
    hipLaunchKernelGGL(zone_check_init, dim3(1), dim3(GH_BLOCK), 0, c->s, c->load_chk, nchk);
    HIPCHK(hipGetLastError());
    // through the sort keys and the second zone array, free outside a sort
    const CopySegment seg = {(void *)iz, c->key, sizeof(int32_t) * (size_t)n};
    int rc = copy_segments(c, &seg, 1, false);
    if (rc) return rc;
    const int per = 16 * GH_BLOCK;
    const int nb = c->ens ? c->nblk : (int)((n + per - 1) / per);
    hipLaunchKernelGGL(zone_load_kernel, dim3(nb), dim3(GH_BLOCK), 0, c->s,
                       (const int *)c->key, c->zone2, c->nz, n, per,
                       c->ens ? (const int4 *)c->blk_d : (const int4 *)nullptr, c->load_chk);
    HIPCHK(hipGetLastError());
    long long bad = 0;
    HIPCHK(hipMemcpyAsync(&bad, c->load_chk, sizeof bad, hipMemcpyDeviceToHost, c->s));
    HIPCHK(hipStreamSynchronize(c->s));
    if (bad < n)
        return gh_fail(GALHIP_EINVAL, "particle %lld has zone %d outside 1..%d", bad, iz[bad],
                       c->nz + 1);
    hipLaunchKernelGGL(zone_accept_kernel,
                       dim3((unsigned)((n + 16 * GH_BLOCK - 1) / (16 * GH_BLOCK))),
                       dim3(GH_BLOCK), 0, c->s, c->zone2, c->zone, n, c->load_chk, c->counters,
                       nchk - 4);
    HIPCHK(hipGetLastError());
    return 0;
}

namespace gh {
hipError_t launch_planar_lo(const float2 *lo, const unsigned *id, float *d, long long n,
                            hipStream_t s) {
    hipLaunchKernelGGL(planar_lo_kernel, dim3((unsigned)((n + GH_BLOCK - 1) / GH_BLOCK)),
                       dim3(GH_BLOCK), 0, s, lo, id, d, n);
    return hipGetLastError();
}
}  // namespace gh
