// transfer.hip -- arrays between the caller's host memory and the device.
//
// The caller's arrays are ordinary pageable memory, new ones often not mapped
// yet.  The runtime's own copies of such memory go through one thread (4 GB/s
// into a new array, whose pages the kernel clears as they are touched, 18 GB/s
// into a mapped one, 29 GB/s out of one) where the link moves 56 GB/s.  Here the
// link works on pinned buffers, batch after batch, while several host threads
// copy between those and the caller's array; indices travel as the device's
// 32-bit numbers and are widened (or narrowed and checked) by the same threads.
// finish() of a 29.4-million-entry matrix 45 -> 8.4 ms (the link alone: 6.3);
// six million COO entries in and 2.4 million out 8.0 -> 3.8 ms.
//
// A ring of pinned memory, XF_SLOTS batches of XF_BATCH bytes, is shared by all
// contexts of a device (one transfer holds it at a time, with its device work
// already done: a second would halve the link's share of both), allocated by the
// first that needs it (0.2 ms; its pages are mapped as they are used) and freed
// with the device's last context.  Where it cannot be pinned it is ordinary
// memory, which the runtime copies through buffers of its own.
//
// Up to XF_SMALL bytes on the device the fixed costs are the time: a copy, an
// event and a wait an array.  Such a transfer goes through pinned memory of the
// context's own, its arrays side by side, moved by one kernel that reads or writes
// that memory over the link; out of the device it waits once and the calling
// thread copies, into it nothing waits (the next transfer that finds no room
// does).  A whole REUSE step with new coefficients, matrix and load read back, heat Q4 48x48:
// the runtime's copies 133 us, through the ring 163, so 64; 100x100 192, 204, 104.
#include <emmintrin.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <mutex>

#include "common.h"

int env_int(const char *name, int dflt);  // reuse.hip

namespace {

// (29.4 million entries out, ms: batches of 2 MiB 10.2; 6, 9, 12, 15 threads
// 9.0, 8.6, 8.4, 8.4)
constexpr int64_t XF_BATCH = 4 << 20;  // bytes on the device of one batch, at most
constexpr int XF_SLOTS = 8;
constexpr int64_t XF_PAGE = 2 << 20;   // parts end at multiples of it in the caller's array (a large page is one thread's)
constexpr int XF_THREADS = 12;
constexpr int64_t XF_PER_THREAD = 1 << 20;  // bytes of the caller's memory that pay for one more thread
constexpr int64_t XF_SMALL = 2 << 20;
constexpr int XF_MOVES = 4;            // arrays of a small transfer

// Pinned memory; null: there is none (ELFEL_HIP_PINNED=0: as if there were none).
void *pin(size_t bytes)
{
    void *p = nullptr;
    if (env_int("ELFEL_HIP_PINNED", 1) != 0 && hipHostMalloc(&p, bytes, hipHostMallocPortable) == hipSuccess) return p;
    (void)hipGetLastError();
    return nullptr;
}

struct Ring {
    std::mutex hold;  // during a transfer
    std::mutex life;  // guards what follows
    char *mem = nullptr;
    bool pinned = false;
    int users = 0;
};
Ring rings[ELFEL_MAXDEV];

char *ring_get(Ring &R)
{
    std::lock_guard<std::mutex> g(R.life);
    if (!R.mem) {
        R.mem = (char *)pin(XF_BATCH * XF_SLOTS);
        R.pinned = R.mem != nullptr;
        if (!R.mem) R.mem = (char *)aligned_alloc(XF_PAGE, XF_BATCH * XF_SLOTS);
    }
    return R.mem;
}

// One thread's share of a batch: `n` words of the caller's array.
struct Part {
    int batch;
    int64_t at, n;      // words from the segment's start; count
    int64_t slot_off;   // bytes from the slot's start
};
struct Batch {
    int seg;
    int64_t at, n;
    int parts;
};

// int32 -> int64 + base; streaming stores here and below (ordinary ones measured
// the same for results that fit the host's caches, 3 % slower for larger)
void widen(int64_t *dst, const int32_t *src, int64_t n, int64_t base)
{
    int64_t i = 0;
    for (; i < n && ((uintptr_t)(dst + i) & 15); i++) dst[i] = (int64_t)src[i] + base;
    const __m128i b = _mm_set1_epi64x(base), z = _mm_setzero_si128();
    for (; i + 4 <= n; i += 4) {  // device indices are not negative
        const __m128i v = _mm_loadu_si128((const __m128i *)(src + i));
        _mm_stream_si128((__m128i *)(dst + i), _mm_add_epi64(_mm_unpacklo_epi32(v, z), b));
        _mm_stream_si128((__m128i *)(dst + i + 2), _mm_add_epi64(_mm_unpackhi_epi32(v, z), b));
    }
    for (; i < n; i++) dst[i] = (int64_t)src[i] + base;
    _mm_sfence();
}

void copy_out(char *dst, const char *src, int64_t n)
{
    int64_t i = std::min<int64_t>(n, (16 - ((uintptr_t)dst & 15)) & 15);
    memcpy(dst, src, (size_t)i);
    for (; i + 64 <= n; i += 64) {
        const __m128i a = _mm_loadu_si128((const __m128i *)(src + i)), b = _mm_loadu_si128((const __m128i *)(src + i + 16));
        const __m128i c = _mm_loadu_si128((const __m128i *)(src + i + 32)), d = _mm_loadu_si128((const __m128i *)(src + i + 48));
        _mm_stream_si128((__m128i *)(dst + i), a);
        _mm_stream_si128((__m128i *)(dst + i + 16), b);
        _mm_stream_si128((__m128i *)(dst + i + 32), c);
        _mm_stream_si128((__m128i *)(dst + i + 48), d);
    }
    memcpy(dst + i, src + i, (size_t)(n - i));
    _mm_sfence();
}

// int64 in lo..hi -> int32, 0-based; false: some value lies outside (and counts
// as lo).  v - lo or hi - v is negative there and nowhere else, so one sign bit of
// all tells, without a comparison a value (0.3 -> 0.2 ns a value).
bool narrow(int32_t *dst, const int64_t *src, int64_t n, int64_t lo, int64_t hi)
{
    const uint64_t range = (uint64_t)(hi - lo);
    const uint32_t first = (uint32_t)(lo - 1);
    uint64_t outside = 0;
    for (int64_t i = 0; i < n; i++) {
        const uint64_t u = (uint64_t)src[i] - (uint64_t)lo;
        outside |= u | (range - u);
        dst[i] = (int32_t)((uint32_t)u + first);
    }
    if (outside >> 63 == 0) return true;
    for (int64_t i = 0; i < n; i++) dst[i] = (int32_t)((src[i] >= lo && src[i] <= hi ? src[i] : lo) - 1);
    return false;
}

// What both directions share: the list of batches and parts, the threads.
struct Job {
    std::vector<Batch> batches;
    std::vector<Part> parts;
    std::atomic<int> next{0};                 // next part to take
    std::atomic<bool> stop{false};
    std::vector<std::atomic<int>> left;       // parts of a batch still to do
    int threads = 1;

    // words of `hw` host and `dw` device bytes each; parts end at XF_PAGE
    // multiples of the host address
    void add(int seg, const void *host, int64_t n, int64_t hw, int64_t dw, int64_t part_bytes)
    {
        int64_t at = 0;
        while (at < n) {
            Batch b{seg, at, 0, 0};
            while (at < n && b.n * dw < XF_BATCH) {
                const uintptr_t p = (uintptr_t)host + (uintptr_t)(at * hw);
                int64_t bytes = part_bytes >= XF_PAGE ? XF_PAGE - (int64_t)(p & (XF_PAGE - 1)) : part_bytes;
                int64_t m = std::max<int64_t>(1, bytes / hw);
                m = std::min(m, n - at);
                m = std::min(m, XF_BATCH / dw - b.n);
                parts.push_back(Part{(int)batches.size(), at, m, b.n * dw});
                b.parts++;
                b.n += m;
                at += m;
            }
            batches.push_back(b);
        }
    }
    // the next part, if its batch is below `upto` (any for -1); -1: none
    int take(int upto)
    {
        int k = next.load(std::memory_order_relaxed);
        do {
            if (k >= (int)parts.size() || (upto >= 0 && parts[k].batch >= upto)) return -1;
        } while (!next.compare_exchange_weak(k, k + 1, std::memory_order_relaxed));
        return k;
    }
    void ready(int64_t host_bytes)
    {
        left = std::vector<std::atomic<int>>(batches.size());
        for (size_t k = 0; k < batches.size(); k++) left[k].store(batches[k].parts, std::memory_order_relaxed);
        const int64_t hw = std::max<int64_t>(1, (int64_t)std::thread::hardware_concurrency());
        threads = (int)std::max<int64_t>(1, std::min<int64_t>({XF_THREADS, hw, host_bytes / XF_PER_THREAD, (int64_t)parts.size()}));
    }
};

int64_t part_size(int64_t host_bytes)
{
    return host_bytes >= 16 * XF_PAGE ? XF_PAGE : std::max<int64_t>(128 << 10, host_bytes / 16);
}

// A wait for another thread: some microseconds of polling, about as long as one
// part takes, then the processor is offered to others at each poll.  (A process
// may have fewer of them than threads: nine million words in and nine out on 4
// processors 8.4 ms with polling alone and 4.5 so, on 2 10.7 and 6.7; on 16 3.3
// and 3.4.)
struct Spin {
    int polls = 0;
    void operator()()
    {
        if (++polls <= 256) _mm_pause();
        else std::this_thread::yield();
    }
};

int events_ready(elfel_hip_ctx *c)
{
    for (auto &e : c->xfer_ev)
        if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
            e = nullptr;
            return set_err(c, ELFEL_EHIP, "hipEventCreate failed");
        }
    return 0;
}

// One array of a small transfer: n words of 4 or 8 bytes; gap: the destination's
// blocks of 2^PAD_LOG2 words lie that many words apart.
struct Move {
    const void *src;
    void *dst;
    int64_t n;
    int word, gap;
};
struct Moves {
    Move m[XF_MOVES];
};

// 64 KB 9 us and 1 MB 35 us, where four copies of a quarter each take 21 and 54.
__global__ __launch_bounds__(256) void k_move(Moves M)
{
    const Move m = M.m[blockIdx.y];
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < m.n; i += (int64_t)gridDim.x * 256) {
        if (m.word == 8) ((uint64_t *)m.dst)[padded(i, m.gap)] = ((const uint64_t *)m.src)[i];
        else ((uint32_t *)m.dst)[i] = ((const uint32_t *)m.src)[i];
    }
}

int64_t round64(int64_t n) { return (n + 63) & ~(int64_t)63; }

// `need` bytes of the context's own pinned memory that no earlier transfer still
// reads; null: there is none.
char *small_room(elfel_hip_ctx *c, int64_t need)
{
    if (need > XF_SMALL) return nullptr;
    if (!c->xs && !(c->xs = pin(XF_SMALL))) return nullptr;
    if (c->xs_at + need > XF_SMALL) {
        if (hipStreamSynchronize(c->stream) != hipSuccess) return nullptr;
        c->xs_at = 0;
    }
    return (char *)c->xs + c->xs_at;
}

int launch_moves(elfel_hip_ctx *c, const Moves &M, int n)
{
    int64_t most = 0;
    for (int k = 0; k < n; k++) most = std::max(most, M.m[k].n);
    hipLaunchKernelGGL(k_move, dim3((unsigned)std::min<int64_t>(ceil_div(most, 256), 256), (unsigned)n), dim3(256), 0, c->stream, M);
    HIPCHK(c, hipGetLastError());
    return 0;
}

}  // namespace

void transfer_user(int device, bool add)
{
    Ring &R = rings[device];
    std::lock_guard<std::mutex> g(R.life);
    R.users += add ? 1 : -1;
    if (R.users == 0 && R.mem) {
        if (R.pinned) hipHostFree(R.mem);
        else free(R.mem);
        R.mem = nullptr;
    }
}

int to_host(elfel_hip_ctx *c, const HostOut *segs, int nseg)
{
    static_assert(XF_SLOTS <= sizeof(c->xfer_ev) / sizeof(c->xfer_ev[0]), "an event a slot");
    int64_t total = 0;
    for (int s = 0; s < nseg; s++) total += segs[s].host ? 8 * segs[s].n : 0;
    if (total == 0) {
        HIPCHK(c, hipStreamSynchronize(c->stream));
        c->xs_at = 0;
        return 0;
    }
    int64_t need = 0;
    for (int s = 0; s < nseg; s++) need += segs[s].host ? round64((segs[s].wide ? 4 : 8) * segs[s].n) : 0;
    if (char *room = nseg <= XF_MOVES ? small_room(c, need) : nullptr) {
        Moves M;
        int k = 0;
        char *at = room;
        for (int s = 0; s < nseg; s++) {
            if (!segs[s].host || segs[s].n == 0) continue;
            M.m[k++] = Move{segs[s].dev, at, segs[s].n, segs[s].wide ? 4 : 8, 0};
            at += round64((segs[s].wide ? 4 : 8) * segs[s].n);
        }
        // (one array: a copy is 3 us faster than the kernel at 64 KB, 9 at 1 MB)
        if (k == 1) HIPCHK(c, hipMemcpyAsync(M.m[0].dst, M.m[0].src, (size_t)(M.m[0].word * M.m[0].n), hipMemcpyDeviceToHost, c->stream));
        else if (int rc = launch_moves(c, M, k)) return rc;
        HIPCHK(c, hipStreamSynchronize(c->stream));
        c->xs_at = 0;
        k = 0;
        for (int s = 0; s < nseg; s++) {
            if (!segs[s].host || segs[s].n == 0) continue;
            const char *from = (const char *)M.m[k++].dst;
            if (segs[s].wide) widen((int64_t *)segs[s].host, (const int32_t *)from, segs[s].n, segs[s].base);
            else copy_out((char *)segs[s].host, from, 8 * segs[s].n);
        }
        return 0;
    }
    Job J;
    for (int s = 0; s < nseg; s++)
        if (segs[s].host && segs[s].n > 0) J.add(s, segs[s].host, segs[s].n, 8, segs[s].wide ? 4 : 8, part_size(total));
    J.ready(total);
    int rc = events_ready(c);
    if (rc) return rc;
    // the device's own work is done before the ring is taken
    HIPCHK(c, hipStreamSynchronize(c->stream));
    c->xs_at = 0;
    Ring &R = rings[c->device];
    std::lock_guard<std::mutex> hold(R.hold);
    char *base = ring_get(R);
    if (!base) return set_err(c, ELFEL_ENOMEM, "host memory for a transfer");
    const int nb = (int)J.batches.size();
    std::atomic<int> issued{0};
    std::vector<std::atomic<int>> here(nb);  // 0: not known, 1: a thread waits for it, 2: in the slot
    for (auto &h : here) h.store(0, std::memory_order_relaxed);
    auto issue = [&](int b) -> hipError_t {
        const Batch &B = J.batches[b];
        const HostOut &S = segs[B.seg];
        const int64_t dw = S.wide ? 4 : 8;
        hipError_t e = hipMemcpyAsync(base + (b % XF_SLOTS) * XF_BATCH, (const char *)S.dev + B.at * dw, (size_t)(B.n * dw),
                                      hipMemcpyDeviceToHost, c->stream);
        if (e == hipSuccess) e = hipEventRecord(c->xfer_ev[b % XF_SLOTS], c->stream);
        return e;
    };
    // one part of a batch below `upto` (of any for -1); false: there is none, or the job was stopped
    auto work = [&](int upto) -> bool {
        const int k = J.take(upto);
        if (k < 0) return false;
        const Part &P = J.parts[k];
        const int b = P.batch;
        for (Spin spin; issued.load(std::memory_order_acquire) <= b; spin())
            if (J.stop.load(std::memory_order_relaxed)) return false;
        int st = here[b].load(std::memory_order_acquire);
        if (st != 2) {
            if (st == 0 && here[b].compare_exchange_strong(st, 1)) {
                if (hipEventSynchronize(c->xfer_ev[b % XF_SLOTS]) != hipSuccess) {
                    J.stop.store(true);
                    return false;
                }
                here[b].store(2, std::memory_order_release);
            } else {
                for (Spin spin; here[b].load(std::memory_order_acquire) != 2; spin())
                    if (J.stop.load(std::memory_order_relaxed)) return false;
            }
        }
        const HostOut &S = segs[J.batches[b].seg];
        const char *src = base + (b % XF_SLOTS) * XF_BATCH + P.slot_off;
        if (S.wide) widen((int64_t *)S.host + P.at, (const int32_t *)src, P.n, S.base);
        else copy_out((char *)S.host + 8 * P.at, src, 8 * P.n);
        J.left[b].fetch_sub(1, std::memory_order_release);
        return true;
    };
    hipError_t e = hipSuccess;
    int b = 0;
    for (; b < std::min(nb, XF_SLOTS) && e == hipSuccess; b++) {
        e = issue(b);
        issued.store(b + 1, std::memory_order_release);
    }
    {
        std::vector<std::thread> team;
        auto joiner = join_on_exit(team, [] {});
        (void)joiner;
        try {
            for (int t = 1; t < J.threads && e == hipSuccess; t++)
                team.emplace_back([&] {
                    while (work(-1)) {}
                });
        } catch (...) {  // fewer threads
        }
        Spin spin;
        while (e == hipSuccess && !J.stop.load(std::memory_order_relaxed)) {
            if (b < nb && J.left[b - XF_SLOTS].load(std::memory_order_acquire) == 0) {
                e = issue(b);
                issued.store(++b, std::memory_order_release);
                continue;
            }
            // this thread sends batches and works between them; of the parts only
            // those whose batch is on its way (it would wait for itself)
            if (!work(b)) {
                if (b >= nb) break;
                spin();
            } else {
                spin = Spin();
            }
        }
        if (e != hipSuccess) J.stop.store(true);
    }
    if (e == hipSuccess && J.stop.load()) e = hipErrorUnknown;
    if (e != hipSuccess) {
        (void)hipStreamSynchronize(c->stream);
        return set_err(c, ELFEL_EHIP, std::string("copy to the host: ") + hipGetErrorString(e));
    }
    return 0;
}

int to_device(elfel_hip_ctx *c, const HostIn *segs, int nseg, bool *out_of_range)
{
    int64_t total = 0;
    for (int s = 0; s < nseg; s++) total += segs[s].host ? 8 * segs[s].n : 0;
    if (out_of_range) *out_of_range = false;
    if (total == 0) return 0;
    int64_t need = 0, gapped = 0;
    for (int s = 0; s < nseg; s++) {
        need += segs[s].host ? round64((segs[s].narrow ? 4 : 8) * segs[s].n) : 0;
        gapped += segs[s].host && segs[s].gap ? 8 * segs[s].n : 0;
    }
    if (char *room = nseg <= XF_MOVES ? small_room(c, need) : nullptr) {
        Moves M;
        int k = 0;
        bool ok = true;
        char *at = room;
        for (int s = 0; s < nseg; s++) {
            const HostIn &S = segs[s];
            if (!S.host || S.n == 0) continue;
            if (S.narrow) ok &= narrow((int32_t *)at, (const int64_t *)S.host, S.n, S.lo, S.hi);
            else memcpy(at, S.host, 8 * (size_t)S.n);
            M.m[k++] = Move{at, S.dev, S.n, S.narrow ? 4 : 8, S.gap};
            at += round64((S.narrow ? 4 : 8) * S.n);
        }
        if (int rc = launch_moves(c, M, k)) return rc;
        c->xs_at += need;
        if (out_of_range) *out_of_range = !ok;
        return 0;
    }
    Job J;
    for (int s = 0; s < nseg; s++)
        if (segs[s].host && segs[s].n > 0) J.add(s, segs[s].host, segs[s].n, 8, segs[s].narrow ? 4 : 8, part_size(total));
    J.ready(total);
    int rc = events_ready(c);
    if (rc) return rc;
    // arrays with gaps come side by side first
    if (gapped && (rc = ensure(c, c->stage64, gapped))) return rc;
    std::vector<char *> to(nseg);
    char *flat = (char *)c->stage64.p;
    for (int s = 0; s < nseg; s++) {
        to[s] = segs[s].gap ? flat : (char *)segs[s].dev;
        if (segs[s].host && segs[s].gap) flat += 8 * segs[s].n;
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    c->xs_at = 0;
    Ring &R = rings[c->device];
    std::lock_guard<std::mutex> hold(R.hold);
    char *base = ring_get(R);
    if (!base) return set_err(c, ELFEL_ENOMEM, "host memory for a transfer");
    const int nb = (int)J.batches.size();
    std::atomic<int> open{std::min(nb, XF_SLOTS)};  // batches whose slot may be filled
    std::atomic<bool> bad{false};
    auto work = [&](int upto) -> bool {  // as above
        const int k = J.take(upto);
        if (k < 0) return false;
        const Part &P = J.parts[k];
        const int b = P.batch;
        for (Spin spin; open.load(std::memory_order_acquire) <= b; spin())
            if (J.stop.load(std::memory_order_relaxed)) return false;
        const HostIn &S = segs[J.batches[b].seg];
        char *dst = base + (b % XF_SLOTS) * XF_BATCH + P.slot_off;
        if (S.narrow) {
            if (!narrow((int32_t *)dst, (const int64_t *)S.host + P.at, P.n, S.lo, S.hi)) bad.store(true);
        } else {
            memcpy(dst, (const char *)S.host + 8 * P.at, 8 * (size_t)P.n);
        }
        J.left[b].fetch_sub(1, std::memory_order_release);
        return true;
    };
    hipError_t e = hipSuccess;
    {
        std::vector<std::thread> team;
        auto joiner = join_on_exit(team, [] {});
        (void)joiner;
        try {
            for (int t = 1; t < J.threads; t++)
                team.emplace_back([&] {
                    while (work(-1)) {}
                });
        } catch (...) {  // fewer threads
        }
        Spin spin;
        int sent = 0, back = 0;  // batches sent; batches whose slot is free again
        while (sent < nb && e == hipSuccess) {
            if (J.left[sent].load(std::memory_order_acquire) == 0) {
                const Batch &B = J.batches[sent];
                const HostIn &S = segs[B.seg];
                const int64_t dw = S.narrow ? 4 : 8;
                e = hipMemcpyAsync(to[B.seg] + B.at * dw, base + (sent % XF_SLOTS) * XF_BATCH, (size_t)(B.n * dw),
                                   hipMemcpyHostToDevice, c->stream);
                if (e == hipSuccess) e = hipEventRecord(c->xfer_ev[sent % XF_SLOTS], c->stream);
                sent++;
                continue;
            }
            if (open.load(std::memory_order_relaxed) < nb && back < sent) {
                const hipError_t q = hipEventQuery(c->xfer_ev[back % XF_SLOTS]);
                if (q == hipSuccess) {
                    back++;
                    open.store(std::min(nb, back + XF_SLOTS), std::memory_order_release);
                    continue;
                }
                if (q != hipErrorNotReady) {
                    e = q;
                    break;
                }
            }
            if (work(open.load(std::memory_order_relaxed))) spin = Spin();
            else spin();
        }
        if (e != hipSuccess) J.stop.store(true);
    }
    (void)hipGetLastError();  // an unfinished event is not an error
    for (int s = 0; s < nseg && e == hipSuccess; s++)
        if (segs[s].host && segs[s].gap && (rc = copy_padded(c, segs[s].dev, to[s], segs[s].n, 8, segs[s].gap))) return rc;
    const hipError_t w = hipStreamSynchronize(c->stream);
    if (e == hipSuccess) e = w;
    if (e != hipSuccess) return set_err(c, ELFEL_EHIP, std::string("copy to the device: ") + hipGetErrorString(e));
    if (out_of_range) *out_of_range = bad.load();
    return 0;
}
