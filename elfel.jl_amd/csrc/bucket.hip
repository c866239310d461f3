// bucket.hip -- COO -> CSR/CSC build by row buckets: the entries of each major
// row brought together by one counting pass, then every row ordered, summed
// and written by one workgroup out of LDS.
//
// The result is that of the stable sort of sort.hip (SparseArrays.sparse,
// src/Assemblers.jl:121-123): within a row the entries are ordered by (minor
// index, stream position), and each run of equal minor indices is summed left
// to right.  Stream positions are distinct, so the order does not depend on
// where the counting pass happened to put an entry, and every run gives the
// same bits.
//
//   k_bk_zero     the row counts, the look-back states and the counters
//   k_bk_count    entries per major row; each entry's place in its row
//   k_bk_scan     exclusive scan of the counts (one pass, decoupled look-back),
//                 and the first row of every tile
//   k_bk_scatter  (minor, stream position) of every entry into its row
//   k_bk_items    for element blocks of equal rows, the items alone
//   k_bk_tile     per tile: rank every entry within its row, find the runs,
//                 sum them, and write the row pointers, indices and values at
//                 the place that a second look-back over the tiles gives
//   k_bk_one      all of it by one workgroup, for a few thousand entries
//
// Bytes per entry (n entries, u of them distinct): the two indices twice (32),
// its place written and read (8), the packed entry written and read (16), the
// value (8, gathered), and 12 u/n of output -- against 40 a pass of the radix
// sort and five to six passes.  Measured against it (whole calls): 1 045 458
// entries of a T3 mesh on the device 249 -> 62 us, 4608 entries 148 -> 32 us.
#include <algorithm>

#include "common.h"

#define BK_BLOCK 256
#define BK_TB 1024                  // work-items of a tile
#define BK_CAP 4096                 // entries that a tile holds
#define BK_CAP_FEW 2048             // ... of a stream of at most BK_FEW entries, or of so many that a place in a tile has 11 bits
#define BK_ROWMAX 512               // room for the last row's overhang, the rest is for those that start in the tile;
                                    // with a longer row, half and half; one longer than half goes to the sort
#define BK_FEW (256 * 1536)
#define BK_CAP_LOG2 12
#define BK_CAP_FEW_LOG2 11
#define BK_COUNT_ITEMS 2            // entries per work-item of the counting pass
#define BK_HASH_LOG2 10             // its LDS slots, twice its entries
#define BK_HASH (1 << BK_HASH_LOG2)
#define BK_SCAN_ITEMS 16
#define BK_SCAN_CHUNK (BK_BLOCK * BK_SCAN_ITEMS)

static_assert(BK_CAP <= 1 << BK_CAP_LOG2 && BK_CAP_FEW <= 1 << BK_CAP_FEW_LOG2, "the bits of a place in a tile");
static_assert(BK_HASH >= 2 * BK_BLOCK * BK_COUNT_ITEMS, "the hash of the counting pass is at most half full");

// ---- decoupled look-back -------------------------------------------------------
// (Merrill and Garland, Single-pass Parallel Prefix Scan with Decoupled
// Look-back, NVIDIA Technical Report NVR-2016-002.)  One 64-bit word per block of the scan: the upper half says whether the lower
// holds nothing yet, the block's own total or the total up to and including
// it.  Blocks take their numbers from a counter when they start, so every
// block that one waits for has started and waits only for earlier ones: the
// wait ends.  The word carries its own flag, so relaxed agent-scope accesses
// are enough.  (Words for groups of 64 blocks, counted up by atomics and read
// back 64 at a time, took 181 us where this takes 119, and wider windows of
// single blocks 139 to 193: what is waited on is the few lines that all read.)
enum { LB_EMPTY = 0, LB_TOTAL = 1, LB_PREFIX = 2 };

__device__ __forceinline__ void lb_store(uint64_t *st, uint32_t flag, uint32_t v)
{
    __hip_atomic_store(st, ((uint64_t)flag << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void lb_publish(uint64_t *st, uint32_t t, uint32_t total)
{
    lb_store(st + t, t == 0 ? LB_PREFIX : LB_TOTAL, total);
}

// The sum of the totals of blocks 0 .. t - 1, for one whole wave (the same in
// every lane); publishes the inclusive sum of block t.
__device__ __forceinline__ uint32_t lb_wait(uint64_t *st, uint32_t t, uint32_t total)
{
    const int lane = threadIdx.x & 63;
    uint32_t run = 0;
    for (int64_t hi = (int64_t)t - 1; hi >= 0; hi -= 64) {
        const int64_t j = hi - lane;
        uint64_t w;
        uint64_t have_prefix;
        do {
            w = j >= 0 ? __hip_atomic_load(st + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : (uint64_t)LB_TOTAL << 32;
            have_prefix = __ballot((uint32_t)(w >> 32) == LB_PREFIX);
            const uint64_t empty = __ballot((uint32_t)(w >> 32) == LB_EMPTY);
            // lanes nearer than the first inclusive sum must all hold something
            const uint64_t need = have_prefix ? (have_prefix & (~have_prefix + 1)) - 1 : ~0ull;
            if (!(empty & need)) break;
            __builtin_amdgcn_s_sleep(1);
        } while (true);
        const int first = have_prefix ? __builtin_ctzll(have_prefix) : 63;
        uint32_t v = lane <= first ? (uint32_t)w : 0u;
        for (int d = 32; d > 0; d >>= 1) v += (uint32_t)__shfl_xor((int)v, d, 64);
        run += v;
        if (have_prefix) break;
    }
    if (t != 0 && lane == 0) lb_store(st + t, LB_PREFIX, run + total);
    return run;
}

// ---- control words ---------------------------------------------------------------
// BK_LONG: a row longer than BK_ROWMAX exists: the tiles are those of the second
// set.  BK_TOOLONG: one that no tile holds; the kernels after the scan then
// leave every output alone.
enum { BK_T_SCAN = 0, BK_T_TILE = 1, BK_LONG = 2, BK_TOOLONG = 3, BK_NCTL = 4 };

// The first row and entry of every tile: for rows of at most BK_ROWMAX entries,
// and of at most half a tile.
struct Tiles {
    uint32_t *row, *first;
    uint32_t nt;
};
struct TileSets {
    Tiles set[2];
};

__global__ void k_bk_zero(uint4 *__restrict__ p, int64_t n4)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n4) p[i] = make_uint4(0, 0, 0, 0);
}

// ---- the stream -------------------------------------------------------------------
// A COO stream: every entry is an item of the counting pass, one entry wide.
struct CooSource {
    const int64_t *row, *col;
    int64_t nrow, ncol;
    int csc;
    __device__ __forceinline__ bool get(int64_t k, uint32_t &major, uint32_t &minor) const
    {
        const int64_t r = row[k], q = col[k];
        const bool ok = r >= 1 && r <= nrow && q >= 1 && q <= ncol;
        major = ok ? (uint32_t)(csc ? q - 1 : r - 1) : 0u;
        minor = ok ? (uint32_t)(csc ? r - 1 : q - 1) : 0u;
        return ok;
    }
    __device__ __forceinline__ bool item(int64_t k, uint32_t &major, uint32_t &wide) const
    {
        uint32_t minor;
        wide = 1;
        return get(k, major, minor);
    }
};

// The same with checked, 0-based indices.
struct CooSource32 {
    const int32_t *major, *minor;
    __device__ __forceinline__ bool get(int64_t k, uint32_t &mj, uint32_t &mn) const
    {
        mj = (uint32_t)major[k];
        mn = (uint32_t)minor[k];
        return true;
    }
    __device__ __forceinline__ bool item(int64_t k, uint32_t &mj, uint32_t &wide) const
    {
        mj = (uint32_t)major[k];
        wide = 1;
        return true;
    }
};

// The stream of an element loop: a local dof of an element is one item, as wide
// as its row of the element block.
template <int ND>
struct FormSource {
    const int32_t *edof;
    uint32_t wide[2];  // entries of the first `nfull` local rows, and of the others
    int nfull;
    __device__ __forceinline__ bool item(int64_t k, uint32_t &major, uint32_t &w) const
    {
        major = (uint32_t)edof[k];
        w = (int)((uint32_t)k % ND) < nfull ? wide[0] : wide[1];
        return true;
    }
};

// Entries per row and every item's place in its row (n items).  One atomic per entry on
// the rows' counters is bound by atomics to the same address (a million
// entries of a T3 mesh 42 us, all in one row 11 ms), so a workgroup first
// counts the rows of its entries in an LDS hash and then adds each distinct
// row once.  512 entries a workgroup: 2048 took 56 against 43 us for six million
// entries and 12 against 4 us for 4608, where the chain of hash probes of one
// work-item is the time.
template <typename Source>
__global__ __launch_bounds__(BK_BLOCK) void k_bk_count(Source src, int64_t n, uint32_t *__restrict__ cnt,
                                                       uint32_t *__restrict__ place, int *__restrict__ err)
{
    __shared__ int32_t key[BK_HASH];
    __shared__ uint32_t num[BK_HASH];
    for (int i = threadIdx.x; i < BK_HASH; i += BK_BLOCK) {
        key[i] = -1;
        num[i] = 0;
    }
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * (BK_BLOCK * BK_COUNT_ITEMS);
    uint32_t slot[BK_COUNT_ITEMS], loc[BK_COUNT_ITEMS], wide[BK_COUNT_ITEMS];
    bool bad = false;
#pragma unroll
    for (int q = 0; q < BK_COUNT_ITEMS; q++) {
        const int64_t k = base + q * BK_BLOCK + threadIdx.x;
        uint32_t major = 0;
        wide[q] = 0;
        if (k < n && !src.item(k, major, wide[q])) bad = true;
        slot[q] = major;
    }
#pragma unroll
    for (int q = 0; q < BK_COUNT_ITEMS; q++) {
        if (base + q * BK_BLOCK + threadIdx.x < n) {
            const int32_t r = (int32_t)slot[q];
            uint32_t s = ((uint32_t)r * 2654435761u) >> (32 - BK_HASH_LOG2);
            while (true) {
                const int32_t old = atomicCAS(&key[s], -1, r);
                if (old == -1 || old == r) break;
                s = (s + 1) & (BK_HASH - 1);
            }
            slot[q] = s;
            loc[q] = atomicAdd(&num[s], wide[q]);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < BK_HASH; i += BK_BLOCK)
        if (key[i] >= 0) num[i] = atomicAdd(&cnt[key[i]], num[i]);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < BK_COUNT_ITEMS; q++) {
        const int64_t k = base + q * BK_BLOCK + threadIdx.x;
        if (k < n) place[k] = num[slot[q]] + loc[q];
    }
    if (bad) atomicOr(err, DERR_RANGE);
}

// cnt[0 .. nmaj] (cnt[nmaj] = 0) -> the rows' first entries, and for every tile
// t of both sets the first row that starts at or after t * tile with that start
// (tile nt: nmaj and n).  A row's interval (s, s + len] holds the tile boundaries
// that the next row is the first to reach.
template <int CAP>
__global__ __launch_bounds__(BK_BLOCK) void k_bk_scan(uint32_t *__restrict__ cnt, int64_t nmaj, uint32_t n, TileSets T,
                                                      uint64_t *__restrict__ st, uint32_t *__restrict__ ctl)
{
    __shared__ uint32_t wsum[BK_BLOCK / 64], sh_b, sh_base;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if (tid == 0) sh_b = atomicAdd(&ctl[BK_T_SCAN], 1u);
    __syncthreads();
    const uint32_t b = sh_b;
    const int64_t r0 = (int64_t)b * BK_SCAN_CHUNK + tid * BK_SCAN_ITEMS;
    uint32_t v[BK_SCAN_ITEMS], sum = 0, most = 0;
#pragma unroll
    for (int i = 0; i < BK_SCAN_ITEMS; i += 4) {
        uint4 q = make_uint4(0, 0, 0, 0);
        if (r0 + i + 3 <= nmaj) q = *(const uint4 *)(cnt + r0 + i);
        else {
            if (r0 + i <= nmaj) q.x = cnt[r0 + i];
            if (r0 + i + 1 <= nmaj) q.y = cnt[r0 + i + 1];
            if (r0 + i + 2 <= nmaj) q.z = cnt[r0 + i + 2];
        }
        v[i] = q.x; v[i + 1] = q.y; v[i + 2] = q.z; v[i + 3] = q.w;
    }
#pragma unroll
    for (int i = 0; i < BK_SCAN_ITEMS; i++) {
        sum += v[i];
        most = max(most, v[i]);
    }
    uint32_t inc = sum;
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)inc, d, 64);
        if (lane >= d) inc += o;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    uint32_t woff = 0, total = 0;
    for (int k = 0; k < BK_BLOCK / 64; k++) {
        if (k < w) woff += wsum[k];
        total += wsum[k];
    }
    if (w == 0) {
        if (lane == 0) lb_publish(st, b, total);
        const uint32_t base = lb_wait(st, b, total);
        if (lane == 0) sh_base = base;
    }
    __syncthreads();
    uint32_t s = sh_base + woff + inc - sum;
    if (most > BK_ROWMAX) ctl[BK_LONG] = 1u;
    if (most > CAP / 2) ctl[BK_TOOLONG] = 1u;
#pragma unroll
    for (int i = 0; i < BK_SCAN_ITEMS; i++) {
        const uint32_t c = v[i];
        v[i] = s;
        const uint32_t e = s + c;  // c = 0 past the last row
        for (uint32_t t = s / (CAP - BK_ROWMAX) + 1; t <= e / (CAP - BK_ROWMAX); t++) {
            T.set[0].row[t] = (uint32_t)(r0 + i + 1);
            T.set[0].first[t] = e;
        }
        for (uint32_t t = s / (CAP / 2) + 1; t <= e / (CAP / 2); t++) {
            T.set[1].row[t] = (uint32_t)(r0 + i + 1);
            T.set[1].first[t] = e;
        }
        s += c;
    }
#pragma unroll
    for (int i = 0; i < BK_SCAN_ITEMS; i += 4) {
        if (r0 + i + 3 <= nmaj) *(uint4 *)(cnt + r0 + i) = make_uint4(v[i], v[i + 1], v[i + 2], v[i + 3]);
        else {
            if (r0 + i <= nmaj) cnt[r0 + i] = v[i];
            if (r0 + i + 1 <= nmaj) cnt[r0 + i + 1] = v[i + 1];
            if (r0 + i + 2 <= nmaj) cnt[r0 + i + 2] = v[i + 2];
        }
    }
    if (b == 0 && tid < 2) {
        const Tiles &t = T.set[tid];
        t.row[0] = 0;
        t.first[0] = 0;
        t.row[t.nt] = (uint32_t)nmaj;
        t.first[t.nt] = n;
    }
}

// The entries of a row side by side, each packed with its row's first entry in
// the bits above `bits` = minor bits + kbits (those that overflow drop out: a
// tile spans at most 2^12 entries, and starts no row that many after its first), its minor index and its stream position.
template <typename Source>
__global__ __launch_bounds__(BK_BLOCK) void k_bk_scatter(Source src, int64_t n, const uint32_t *__restrict__ start,
                                                         const uint32_t *__restrict__ place, int bits, int kbits,
                                                         uint64_t *__restrict__ packed, const uint32_t *__restrict__ ctl)
{
    const int64_t k = (int64_t)blockIdx.x * BK_BLOCK + threadIdx.x;
    if (k >= n || ctl[BK_TOOLONG] != 0) return;
    uint32_t major, minor;
    src.get(k, major, minor);
    const uint32_t s = start[major];
    packed[(int64_t)s + place[k]] = ((uint64_t)s << bits) | ((uint64_t)minor << kbits) | (uint64_t)k;
}

// The same for the stream of an element loop: work-item x is the entry of local
// row a and local column b of an element.
template <int ND>
__global__ __launch_bounds__(BK_BLOCK) void k_bk_scatter_form(FormMap map, int64_t n2, const int32_t *__restrict__ edof,
                                                              const uint32_t *__restrict__ start,
                                                              const uint32_t *__restrict__ place, int bits, int kbits,
                                                              uint64_t *__restrict__ packed)
{
    const int64_t x = (int64_t)blockIdx.x * BK_BLOCK + threadIdx.x;
    if (x >= n2) return;
    const int64_t ea = x / ND, e = ea / ND;
    const int b = (int)(x - ea * ND), a = (int)(ea - e * ND);
    if (b >= map.ncol[a]) return;
    const uint32_t s = start[edof[ea]];
    const uint64_t k = (uint64_t)(e * map.nmat + map.pos[a * ND + b]);
    packed[(int64_t)s + place[ea] + b] = ((uint64_t)s << bits) | ((uint64_t)(uint32_t)edof[e * ND + b] << kbits) | k;
}

// Where every item of an element stream is nd entries wide, the items alone go
// into their rows, 4 bytes in place of 8 nd, and the tile forms the words from
// them and the element dofs (scatter and tile: elasticity T6 200^2 152 -> 130
// us, T4 36^3 97 -> 93; plain assembly of elasticity T6 400^2 0.89 -> 0.73 ms).
__global__ __launch_bounds__(BK_BLOCK) void k_bk_items(int64_t items, uint32_t nd, const int32_t *__restrict__ edof,
                                                       const uint32_t *__restrict__ start,
                                                       const uint32_t *__restrict__ place, int32_t *__restrict__ list,
                                                       const uint32_t *__restrict__ ctl)
{
    const int64_t x = (int64_t)blockIdx.x * BK_BLOCK + threadIdx.x;
    if (x >= items || ctl[BK_TOOLONG] != 0) return;
    list[(start[edof[x]] + place[x]) / nd] = (int32_t)x;
}

// Entry P of the rows, as a tile whose first entry is s0 compares it: the row
// begin in the tile, the minor index, the stream position.
struct PackedWords {
    const uint64_t *packed;
    __device__ __forceinline__ uint64_t get(uint32_t P, uint32_t s0, const uint32_t *, int bits, int) const
    {
        return packed[P] - ((uint64_t)s0 << bits);
    }
};
struct ItemWords {
    const int32_t *list, *edof;
    double inv;  // 1 / nd
    uint32_t nd;
    int csc;
    __device__ __forceinline__ uint32_t over(uint32_t x) const { return (uint32_t)(((double)x + 0.5) * inv); }  // x / nd
    __device__ __forceinline__ uint64_t get(uint32_t P, uint32_t s0, const uint32_t *start, int bits, int kbits) const
    {
        const uint32_t slot = over(P), b = P - slot * nd, ea = (uint32_t)list[slot], e = over(ea), a = ea - e * nd;
        const uint32_t minor = (uint32_t)edof[e * nd + b], row = start[edof[ea]];
        const uint64_t k = (uint64_t)e * (nd * nd) + (csc ? b + nd * a : a + nd * b);
        return ((uint64_t)(row - s0) << bits) | ((uint64_t)minor << kbits) | k;
    }
};

// acc + v[j] + ... + v[e - 1], left to right; four loads at a time
__device__ __forceinline__ double run_sum(const double *v, int j, int e, double acc)
{
    for (; j + 4 <= e; j += 4) {
        const double a = v[j], b = v[j + 1], c = v[j + 2], d = v[j + 3];
        acc += a;
        acc += b;
        acc += c;
        acc += d;
    }
    for (; j < e; j++) acc += v[j];
    return acc;
}

// the set bits of positions p .. e - 1
__device__ __forceinline__ int bits_between(const uint64_t *m, int p, int e)
{
    int n = 0;
    for (int x = p >> 6; x <= (e - 1) >> 6; x++) {
        uint64_t g = m[x];
        if (x == p >> 6) g &= ~0ull << (p & 63);
        if (x == (e - 1) >> 6) g &= ~0ull >> (63 - ((e - 1) & 63));
        n += __popcll(g);
    }
    return n;
}

// One workgroup per tile of whole rows: those that start in a tile's entries, each
// of at most half of it.  An entry less the tile's first entry (in the row field)
// is (row begin, minor, stream position), so entries of a tile compare as plain
// integers.  Each work-item counts, for four neighbouring entries at once, how
// many entries of their rows are smaller: broadcast reads from LDS, for the 20
// to 100 entries of a finite-element row as many steps as a sorting network
// would take, without its exchanges.
// What bounds it beyond the gathers: a tile takes its number from one counter
// (11 ns each, in turn) and looks back over the tiles before it, so few large
// tiles: 3584 entries by 1024 work-items, two workgroups a CU, against 1536 by
// 512, four a CU, 139 -> 119 us (11.5 million entries), 81 -> 69 (6 million),
// 1024 work-items on 1536 entries 165.  A stream that such small tiles put on
// the CUs once (BK_FEW) is faster so: 4608 entries 11.4 -> 8.8 us, 394 000 whole
// calls 49.9 -> 48.7, 551 000 53.2 -> 54.0.
//
// SUM: the values and (LOAD) the load vector; else the sort order.  LOAD: the
// load-vector entries of a dof are those of the (element, local dof) pairs on
// the diagonal of its row, which the run of the diagonal holds in stream
// order; they are gathered with the values and summed by the work-item of that
// run (one work-item a row that looked for the run and then loaded them one
// after the other: 4.5 million entries 108 us, now 84).
//
// tile_rows: the rows of a tile, their entries in sk (and kr: entry q * BK_TB + tid); ~0 past m.
// Gives back the runs up to the tile's end.  place: where the tile's runs begin.
template <bool SUM, bool LOAD, int CAP, typename Place>
__device__ __forceinline__ uint32_t tile_rows(uint64_t *sk, uint64_t *ss, uint16_t *se, uint64_t *hm, uint64_t *dm,
                                              uint32_t *sh_base, uint64_t *kr, int m, uint32_t s0, int64_t row0, int64_t row1,
                                              const uint32_t *start, const double *__restrict__ vals,
                                              const double *__restrict__ fvals, uint32_t nd, int bits, int kbits,
                                              const Place &place, const BucketOut &o)
{
    constexpr int ROUNDS = CAP / BK_TB;
    static_assert(CAP % BK_TB == 0, "a tile is a whole number of rounds");
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
#pragma unroll
    for (int q = 0; q < ROUNDS; q++) {
        const int p = q * BK_TB + tid;
        const uint32_t b = (uint32_t)(kr[q] >> bits);
        if (p < m && (p == m - 1 || (uint32_t)(sk[p + 1] >> bits) != b)) se[b] = (uint16_t)(p + 1);
    }
    __syncthreads();
    for (int p = 4 * tid; p < m; p += 4 * BK_TB) {
        const uint64_t k0 = sk[p], k1 = sk[p + 1], k2 = sk[p + 2], k3 = sk[p + 3];  // past m: larger than any entry
        const int last = min(p + 3, m - 1);
        const int b = (int)(k0 >> bits), e = se[(uint32_t)(sk[last] >> bits)];
        int c0 = b, c1 = b, c2 = b, c3 = b, j = b;
        for (; j + 4 <= e; j += 4) {
            const uint64_t o0 = sk[j], o1 = sk[j + 1], o2 = sk[j + 2], o3 = sk[j + 3];
            c0 += (o0 < k0) + (o1 < k0) + (o2 < k0) + (o3 < k0);
            c1 += (o0 < k1) + (o1 < k1) + (o2 < k1) + (o3 < k1);
            c2 += (o0 < k2) + (o1 < k2) + (o2 < k2) + (o3 < k2);
            c3 += (o0 < k3) + (o1 < k3) + (o2 < k3) + (o3 < k3);
        }
        for (; j < e; j++) {
            const uint64_t o = sk[j];
            c0 += o < k0;
            c1 += o < k1;
            c2 += o < k2;
            c3 += o < k3;
        }
        ss[c0] = k0;
        if (p + 1 < m) ss[c1] = k1;
        if (p + 2 < m) ss[c2] = k2;
        if (p + 3 < m) ss[c3] = k3;
    }
    __syncthreads();
    // runs: entries that differ in more than the stream position start one
    const uint64_t kmask = (1ull << kbits) - 1;
    const uint32_t mmask = (uint32_t)((1ull << (bits - kbits)) - 1);
    double vr[ROUNDS], fr[ROUNDS];
#pragma unroll
    for (int q = 0; q < ROUNDS; q++) {
        const int p = q * BK_TB + tid;
        kr[q] = p < m ? ss[p] : 0;
        if constexpr (SUM) vr[q] = p < m ? vals[kr[q] & kmask] : 0.0;
        else if (p < m) o.perm[(int64_t)s0 + p] = (int32_t)(kr[q] & kmask);
        if constexpr (LOAD) {
            const uint32_t k = (uint32_t)(kr[q] & kmask), el = k / (nd * nd), ab = k - el * (nd * nd), a = ab / nd;
            const bool d = p < m && ab == a * (nd + 1);
            fr[q] = d && SUM ? fvals[(int64_t)el * nd + a] : 0.0;
            const uint64_t g = __ballot(d);
            if (lane == 0) dm[q * (BK_TB / 64) + w] = g;
        }
    }
#pragma unroll
    for (int q = 0; q < ROUNDS; q++) {
        const int p = q * BK_TB + tid;
        const uint64_t h = __ballot(p < m && (p == 0 || (ss[p - 1] >> kbits) != (kr[q] >> kbits)));
        if (lane == 0) hm[q * (BK_TB / 64) + w] = h;
    }
    __syncthreads();
    // runs before each word of hm (every wave computes them, lanes as words)
    constexpr int WORDS = CAP / 64, PER = (WORDS + 63) / 64;  // PER words a lane
    uint32_t pc = 0;
#pragma unroll
    for (int i = 0; i < PER; i++) pc += PER * lane + i < WORDS ? (uint32_t)__popcll(hm[PER * lane + i]) : 0u;
    uint32_t inc = pc;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)inc, d, 64);
        if (lane >= d) inc += o;
    }
    const uint32_t total = (uint32_t)__shfl((int)inc, 63, 64);
    if (tid == 0) place.publish(total);
    double *sv = (double *)sk, *sf = (double *)ss;
    uint32_t un[ROUNDS];
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int q = 0; q < ROUNDS; q++) {
        const int p = q * BK_TB + tid, word = q * (BK_TB / 64) + w;
        un[q] = (uint32_t)__shfl((int)(inc - pc), word / PER, 64) + (uint32_t)__popcll(hm[word] & lt);
#pragma unroll
        for (int i = 1; i < PER; i++) un[q] += word % PER >= i ? (uint32_t)__popcll(hm[word - i]) : 0u;
        if (p < m) {
            if constexpr (SUM) sv[p] = vr[q];
            if constexpr (SUM && LOAD) sf[p] = fr[q];
            se[p] = (uint16_t)un[q];
        }
    }
    if (tid == 0) se[m] = (uint16_t)total;
    __syncthreads();
    // the sums, while the tiles before this one finish theirs
#pragma unroll
    for (int q = 0; q < ROUNDS; q++) {
        const int p = q * BK_TB + tid, word = q * (BK_TB / 64) + w;
        if (p >= m || !((hm[word] >> lane) & 1)) continue;
        if constexpr (!SUM && !LOAD) continue;
        // the next run's start, or the tile's end
        const uint64_t above = lane == 63 ? 0ull : hm[word] >> (lane + 1);
        int e = above ? p + 1 + __builtin_ctzll(above) : -1;
        for (int x = word + 1; e < 0; x++) {
            if (x * 64 >= m) e = m;
            else if (hm[x]) e = x * 64 + __builtin_ctzll(hm[x]);
        }
        if constexpr (SUM) vr[q] = run_sum(sv, p + 1, e, vr[q]);
        if constexpr (LOAD) {
            // the diagonal's run, and no other, has entries of a local dof with itself
            const int n = bits_between(dm, p, e);
            if (n == 0) continue;
            if constexpr (SUM) {
                double f = 0.0;
                if (n == e - p) {
                    f = run_sum(sf, p + 1, e, fr[q]);
                } else {  // an element with two local dofs of one number
                    int cnt = 0;
                    for (int j = p; j < e; j++)
                        if ((dm[j >> 6] >> (j & 63)) & 1) f = cnt++ == 0 ? sf[j] : f + sf[j];
                }
                o.F[(uint32_t)(kr[q] >> kbits) & mmask] = 0.0 + f;  // start! zeros the vector, assemble! adds
            } else {
                const int64_t to = ((int64_t)s0 + (int64_t)(kr[q] >> bits)) / nd;
                int cnt = 0;
                for (int j = p; j < e; j++) {
                    if (!((dm[j >> 6] >> (j & 63)) & 1)) continue;
                    const uint32_t k = (uint32_t)(ss[j] & kmask), el = k / (nd * nd), ab = k - el * (nd * nd);
                    o.fperm[to + cnt++] = (int32_t)(el * nd + ab / nd);
                }
            }
        }
    }
    if (w == 0) {
        const uint32_t base = place.wait(total);
        if (lane == 0) *sh_base = base;
    }
    __syncthreads();
    const uint32_t base = *sh_base;
#pragma unroll
    for (int q = 0; q < ROUNDS; q++) {
        const int p = q * BK_TB + tid, word = q * (BK_TB / 64) + w;
        if (p >= m || !((hm[word] >> lane) & 1)) continue;
        const int64_t u = (int64_t)base + un[q];
        o.ind[u] = (int32_t)((uint32_t)(kr[q] >> kbits) & mmask);
        if constexpr (SUM) o.val[u] = vr[q];
        else o.seg[u] = (int32_t)(s0 + p);
    }
    for (int64_t r = row0 + tid; r < row1; r += BK_TB) {
        const uint32_t b = start[r];
        o.ptr[r] = (int32_t)(base + se[b - s0]);
        if constexpr (LOAD && SUM) {
            if (start[r + 1] == b) o.F[r] = 0.0;  // a dof of no element
        }
        if constexpr (LOAD && !SUM) o.fbeg[r] = (int32_t)(b / nd);
    }
    return base + total;
}

__device__ __forceinline__ void tell_build(uint32_t nnz, const uint32_t *start, int64_t nmaj, uint32_t nd, bool sum, bool load,
                                           const BucketOut &o, int32_t *nnz_dev, int32_t *told)
{
    o.ptr[nmaj] = (int32_t)nnz;
    if (!sum) {
        o.seg[nnz] = (int32_t)start[nmaj];
        if (load) o.fbeg[nmaj] = (int32_t)(start[nmaj] / nd);
    }
    *nnz_dev = (int32_t)nnz;
    told[0] = (int32_t)nnz;
    told[1] = 0;
    told[2] = 0;
}

struct AfterTiles {
    uint64_t *st;
    uint32_t t;
    __device__ __forceinline__ void publish(uint32_t total) const { lb_publish(st, t, total); }
    __device__ __forceinline__ uint32_t wait(uint32_t total) const { return lb_wait(st, t, total); }
};

template <bool SUM, bool LOAD, int CAP, typename Words>
__global__ __launch_bounds__(BK_TB) void k_bk_tile(Words words, const double *__restrict__ vals,
                                                   const double *__restrict__ fvals, uint32_t nd,
                                                   const uint32_t *__restrict__ start, TileSets T, int64_t nmaj,
                                                   int bits, int kbits, uint64_t *__restrict__ st,
                                                   uint32_t *__restrict__ ctl, const int *__restrict__ err, BucketOut o,
                                                   int32_t *__restrict__ nnz_dev, int32_t *__restrict__ told)
{
    constexpr int ROUNDS = CAP / BK_TB;
    __shared__ __align__(16) uint64_t sk[CAP + 4];  // the entries by row; then the values in sorted order
    __shared__ uint64_t ss[CAP];                    // the entries, sorted
    __shared__ uint16_t se[CAP + 1];                // end of a row, at its begin; then the runs before an entry
    __shared__ uint64_t hm[CAP / 64];               // one bit per entry that starts a run
    __shared__ uint64_t dm[LOAD ? CAP / 64 : 1];    // one bit per entry of a local dof with itself
    __shared__ uint32_t sh_t, sh_base;
    const int tid = threadIdx.x;
    // nothing is written when an index was out of range or a row is too long
    // (the flags were set by earlier kernels: the same for every workgroup)
    if (*err != 0 || ctl[BK_TOOLONG] != 0) {
        if (blockIdx.x == 0 && tid == 0) {
            told[0] = 0;
            told[1] = *err;
            told[2] = (int32_t)ctl[BK_TOOLONG];
        }
        return;
    }
    const bool longrows = ctl[BK_LONG] != 0;
    const uint32_t nt = longrows ? T.set[1].nt : T.set[0].nt;
    const uint32_t *trow = longrows ? T.set[1].row : T.set[0].row, *tstart = longrows ? T.set[1].first : T.set[0].first;
    if (blockIdx.x >= nt) return;  // launched for the larger of the two sets: nt numbers are taken
    if (tid == 0) sh_t = atomicAdd(&ctl[BK_T_TILE], 1u);
    __syncthreads();
    const uint32_t t = sh_t;
    const int64_t row0 = trow[t], row1 = trow[t + 1];
    const uint32_t s0 = tstart[t];
    const int m = (int)(tstart[t + 1] - s0);  // <= CAP
    uint64_t kr[ROUNDS];
#pragma unroll
    for (int q = 0; q < ROUNDS; q++) {
        const int p = q * BK_TB + tid;
        kr[q] = p < m ? words.get(s0 + (uint32_t)p, s0, start, bits, kbits) : ~0ull;
    }
#pragma unroll
    for (int q = 0; q < ROUNDS; q++) sk[q * BK_TB + tid] = kr[q];
    __syncthreads();
    const uint32_t nnz = tile_rows<SUM, LOAD, CAP>(sk, ss, se, hm, dm, &sh_base, kr, m, s0, row0, row1, start, vals, fvals, nd,
                                                   bits, kbits, AfterTiles{st, t}, o);
    if (t == nt - 1 && tid == 0) tell_build(nnz, start, nmaj, nd, SUM, LOAD, o, nnz_dev, told);
}

// ---- one workgroup for all ----------------------------------------------------------
// The whole build of a stream of at most BK_ONE entries and BK_ONE_ROWS rows by
// one workgroup, its counts and places in LDS (145 KB): one launch in place of
// five, whose latencies are the time of so small a call (whole calls on the
// device, five launches -> one: 72 entries 35 -> 25 us, 1152 37 -> 27, 4608 39
// -> 34, 5832 39.6 -> 36.7).
#define BK_ONE 6144
#define BK_ONE_ROWS 8191

// Item x of a stream: its row, column and stream position; false: none, or
// (COO, *bad) an index out of range.
template <typename Source>
__device__ __forceinline__ bool one_item(const Source &src, uint32_t x, uint32_t &major, uint32_t &minor, uint32_t &k, bool &bad)
{
    k = x;
    const bool ok = src.get(x, major, minor);
    bad |= !ok;
    return ok;
}
struct FormItems {
    FormMap map;
    const int32_t *edof;
};
__device__ __forceinline__ bool one_item(const FormItems &f, uint32_t x, uint32_t &major, uint32_t &minor, uint32_t &k, bool &bad)
{
    const uint32_t nd = (uint32_t)f.map.nd, ea = x / nd, b = x - ea * nd, e = ea / nd, a = ea - e * nd;
    if ((int)b >= f.map.ncol[a]) return false;
    major = (uint32_t)f.edof[ea];
    minor = (uint32_t)f.edof[e * nd + b];
    k = e * (uint32_t)f.map.nmat + (uint32_t)f.map.pos[a * nd + b];
    return true;
}

struct FirstPlace {
    __device__ __forceinline__ void publish(uint32_t) const {}
    __device__ __forceinline__ uint32_t wait(uint32_t) const { return 0; }
};

template <bool SUM, bool LOAD, typename Source>
__global__ __launch_bounds__(BK_TB) void k_bk_one(Source src, uint32_t items, int m, const double *__restrict__ vals,
                                                  const double *__restrict__ fvals, uint32_t nd, int nmaj, int bits, int kbits,
                                                  BucketOut o, int32_t *__restrict__ nnz_dev, int32_t *__restrict__ told)
{
    constexpr int ROUNDS = BK_ONE / BK_TB, PER = (BK_ONE_ROWS + 1) / BK_TB;
    __shared__ __align__(16) uint64_t sk[BK_ONE + 4];
    __shared__ uint64_t ss[BK_ONE];
    __shared__ uint16_t se[BK_ONE + 1];
    __shared__ uint64_t hm[BK_ONE / 64], dm[LOAD ? BK_ONE / 64 : 1];
    __shared__ __align__(16) uint32_t first[BK_ONE_ROWS + 1];  // row r's entries at r + 1, then the end of its places so far
    __shared__ uint32_t wsum[BK_TB / 64], sh_base, sh_bad;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
#pragma unroll
    for (int i = 0; i < PER; i += 4) *(uint4 *)(first + PER * tid + i) = make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int q = 0; q < ROUNDS; q++) sk[q * BK_TB + tid] = ~0ull;
    if (tid == 0) sh_bad = 0;
    __syncthreads();
    uint32_t major[ROUNDS], minor[ROUNDS], k[ROUNDS];
    bool bad = false, is[ROUNDS];
    auto load = [&](uint32_t x0) {  // ROUNDS items a work-item at once
#pragma unroll
        for (int q = 0; q < ROUNDS; q++) {
            const uint32_t x = x0 + q * BK_TB + tid;
            is[q] = x < items && one_item(src, x, major[q], minor[q], k[q], bad);
        }
    };
    for (uint32_t x0 = 0; x0 < items; x0 += ROUNDS * BK_TB) {
        load(x0);
#pragma unroll
        for (int q = 0; q < ROUNDS; q++)
            if (is[q]) atomicAdd(&first[major[q] + 1], 1u);
    }
    if (bad) sh_bad = 1;
    __syncthreads();
    // first[r + 1] = entries of the rows before r: where r's places begin
    uint32_t v[PER], sum = 0;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        v[i] = first[PER * tid + i];
        sum += v[i];
    }
    uint32_t inc = sum;
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t u = (uint32_t)__shfl_up((int)inc, d, 64);
        if (lane >= d) inc += u;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    if (sh_bad) {
        if (tid == 0) {
            told[0] = 0;
            told[1] = DERR_RANGE;
            told[2] = 0;
        }
        return;
    }
    uint32_t at = inc - sum;
    for (int i = 0; i < w; i++) at += wsum[i];
#pragma unroll
    for (int i = 0; i < PER; i++) {
        first[PER * tid + i] = at;
        at += v[i];
    }
    __syncthreads();
    // every entry to a place of its row; the row begin in its key is the row's
    // first place, which the runs of smaller rows end at
    for (uint32_t x0 = 0; x0 < items; x0 += ROUNDS * BK_TB) {
        if (items > ROUNDS * BK_TB) load(x0);
#pragma unroll
        for (int q = 0; q < ROUNDS; q++)
            if (is[q]) {
                const uint32_t p = atomicAdd(&first[major[q] + 1], 1u);
                sk[p] = ((uint64_t)major[q] << bits) | ((uint64_t)minor[q] << kbits) | k[q];
            }
    }
    __syncthreads();
    uint64_t kr[ROUNDS];
#pragma unroll
    for (int q = 0; q < ROUNDS; q++) {
        const int p = q * BK_TB + tid;
        kr[q] = sk[p];
        if (p < m) kr[q] = (kr[q] & ((1ull << bits) - 1)) | ((uint64_t)first[kr[q] >> bits] << bits);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < ROUNDS; q++) sk[q * BK_TB + tid] = kr[q];
    __syncthreads();
    const uint32_t nnz = tile_rows<SUM, LOAD, BK_ONE>(sk, ss, se, hm, dm, &sh_base, kr, m, 0u, 0, nmaj, first, vals, fvals, nd,
                                                      bits, kbits, FirstPlace{}, o);
    if (tid == 0) tell_build(nnz, first, nmaj, nd, SUM, LOAD, o, nnz_dev, told);
}

// ---- host -------------------------------------------------------------------------
// (heat Q4 4096x4096, 268 million entries, is one bit over the larger tiles: the
// plain assembly takes 30.0 ms by the sort, 8.0 with the smaller ones)
static int bk_cap(int64_t n, int64_t nmin)
{
    return n <= BK_FEW || bits_for(nmin) + bits_for(n) + BK_CAP_LOG2 > 64 ? BK_CAP_FEW : BK_CAP;
}
static int64_t bk_tiles(int64_t n, int cap, bool longrows) { return n / (longrows ? cap / 2 : cap - BK_ROWMAX) + 1; }
static int64_t bk_scan_blocks(int64_t nmaj) { return ceil_div(nmaj + 1, BK_SCAN_CHUNK); }
// words zeroed before a build: control words, the look-back states, the counts
static int64_t bk_zero_words(int64_t n, int64_t nmaj)
{
    return (BK_NCTL + 2 * bk_scan_blocks(nmaj) + 2 * bk_tiles(n, BK_CAP_FEW, true) + nmaj + 1 + 7) & ~(int64_t)3;
}

// The scratch: the packed entries, what is zeroed (control words, look-back
// states, row counts), the tiles' first rows and entries, the items' places.
namespace {
struct Scratch {
    uint64_t *packed, *st_scan, *st_tile;
    uint32_t *ctl, *cnt, *place;
    TileSets T;
    int cap;
    int64_t zero_words, nt, nsb;
};
}  // namespace

static size_t scratch_bytes(int64_t n, int64_t items, int64_t nmaj)
{
    return 8 * (size_t)n + 4 * (size_t)items + 4 * (size_t)bk_zero_words(n, nmaj) + 
           8 * (size_t)(bk_tiles(n, BK_CAP_FEW, false) + bk_tiles(n, BK_CAP_FEW, true) + 2) + 80;
}

static Scratch scratch_layout(void *p, int64_t n, int64_t nmaj, int64_t nmin)
{
    Scratch S;
    S.cap = bk_cap(n, nmin);
    S.nt = bk_tiles(n, S.cap, true);
    S.nsb = bk_scan_blocks(nmaj);
    S.packed = (uint64_t *)p;
    S.ctl = (uint32_t *)(S.packed + n);
    S.ctl += ((16 - ((uintptr_t)S.ctl & 15)) & 15) / 4;  // 16-byte words
    S.st_scan = (uint64_t *)(S.ctl + BK_NCTL);
    S.st_tile = S.st_scan + S.nsb;
    S.cnt = (uint32_t *)(S.st_tile + S.nt);
    S.cnt += ((16 - ((uintptr_t)S.cnt & 15)) & 15) / 4;
    S.zero_words = bk_zero_words(n, nmaj);
    S.place = S.ctl + S.zero_words;
    for (int q = 0; q < 2; q++) {
        Tiles &t = S.T.set[q];
        t.nt = (uint32_t)bk_tiles(n, S.cap, q);
        t.row = S.place;
        t.first = t.row + t.nt + 1;
        S.place = t.first + t.nt + 1;
    }
    return S;
}

size_t bucket_scratch_bytes(int64_t n, int64_t nmaj) { return scratch_bytes(n, n, nmaj); }
size_t bucket_form_bytes(const FormMap &m, int64_t E, int64_t ndofs)
{
    return scratch_bytes(E * m.nmat, E * m.nd, ndofs);
}

// Where the buckets apply: the counts are zeroed, scanned and read over all
// rows, so a matrix of far more rows than entries keeps the sort; so does one of
// more than 128 entries a row on average, more than any element's mesh here has,
// where the counting pass waits for few counters if the stream is in no order
// (650 000 entries in random order, whole calls by the buckets and by the sort:
// rows of 600 721 and 645 us, of 250 696 and 649, of 120 571 and 685); and a
// minor index, a stream position and a place in a tile have to fit one 64-bit
// word.
bool bucket_takes(int64_t n, int64_t nmaj, int64_t nmin)
{
    return n > 0 && n < INT32_MAX && nmaj <= 16 * n + 65536 && (n <= BK_ONE || n <= 128 * nmaj) &&
           bits_for(nmin) + bits_for(n) + BK_CAP_FEW_LOG2 <= 64;
}
bool bucket_form_takes(const FormMap &m, int64_t E, int64_t ndofs)
{
    return E * m.nd < INT32_MAX && bucket_takes(E * m.nmat, ndofs, ndofs);
}

template <bool SUM, bool LOAD, typename Words>
static void launch_tiles(elfel_hip_ctx *c, const Scratch &S, const Words &words, const double *vals, const double *fvals, int nd,
                         int64_t nmaj, int bits, int kbits, const BucketOut &o, int32_t *nnz_dev, int32_t *told)
{
    hipLaunchKernelGGL((S.cap == BK_CAP ? k_bk_tile<SUM, LOAD, BK_CAP, Words> : k_bk_tile<SUM, LOAD, BK_CAP_FEW, Words>),
                       dim3((unsigned)S.nt), dim3(BK_TB), 0, c->stream, words, vals, fvals, (uint32_t)nd, S.cnt, S.T, nmaj, bits,
                       kbits, S.st_tile, S.ctl, (const int *)c->dscal.p + 1, o, nnz_dev, told);
}

static bool one_takes(int64_t n, int64_t nmaj) { return n <= BK_ONE && nmaj <= BK_ONE_ROWS; }

static void launch_zero_scan(elfel_hip_ctx *c, const Scratch &S, bool zero, int64_t n, int64_t nmaj)
{
    if (zero)
        hipLaunchKernelGGL(k_bk_zero, dim3(ceil_div(S.zero_words / 4, 256)), dim3(256), 0, c->stream, (uint4 *)S.ctl,
                           S.zero_words / 4);
    else
        hipLaunchKernelGGL((S.cap == BK_CAP ? k_bk_scan<BK_CAP> : k_bk_scan<BK_CAP_FEW>), dim3((unsigned)S.nsb),
                           dim3(BK_BLOCK), 0, c->stream, S.cnt, nmaj, (uint32_t)n,
                           S.T, S.st_scan, S.ctl);
}

template <typename Source>
static int run_coo(elfel_hip_ctx *c, void *scratch, const Source &src, int64_t n, const double *val, int64_t nmaj,
                   int64_t nmin, const BucketOut &o)
{
    const Scratch S = scratch_layout(scratch, n, nmaj, nmin);
    const int kbits = bits_for(n), bits = kbits + bits_for(nmin);
    int *err = (int *)c->dscal.p + 1;
    if (one_takes(n, nmaj)) {
        hipLaunchKernelGGL((k_bk_one<true, false, Source>), dim3(1), dim3(BK_TB), 0, c->stream, src, (uint32_t)n, (int)n, val,
                           (const double *)nullptr, 1u, (int)nmaj, bits, kbits, o, (int32_t *)c->dscal.p + 2,
                           (int32_t *)c->told + 4);
        HIPCHK(c, hipGetLastError());
        HIPCHK(c, hipStreamSynchronize(c->stream));
        return 0;
    }
    launch_zero_scan(c, S, true, n, nmaj);
    hipLaunchKernelGGL(k_bk_count<Source>, dim3(ceil_div(n, BK_BLOCK * BK_COUNT_ITEMS)), dim3(BK_BLOCK), 0, c->stream, src,
                       n, S.cnt, S.place, err);
    launch_zero_scan(c, S, false, n, nmaj);
    hipLaunchKernelGGL(k_bk_scatter<Source>, dim3(ceil_div(n, BK_BLOCK)), dim3(BK_BLOCK), 0, c->stream, src, n, S.cnt,
                       S.place, bits, kbits, S.packed, S.ctl);
    // told: words 0-3 are the context's result's, these 4-7
    launch_tiles<true, false>(c, S, PackedWords{S.packed}, val, nullptr, 1, nmaj, bits, kbits, o, (int32_t *)c->dscal.p + 2,
                              (int32_t *)c->told + 4);
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return 0;
}

int bucket_coo(elfel_hip_ctx *c, void *scratch, int64_t n, const int64_t *row, const int64_t *col, const double *val,
               int64_t nrow, int64_t ncol, int csc, int32_t *ptr, int32_t *ind, double *out, int *flags, bool *toolong,
               int64_t *nnz)
{
    const BucketOut o{ptr, ind, out, nullptr, nullptr, nullptr, nullptr, nullptr};
    const int rc = run_coo(c, scratch, CooSource{row, col, nrow, ncol, csc}, n, val, csc ? ncol : nrow, csc ? nrow : ncol, o);
    const int32_t *told = (const int32_t *)c->told + 4;
    *nnz = told[0];
    *flags = told[1];
    *toolong = told[2] != 0;
    return rc;
}

int bucket_coo32(elfel_hip_ctx *c, void *scratch, int64_t n, const int32_t *row, const int32_t *col, const double *val,
                 int64_t nrow, int64_t ncol, int csc, int32_t *ptr, int32_t *ind, double *out, bool *toolong, int64_t *nnz)
{
    const BucketOut o{ptr, ind, out, nullptr, nullptr, nullptr, nullptr, nullptr};
    const int rc = run_coo(c, scratch, CooSource32{csc ? col : row, csc ? row : col}, n, val, csc ? ncol : nrow,
                           csc ? nrow : ncol, o);
    const int32_t *told = (const int32_t *)c->told + 4;
    *nnz = told[0];
    *toolong = told[2] != 0;
    return rc;
}

// ---- the stream of an element loop ------------------------------------------------
void form_square(FormMap &m, int nd, int csc)
{
    m.nd = nd;
    m.nmat = nd * nd;
    for (int a = 0; a < nd; a++) {
        m.ncol[a] = (uint8_t)nd;
        for (int b = 0; b < nd; b++) m.pos[a * nd + b] = (int16_t)(csc ? b + nd * a : a + nd * b);
    }
}

struct DofTables {
    const int32_t *conn[2], *dof[2], *edof[2];
    int nen[2], ncomp[2], encomp[2];
};

__global__ __launch_bounds__(256) void k_form_dofs(FormMap m, DofTables T, int64_t n, int32_t *__restrict__ edof)
{
    const int64_t x = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (x >= n) return;
    const int64_t e = x / m.nd;
    const FormMap::Src s = m.src[x - e * m.nd];
    edof[x] = s.cell ? T.edof[s.field][e * T.encomp[s.field] + s.comp]
                     : T.dof[s.field][(int64_t)T.conn[s.field][e * T.nen[s.field] + s.node] * T.ncomp[s.field] + s.comp];
}

int form_dofs(elfel_hip_ctx *c, const FormMap &m, int32_t *edof)
{
    DofTables T;
    for (int f = 0; f < 2; f++) {
        const Field &F = c->f[f];
        T.conn[f] = (const int32_t *)F.conn.p;
        T.dof[f] = (const int32_t *)F.dof.p;
        T.edof[f] = (const int32_t *)F.edof.p;
        T.nen[f] = F.nen;
        T.ncomp[f] = F.ncomp;
        T.encomp[f] = F.edof_ncomp;
    }
    const int64_t n = c->f[0].E * m.nd;
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_form_dofs, dim3(ceil_div(n, 256)), dim3(256), 0, c->stream, m, T, n, edof);
    HIPCHK(c, hipGetLastError());
    return 0;
}

__global__ __launch_bounds__(256) void k_form_keys(FormMap m, int64_t n2, const int32_t *__restrict__ edof, int minor_bits,
                                                   uint64_t *__restrict__ keys, uint64_t *__restrict__ fkeys)
{
    const int64_t x = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (x >= n2) return;
    const int64_t ea = x / m.nd, e = ea / m.nd;
    const int b = (int)(x - ea * m.nd), a = (int)(ea - e * m.nd);
    const uint32_t major = (uint32_t)edof[ea];
    if (b < m.ncol[a])
        keys[e * m.nmat + m.pos[a * m.nd + b]] = ((uint64_t)major << minor_bits) | (uint64_t)(uint32_t)edof[e * m.nd + b];
    if (fkeys && b == 0) fkeys[ea] = (uint64_t)major;
}

int form_keys(elfel_hip_ctx *c, const FormMap &m, int64_t E, const int32_t *edof, int minor_bits, uint64_t *keys,
              uint64_t *fkeys)
{
    const int64_t n2 = E * m.nd * m.nd;
    if (n2 == 0) return 0;
    hipLaunchKernelGGL(k_form_keys, dim3((unsigned)((n2 + 255) / 256)), dim3(256), 0, c->stream, m, n2, edof, minor_bits,
                       keys, fkeys);
    HIPCHK(c, hipGetLastError());
    return 0;
}

template <int ND>
static void launch_form(elfel_hip_ctx *c, const Scratch &S, const FormMap &m, int64_t E, const int32_t *edof,
                        int64_t ndofs, int bits, int kbits, bool square)
{
    FormSource<ND> src{edof, {m.ncol[0], m.ncol[ND - 1]}, ND};
    for (int a = ND - 1; a > 0 && m.ncol[a] != m.ncol[0]; a--) src.nfull = a;
    const int64_t items = E * ND, n2 = items * ND;
    launch_zero_scan(c, S, true, E * m.nmat, ndofs);
    hipLaunchKernelGGL(k_bk_count<FormSource<ND>>, dim3(ceil_div(items, BK_BLOCK * BK_COUNT_ITEMS)), dim3(BK_BLOCK), 0,
                       c->stream, src, items, S.cnt, S.place, (int *)c->dscal.p + 1);
    launch_zero_scan(c, S, false, E * m.nmat, ndofs);
    if (square)
        hipLaunchKernelGGL(k_bk_items, dim3(ceil_div(items, BK_BLOCK)), dim3(BK_BLOCK), 0, c->stream, items, (uint32_t)ND, edof,
                           S.cnt, S.place, (int32_t *)S.packed, S.ctl);
    else
        hipLaunchKernelGGL(k_bk_scatter_form<ND>, dim3((unsigned)((n2 + BK_BLOCK - 1) / BK_BLOCK)), dim3(BK_BLOCK), 0,
                           c->stream, m, n2, edof, S.cnt, S.place, bits, kbits, S.packed);
}

int bucket_form(elfel_hip_ctx *c, void *scratch, const FormMap &m, int64_t E, const int32_t *edof, int64_t ndofs,
                const double *vals, const double *fvals, const BucketOut &o)
{
    const int64_t n = E * m.nmat;
    const Scratch S = scratch_layout(scratch, n, ndofs, ndofs);
    const int kbits = bits_for(n), bits = kbits + bits_for(ndofs);
    const bool sum = vals != nullptr, load = m.nvec > 0;
    hipEvent_t ev = nullptr;
    tm_begin(c, ELFEL_PH_SORT, &ev);
    if (one_takes(n, ndofs)) {
        auto kern = sum ? (load ? k_bk_one<true, true, FormItems> : k_bk_one<true, false, FormItems>)
                        : (load ? k_bk_one<false, true, FormItems> : k_bk_one<false, false, FormItems>);
        hipLaunchKernelGGL(kern, dim3(1), dim3(BK_TB), 0, c->stream, FormItems{m, edof}, (uint32_t)(E * m.nd * m.nd), (int)n,
                           vals, fvals, (uint32_t)m.nd, (int)ndofs, bits, kbits, o, (int32_t *)c->dscal.p, (int32_t *)c->told);
        HIPCHK(c, hipGetLastError());
        tm_end(c, ELFEL_PH_SORT, ev);
        tm_begin(c, ELFEL_PH_REDUCE, &ev);  // nothing is left for it
        tm_end(c, ELFEL_PH_REDUCE, ev);
        return 0;
    }
    // (a block of nd x nd entries in either order: form_square's)
    bool square = m.nmat == m.nd * m.nd;
    const int csc = m.pos[1] == 1;
    for (int a = 0; a < m.nd; a++)
        for (int b = 0; square && b < m.nd; b++) square = m.pos[a * m.nd + b] == (csc ? b + m.nd * a : a + m.nd * b);
    switch (m.nd) {
#define F(N) case N: launch_form<N>(c, S, m, E, edof, ndofs, bits, kbits, square); break
        F(2); F(3); F(4); F(6); F(8); F(9); F(11); F(12); F(15);
#undef F
    default: return set_err(c, ELFEL_ENOTSUP, "internal: element dof count without a bucket kernel");
    }
    HIPCHK(c, hipGetLastError());
    tm_end(c, ELFEL_PH_SORT, ev);
    tm_begin(c, ELFEL_PH_REDUCE, &ev);
    int32_t *nnz_dev = (int32_t *)c->dscal.p, *told = (int32_t *)c->told;
    const ItemWords items{(const int32_t *)S.packed, edof, 1.0 / m.nd, (uint32_t)m.nd, csc};
    const PackedWords packed{S.packed};
#define TILES(SUM, LOAD, W) launch_tiles<SUM, LOAD>(c, S, W, vals, fvals, m.nd, ndofs, bits, kbits, o, nnz_dev, told)
    if (load && !square) return set_err(c, ELFEL_ENOTSUP, "internal: a load vector without a square element block");
    if (load) sum ? TILES(true, true, items) : TILES(false, true, items);
    else if (square) sum ? TILES(true, false, items) : TILES(false, false, items);
    else sum ? TILES(true, false, packed) : TILES(false, false, packed);
#undef TILES
    HIPCHK(c, hipGetLastError());
    tm_end(c, ELFEL_PH_REDUCE, ev);
    return 0;
}
