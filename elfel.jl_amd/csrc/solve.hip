// solve.hip -- Jacobi-preconditioned conjugate gradients on the free block of
// the assembled matrix, replacing the driver's `K[1:nu,1:nu] \ (F - K*T)[1:nu]`
// (test/test_heat.jl:73-76) for SPD problems.
//
// FP64 PCG: textbook PCG (Saad, Iterative Methods for Sparse Linear Systems,
// Alg. 9.1) with every vector and the matrix in FP64; when the recurrence
// residual reaches the tolerance, the true residual b - A x is formed and
// replaces it (the iteration goes on if the true one is not yet small enough).
// Mixed: the same PCG with an FP32 matrix copy, FP32 r, z, p and q, the FP64
// iterate x (x += alpha p in FP64), FP64 dot products, and reliable updates
// (Sleijpen & van der Vorst, Computing 56, 1996): whenever the recurrence
// residual has fallen by RU_DROP since the last update, the FP64 residual
// b - A x is formed with the FP64 matrix and replaces the FP32 one, and the
// search direction is kept unless the recurrence has drifted below half the
// true residual (then p restarts from z).  An iteration of the mixed solve
// moves about 0.55 of the bytes of an FP64 one.  With an FP32 iterate (added
// into the FP64 solution at each update) the iteration count rose with the
// mesh: on heat Q4 with lognormal(0, 1) conductivity, +9 % over FP64 PCG at
// 256x256 and +69 % at 1024x1024 (numpy emulation of this code), +45 % at
// 4096x4096 (measured: 19224 against 13280); the FP64 iterate keeps the late,
// small corrections that an FP32 one rounds away (+9 % at 1024x1024).
// Updates at every 10x drop, or never restarting, failed to converge at
// 4096x4096 (FP32 iterate).
// Convergence is declared on the FP64 residual: ||b - A x|| / ||b|| <= tol.
//
// Storage: the free-free block in SELL-64 (one slice per 64 consecutive rows,
// each slice as wide as its longest row, entries column-major inside the
// slice), built once per solve from the CSR result: one thread per row, every
// load coalesced, data columns left out (their part of b is formed once with
// the CSR matrix).  When every free column lies within a 16-bit offset of its
// row (banded numberings: structured grids, RCM-ordered meshes) the columns
// are stored as int16 offsets, 2 bytes per entry instead of 4.
// Per iteration two or three kernels on a fixed grid of 4 workgroups per CU
// (grid-stride loops): q = A p, one partial of p.q per workgroup, with the new
// direction formed on the way or by a kernel of its own before it; and the r / z
// update (every workgroup first sums the p.q partials itself, in the same order)
// with partials of r.z and r.r.  No atomics
// and no extra reduction launches; every run gives the same bits.  The CG
// scalars stay on the device and the host reads the residual every CHECK
// iterations.
// Systems that fit on the chip run all of that in one launch, with the same
// sums and bits: small ones, and on grid-like numberings up to 786 000 rows FP64
// or 2.1 million mixed, with the matrix in registers (k_cg_small,
// k_cg_resident; k_cg_one for a few thousand rows).
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "nine.h"

int env_int(const char *name, int dflt);  // reuse.hip

#define SV_BLOCK 256
#define CHECK 8
#define SELL_UNROLL 12  // slices at most this wide are read with every load in flight at once
#ifndef UP_ROWS
#define UP_ROWS 4       // rows of the update likewise
#endif
#ifndef RU_DROP
#define RU_DROP 1e-2   // reliable update when the recurrence residual has dropped by this factor
#endif
#ifndef RU_KEEP
#define RU_KEEP 0.5    // keep p at an update while ||r recurrence|| >= RU_KEEP ||r true||
#endif

namespace {

// Scalars (double) on the device, for the host's convergence checks.
enum { S_RZ = 0, S_RR = 1, S_BB = 2, S_RR64 = 3, S_ALPHA = 4, S_RZS = 5 /* two words */, S_IT = 7, S_RREC = 8, S_LOST = 9, S_NS = 10 };

__device__ __forceinline__ double block_sum(double v, double *sh)
{
    for (int d = 32; d > 0; d >>= 1) v += __shfl_down(v, d, 64);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();  // sh may still be read by a previous call
    if (lane == 0) sh[w] = v;
    __syncthreads();
    double s = 0.0;
    for (int k = 0; k < (int)(blockDim.x >> 6); k++) s += sh[k];
    return s;  // the same value in every thread
}

// The block of rows that a workgroup takes: workgroups go to the XCDs in turn, so
// XCD x (of 8) takes the x-th eighth of the blocks, and the neighbouring rows
// that a product gathers are read into one L2 instead of three (the solve on
// 1500x1300 quads 240 -> 227 ms).
__device__ __forceinline__ uint32_t row_block()
{
    const uint32_t g = gridDim.x, b = blockIdx.x;
    return (g & 7) == 0 ? (b & 7) * (g >> 3) + (b >> 3) : b;
}

// Fixed-order sum of the g partials of the previous kernel (every block of
// the grid computes it, in the same order, so all get the same bits).
__device__ __forceinline__ double sum_partials(const double *p, int g, double *sh)
{
    double v = 0.0;
    for (int i = threadIdx.x; i < g; i += blockDim.x) v += p[i];
    return block_sum(v, sh);
}

// ---- SELL-64 construction ----------------------------------------------------
// Free entries per row, and whether a free column lies farther than a 16-bit
// offset from the row (then the column indices stay 32-bit).
__global__ void k_sell_rowlen(int64_t nfree, const int32_t *__restrict__ ptr, const int32_t *__restrict__ ind,
                              uint32_t *__restrict__ len, uint32_t *__restrict__ far)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nfree) return;
    uint32_t k = 0, f = 0;
    for (int32_t j = ptr[i]; j < ptr[i + 1]; j++) {
        if (ind[j] >= nfree) continue;
        k++;
        const int64_t d = (int64_t)ind[j] - i;
        f |= (d < -32768 || d > 32767) ? 1u : 0u;
    }
    len[i] = k;
    if (f) *far = 1u;
}

// Column of entry k of a SELL row: 32-bit index, or 16-bit offset from the row.
template <typename C>
__device__ __forceinline__ int32_t sell_col(C c, int64_t row);
template <>
__device__ __forceinline__ int32_t sell_col<int32_t>(int32_t c, int64_t row) { return c; }
template <>
__device__ __forceinline__ int32_t sell_col<int16_t>(int16_t c, int64_t row) { return (int32_t)row + (int32_t)c; }

// One wave per slice: width = longest row; writes 64 * width (the slice size).
__global__ void k_sell_width(int64_t nfree, int64_t nslices, const uint32_t *__restrict__ len,
                             uint32_t *__restrict__ size, uint32_t *__restrict__ wide)
{
    const int64_t s = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    if (s >= nslices) return;
    const int64_t row = s * 64 + lane;
    uint32_t w = row < nfree ? len[row] : 0u;
    for (int d = 32; d > 0; d >>= 1) w = max(w, (uint32_t)__shfl_down((int)w, d, 64));
    if (lane == 0) {  // it holds the maximum
        size[s] = 64u * w;
        if (w > SELL_UNROLL) wide[0] = 1u;
    }
}

template <typename C>
__global__ void k_sell_fill(int64_t nfree, const int32_t *__restrict__ ptr, const int32_t *__restrict__ ind,
                            const double *__restrict__ val, const uint32_t *__restrict__ off,
                            C *__restrict__ col, double *__restrict__ v64, float *__restrict__ v32)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t s = i >> 6;
    const int lane = (int)(i & 63);
    if (s * 64 >= nfree) return;
    const uint32_t o = off[s], w = (off[s + 1] - o) >> 6;
    uint32_t k = 0;
    if (i < nfree) {
        for (int32_t j = ptr[i]; j < ptr[i + 1]; j++) {
            const int32_t cj = ind[j];
            if (cj >= nfree) continue;
            const size_t at = (size_t)o + (size_t)k * 64 + lane;
            col[at] = sizeof(C) == 4 ? (C)cj : (C)(cj - i);
            v64[at] = val[j];
            if (v32) v32[at] = (float)val[j];
            k++;
        }
    }
    for (; k < w; k++) {  // padding: a zero on the row's own column (or row 0 beyond nfree)
        const size_t at = (size_t)o + (size_t)k * 64 + lane;
        col[at] = sizeof(C) == 4 ? (C)(i < nfree ? i : 0) : (C)0;  // rows past nfree are never read
        v64[at] = 0.0;
        if (v32) v32[at] = 0.f;
    }
}

// Slices whose every slot holds one column offset for all its rows (each row
// of the slice has its k-th entry at row + d_k: the stencil of a structured
// grid away from its boundary) are flagged, and their offsets d_k are kept
// once per slot; such a slice reads no per-entry column at all.  many: how many
// of every UNI_STEP-th slice are.  One wave per slice.
#define UNI_STEP 16
template <typename C>
__global__ void k_sell_uniform(int64_t nfree, int64_t nslices, const uint32_t *__restrict__ off,
                               const C *__restrict__ col, uint32_t *__restrict__ uflag, int32_t *__restrict__ uoff,
                               uint32_t *__restrict__ many)
{
    const int64_t s = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    if (s >= nslices) return;
    const int64_t i = s * 64 + lane;
    const uint32_t o = off[s], w = (off[s + 1] - o) >> 6, sb = o >> 6;
    bool uniform = true;
    for (uint32_t k = 0; k < w; k++) {
        const int32_t d = sell_col<C>(col[(size_t)o + (size_t)k * 64 + lane], i) - (int32_t)i;
        const int32_t d0 = __shfl(d, 0, 64);  // row s*64 < nfree: lane 0 is a real row
        if (__ballot((i < nfree) && (d != d0)) != 0ull) uniform = false;
        if (lane == 0) uoff[sb + k] = d0;
    }
    if (lane == 0) {
        uflag[s] = uniform ? 1u : 0u;
        if (uniform && s % UNI_STEP == 0) atomicAdd(many, 1u);
    }
}

// Without them: a slice of no entries alone is flagged (there is no slot that its
// rows could read).
__global__ void k_sell_empty(int64_t nslices, const uint32_t *__restrict__ off, uint32_t *__restrict__ uflag)
{
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s < nslices) uflag[s] = off[s] == off[s + 1] ? 1u : 0u;
}

// A slice for the resident solve (k_cg_resident): its rows' entries lie on the
// diagonal and its two neighbours, in one run of three neighbouring offsets
// below and one above -- the three grid rows of a quadrilateral's or triangle's
// stencil; a row may lack any of the nine.  The record is the runs' first
// offsets; nslow counts the slices that have no such runs.  One wave per slice.
__global__ void k_sell_rec(int64_t nfree, int64_t nslices, const uint32_t *__restrict__ off,
                           const int16_t *__restrict__ col, const uint32_t *__restrict__ len, int2 *__restrict__ rec,
                           uint32_t *__restrict__ nslow)
{
    const int64_t s = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    if (s >= nslices) return;
    const int64_t i = s * 64 + lane;
    const uint32_t o = off[s], w = i < nfree ? len[i] : 0u;
    NineRuns R;
    for (uint32_t k = 0; k < w; k++) R.add(col[(size_t)o + (size_t)k * 64 + lane]);
    for (int t = 32; t > 0; t >>= 1) {
        R.lo = min(R.lo, __shfl_xor(R.lo, t, 64));
        R.hi = min(R.hi, __shfl_xor(R.hi, t, 64));
        R.lo_end = max(R.lo_end, __shfl_xor(R.lo_end, t, 64));
        R.hi_end = max(R.hi_end, __shfl_xor(R.hi_end, t, 64));
    }
    if (lane == 0) {
        rec[s] = make_int2(R.lo, R.hi);  // NINE_NONE: no entry is there, and what is read for it meets zeros
        if (!R.fit()) atomicAdd(nslow, 1u);
    }
}

struct SellU {
    const uint32_t *uflag;  // per slice: 1 when every slot has one column offset for all rows
    const int32_t *uoff;    // per slot: that offset
};

// A slice's start, width and uniform flag (the first loads of its row).
struct SliceMeta {
    uint32_t o, w;
    uint32_t uni;
};
__device__ __forceinline__ SliceMeta slice_meta(int64_t i, const uint32_t *__restrict__ off, SellU U)
{
    // one wave holds one slice: s is the same on every lane
    const int64_t s = __builtin_amdgcn_readfirstlane((int)(i >> 6));
    const uint32_t o = off[s];
    return SliceMeta{o, (off[s + 1] - o) >> 6, U.uflag[s]};
}

// What a product gathers: a vector, or the search direction z + beta p formed
// on the way (the new direction of a neighbour's row is not written yet).
template <typename T>
struct VecGather {
    const T *__restrict__ x;
    struct Part { T a; };
    __device__ __forceinline__ Part load(int32_t j) const { return Part{x[j]}; }
    __device__ __forceinline__ T value(Part v) const { return v.a; }
};
template <typename T>
struct DirGather {
    const T *__restrict__ z, *__restrict__ p;
    T beta;
    struct Part { T a, b; };
    __device__ __forceinline__ Part load(int32_t j) const { return Part{z[j], p[j]}; }
    __device__ __forceinline__ T value(Part v) const { return v.a + beta * v.b; }
};

// A row's loads (slices of at most SELL_UNROLL entries), issued together ahead
// of the sums: the values and (uniform slices) the gathers at once, else the
// columns, then the gathers.  In uniform slices the slots past w are skipped
// (w is the same on every lane), else they read slot 0 again (in bounds) and
// add nothing; the values, read once per product, bypass the caches that hold
// the vectors.
template <typename T, typename C, typename V>
struct RowLoads {
    T v[SELL_UNROLL];
    typename V::Part x[SELL_UNROLL];

    __device__ __forceinline__ void load(int64_t i, const C *__restrict__ col, const T *__restrict__ val,
                                         const V &g, SellU U, SliceMeta m)
    {
        const int lane = (int)(i & 63);
        const T *vp = val + m.o + lane;
        const C *c = col + m.o + lane;
        const int32_t *d = U.uoff + (m.o >> 6);
        const int32_t ri = (int32_t)i;
        if (m.uni) {
            // all offsets at once (the array is as much longer than its slots):
            // read slot by slot behind k < w they came one scalar load after
            // another, 0.2 us each
            int32_t dk[SELL_UNROLL];
#pragma unroll
            for (int k = 0; k < SELL_UNROLL; k++) dk[k] = d[k];
#pragma unroll
            for (int k = 0; k < SELL_UNROLL; k++) {
                if (k < (int)m.w) {
                    v[k] = __builtin_nontemporal_load(vp + (size_t)k * 64);
                    x[k] = g.load(ri + dk[k]);
                }
            }
        } else {
            int32_t cj[SELL_UNROLL];
#pragma unroll
            for (int k = 0; k < SELL_UNROLL; k++) {
                const int kk = k < (int)m.w ? k : 0;
                v[k] = vp[(size_t)kk * 64];
                cj[k] = sell_col<C>(c[(size_t)kk * 64], i);
            }
#pragma unroll
            for (int k = 0; k < SELL_UNROLL; k++) x[k] = g.load(cj[k]);
        }
    }
    __device__ __forceinline__ T sum(const V &g, SliceMeta m) const
    {
        T acc = T(0);
#pragma unroll
        for (int k = 0; k < SELL_UNROLL; k++)
            if (k < (int)m.w) acc += v[k] * g.value(x[k]);
        return acc;
    }
};

template <typename T, typename C, typename V>
__device__ __forceinline__ T sell_row(int64_t i, const C *__restrict__ col, const T *__restrict__ val, const V &g, SellU U,
                                      SliceMeta m)
{
    if (m.w <= SELL_UNROLL) {
        RowLoads<T, C, V> R;
        R.load(i, col, val, g, U, m);
        return R.sum(g, m);
    }
    const int lane = (int)(i & 63);
    const T *v = val + m.o + lane;
    const C *c = col + m.o + lane;
    const int32_t *d = U.uoff + (m.o >> 6);
    const int32_t ri = (int32_t)i;
    T acc = T(0);
    if (m.uni) {
#pragma unroll 4
        for (uint32_t k = 0; k < m.w; k++) acc += v[(size_t)k * 64] * g.value(g.load(ri + d[k]));
    } else {
#pragma unroll 4
        for (uint32_t k = 0; k < m.w; k++) acc += v[(size_t)k * 64] * g.value(g.load(sell_col<C>(c[(size_t)k * 64], i)));
    }
    return acc;
}

// The CG kernels run on a fixed grid of G workgroups with grid-stride loops
// over the rows; each writes one partial per workgroup per dot product.
//   parts layout: pq[G], rz[G], rr[G], aux[G]
//
// Three kernels an iteration: the new direction with the last step of the
// iterate (k_cg_dir), the product, the update.  Or two: the product forms the new
// direction itself, p = z + beta p, for its own row (stored, in the other of two
// buffers) and for each entry it gathers, and adds the last step while it holds
// the last direction, a pass over z, p and p' and a launch less, but every
// gather is of two vectors.  All sums are the same, so the bits are.  Measured,
// three kernels against two, us an iteration: mixed heat Q4 1300^2 36.9, 36.2, T3
// 1000^2 26.7, 25.2, T4 60^3 19.7, 18.7, Q4 4096^2 284, 279; FP64 the same 62.2,
// 66.1; 38.5, 39.9; 23.7, 25.0; 538, 588; rows in random order, T3 1000^2, mixed
// 67, 134, FP64 98, 198; wide rows of two dofs a node, elasticity T6 250^2, 34,
// 41 and 42, 63.  So two kernels for FP32 vectors where most slices are uniform,
// three for the rest.
// Neighbouring blocks' rows on one XCD take 5 us off mixed heat Q4 1500x1300.
// Two rows of loads in flight per work-item measured slower than one (57 us
// against 45: 144 registers, three waves a SIMD where the grid has four), and so
// did taking the grid neighbours' values from the next lane in place of two
// thirds of the gathers (46.6 us: L1 is not the bound).

// The iterate's last step, x += alpha p: the FP64 solve updates its FP64
// iterate (TX = double).  The mixed solve adds alpha p to an FP32 accumulator
// of the last few iterations' steps (TX = float), which k_cg_dir folds into the
// FP64 iterate every CHECK iterations: an FP32 iterate itself absorbs the late,
// small corrections (x + alpha p rounds back to x; the mixed solve then needed
// 69 % more iterations than FP64 PCG on heat Q4 1024^2 against 9 % with an FP64
// iterate, numpy emulation of this code), while the accumulator holds only
// corrections, so each keeps its FP32 relative precision.
//
// DIR: p = z + beta p_old into p, x += alpha p_old; else the product with p_old
// as it is.  q = A p; partial p.q.  SUMS: workgroup 0 leaves this iteration's r.z
// in rzs[par] (else k_cg_dir has).
template <typename T, typename TX, typename C, bool DIR, bool SUMS>
__global__ __launch_bounds__(SV_BLOCK, DIR ? 4 : 1) void k_cg_spmv(int64_t n, const uint32_t *__restrict__ off,
                                                      const C *__restrict__ col, const T *__restrict__ val,
                                                      SellU U, const T *__restrict__ z, const T *__restrict__ p_old,
                                                      T *__restrict__ p, T *__restrict__ q, TX *__restrict__ x,
                                                      const double *__restrict__ part_rz, double *__restrict__ sc, int par,
                                                      double *__restrict__ part_pq)
{
    __shared__ double sh[SV_BLOCK / 64];
    using V = typename std::conditional<DIR, DirGather<T>, VecGather<T>>::type;
    const int64_t stride = (int64_t)gridDim.x * SV_BLOCK;
    // (columns beyond 16 bits are not neighbours: there the blocks in order are
    // up to 10 % faster)
    const uint32_t blk = sizeof(C) == 2 ? row_block() : blockIdx.x;
    int64_t i = (int64_t)blk * SV_BLOCK + threadIdx.x;
    V g;
    if constexpr (DIR) { g.z = z; g.p = p_old; } else g.x = p_old;
    RowLoads<T, C, V> R0;
    SliceMeta m0{0, 0, 0};
    if (i < n) {
        m0 = slice_meta(i, off, U);
        if (m0.w <= SELL_UNROLL) R0.load(i, col, val, g, U, m0);
    }
    double rz = 0.0;
    if constexpr (SUMS) {
        rz = sum_partials(part_rz, gridDim.x, sh);
        if (blockIdx.x == 0 && threadIdx.x == 0) sc[S_RZS + par] = rz;
    }
    TX alphax = TX(0);
    if constexpr (DIR) {
        const double rz_old = sc[S_RZS + (par ^ 1)];
        g.beta = (T)(rz_old != 0.0 ? rz / rz_old : 0.0);
        alphax = (TX)sc[S_ALPHA];
    }
    double d = 0.0;
    auto finish = [&](int64_t r, T y) {
        T pr = p_old[r];
        if constexpr (DIR) {
            x[r] += alphax * (TX)pr;
            pr = z[r] + g.beta * pr;
            p[r] = pr;
        }
        q[r] = y;
        d += (double)pr * (double)y;
    };
    while (i < n) {
        finish(i, m0.w <= SELL_UNROLL ? R0.sum(g, m0) : sell_row<T, C, V>(i, col, val, g, U, m0));
        i += stride;
        if (i < n) {
            m0 = slice_meta(i, off, U);
            if (m0.w <= SELL_UNROLL) R0.load(i, col, val, g, U, m0);
        }
    }
    const double s = block_sum(d, sh);
    if (threadIdx.x == 0) part_pq[blk] = s;
}

// alpha = rz / pq; r -= alpha q; z = M r; partials r.z and r.r
template <typename T>
__global__ __launch_bounds__(SV_BLOCK) void k_cg_update(int64_t n, const T *__restrict__ dinv, T *__restrict__ r,
                                                        T *__restrict__ z, const T *__restrict__ q,
                                                        const double *__restrict__ part_pq, double *__restrict__ sc,
                                                        int par, double *__restrict__ part_rz,
                                                        double *__restrict__ part_rr)
{
    __shared__ double sh[SV_BLOCK / 64];
    const int G = gridDim.x;
    const int64_t stride = (int64_t)G * SV_BLOCK;
    int64_t i = (int64_t)blockIdx.x * SV_BLOCK + threadIdx.x;
    // the first rows' loads are in flight while alpha is formed
    T rr[UP_ROWS], qq[UP_ROWS], dd[UP_ROWS];
    auto load = [&]() {
#pragma unroll
        for (int u = 0; u < UP_ROWS; u++) {
            const int64_t j = i + u * stride < n ? i + u * stride : n - 1;
            rr[u] = r[j];
            qq[u] = q[j];
            dd[u] = dinv[j];
        }
    };
    load();
    const double rz = sc[S_RZS + par];
    const double pq = sum_partials(part_pq, G, sh);
    const double alpha64 = pq != 0.0 ? rz / pq : 0.0;
    const T alpha = (T)alpha64;
    if (blockIdx.x == 0 && threadIdx.x == 0) sc[S_ALPHA] = alpha64;
    double a = 0.0, b = 0.0;
    while (i < n) {
#pragma unroll
        for (int u = 0; u < UP_ROWS; u++) {
            if (i + u * stride >= n) break;
            const T ri = rr[u] - alpha * qq[u];
            const T zi = dd[u] * ri;
            r[i + u * stride] = ri;
            z[i + u * stride] = zi;
            a += (double)ri * (double)zi;
            b += (double)ri * (double)ri;
        }
        i += UP_ROWS * stride;
        if (i < n) load();
    }
    a = block_sum(a, sh);
    b = block_sum(b, sh);
    if (threadIdx.x == 0) { part_rz[blockIdx.x] = a; part_rr[blockIdx.x] = b; }
}

// x += alpha p, p = z + beta p; par: the iteration's parity whose update came
// last.  Workgroup 0 leaves the r.z that beta was formed with in rzs[par ^ 1].
// END, the end of a group of iterations: the accumulated steps xlo go into the
// FP64 iterate too (mixed), and workgroup 0 leaves rz and ||r||^2 for the host.
template <typename T, typename TX, bool END>
__global__ __launch_bounds__(SV_BLOCK) void k_cg_dir(int64_t n, const double *__restrict__ part_rz,
                                                     const double *__restrict__ part_rr, const T *__restrict__ z,
                                                     T *__restrict__ p, TX *__restrict__ xs, double *__restrict__ x,
                                                     double *__restrict__ sc, int par, double *__restrict__ hsc)
{
    __shared__ double sh[SV_BLOCK / 64];
    const int G = gridDim.x;
    const double rz = sum_partials(part_rz, G, sh);
    const double rz_old = sc[S_RZS + par];
    const T beta = (T)(rz_old != 0.0 ? rz / rz_old : 0.0);
    const TX alphax = (TX)sc[S_ALPHA];
    for (int64_t i = (int64_t)blockIdx.x * SV_BLOCK + threadIdx.x; i < n; i += (int64_t)G * SV_BLOCK) {
        const T pr = p[i];
        TX t = xs[i];
        t += alphax * (TX)pr;
        if constexpr (END && sizeof(TX) == 4) {
            x[i] += (double)t;
            xs[i] = TX(0);
        } else {
            xs[i] = t;
        }
        p[i] = z[i] + beta * pr;
    }
    if (!END && blockIdx.x == 0 && threadIdx.x == 0) sc[S_RZS + (par ^ 1)] = rz;
    if (END && blockIdx.x == 0) {
        const double rr = sum_partials(part_rr, G, sh);
        if (threadIdx.x == 0) { sc[S_RZ] = rz; sc[S_RR] = rr; hsc[S_RR] = rr; }
    }
}

// ---- small systems: the whole iteration in one launch ---------------------------
// Where every row has a work-item of its own and the rows are narrow, a group
// of iterations after the other runs in one cooperative launch: a row's entries,
// its residual, direction and iterate stay in registers, and only z and p (for
// the neighbours' gathers) and the dot products' partials go through memory.
// A workgroup is VB blocks of SV_BLOCK rows, each with the partials that the
// grid-wide kernels form for the same block, summed in the same order: the
// same bits.  Heat T3 100^2 FP64, an iteration: 15 us in two launches (each
// half launch and sums of partials) -> 5.8 us.
//
// An exchange of partials is also the barrier between an iteration's two halves:
// a workgroup publishes after its stores of z and p are complete, and who has
// seen all partials may read them.  A slot holds EX_NONE until it is published;
// three sets of slots take turns, and a slot is emptied once the next exchange
// is through (everybody has read it then, and nobody looks at it before the
// exchange after the next, which waits for this workgroup's next partial).
// The launch is cooperative, so that all workgroups run and every wait ends;
// a wait of EX_LIMIT polls, near a second (another process's launch holds some
// of the CUs, and waits too), ends the launch: what it has made of x is the
// start of the iteration of several launches, as any x is.
// VB: the registers of a row (its entries, the gathers in flight) leave 512
// work-items of FP64 rows or 768 of FP32 rows; larger workgroups spill (1024
// FP64: 14.9 us an iteration at 9801 rows), smaller ones are more pollers of the
// same slots (256: 10.5 and 10.8 against 9.4 and 9.0 us at 62 000 rows, the
// slots packed).
// SM_GRID: as many workgroups as measured faster than two launches (iteration
// at 100^2, 250^2, 300^2 rows FP64 5.8, 6.3, 6.5 against 15.3, 15.2, 16.8 us;
// mixed 100^2, 250^2, 400^2 6.2, 6.0, 7.2 against 15.5, 14.8, 17.0), with an
// eighth of the CUs left free.
#define SM_VB8 2
#define SM_VB4 3
#define SM_GRID 224
#define EX_NONE 0xfff8dead5eedbeefull
#define EX_LIMIT (1 << 20)

// z and p are written and gathered, and the slots filled and polled, with
// relaxed agent-scope accesses: they bypass the XCDs' L2 (the compiler's
// agent-scope fences, which write back and empty the whole L2, cost 2 us an
// iteration at 62 000 rows and 3 at 86 000).  Order comes from waiting for the
// wave's stores before the barrier that the partial is published behind, and
// from gathering only behind the barrier that follows the last poll.
template <typename T>
__device__ __forceinline__ T dev_load(const T *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <typename T>
__device__ __forceinline__ void dev_store(T *p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
#define STORES_OUT() asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory")

// The value that lane l + D holds, for the lanes l that a tree of __shfl_down over
// D = 32, 16, ... 1 needs (0 .. D - 1, and those that these need): register
// moves of a few cycles in place of a round through LDS.
template <int D>
__device__ __forceinline__ uint32_t lane_down(uint32_t x)
{
    if constexpr (D == 32) return __builtin_amdgcn_permlane32_swap(x, x, false, false)[1];
    else if constexpr (D == 16) return __builtin_amdgcn_permlane16_swap(x, x, false, false)[1];
    else return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x100 | D, 0xf, 0xf, true);  // row_shl
}
template <int D>
__device__ __forceinline__ double lane_down(double v)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    return __builtin_bit_cast(double, (uint64_t)lane_down<D>((uint32_t)(b >> 32)) << 32 | lane_down<D>((uint32_t)b));
}
// lane 0: the wave's sum in the order of the shuffle tree
__device__ __forceinline__ double wave_sum(double v)
{
    v += lane_down<32>(v);
    v += lane_down<16>(v);
    v += lane_down<8>(v);
    v += lane_down<4>(v);
    v += lane_down<2>(v);
    v += lane_down<1>(v);
    return v;
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#define SC1 16  // cache policy of buffer accesses: device scope
#define NT 2    // ... read once

// Three sets of slots; a block's two partials lie side by side, four blocks to
// 64 bytes, in EX_COPIES copies: every workgroup polls all slots, of the copy
// of its number's remainder.  One copy in a few kilobytes is in the same few
// channels for all of them (us an iteration, packed slots, 1, 4 and 8 copies:
// FP64 300x290 8.6, 6.9, 6.6, 6.5; mixed 1000^2 15.4, 12.5, 12.4, 11.9).
#define EX_COPIES 8
#define EX_LINE (64 * EX_COPIES)
#define EX_STRIDE(g) (((g) + 3) / 4 * EX_LINE)  // bytes of a set of g blocks
struct Exchange {
    uint64_t *slots;
    int G;
    int limit;  // polls of a wait
    __host__ __device__ __forceinline__ int stride() const { return EX_STRIDE(G); }  // bytes of a set
    __device__ __forceinline__ uint32_t at(uint32_t e, int blk, int copy) const
    {
        return (e % 3) * (uint32_t)stride() + (uint32_t)(blk >> 2) * EX_LINE + (uint32_t)copy * 64 + (uint32_t)(blk & 3) * 16;
    }
    __device__ __forceinline__ void put(uint32_t e, int blk, int copy, int two, uint64_t v) const
    {
        dev_store((uint64_t *)((char *)slots + at(e, blk, copy) + 8 * two), v);
    }
    template <bool TWO>
    __device__ __forceinline__ void get(uint32_t e, int blk, uint64_t &u, uint64_t &v) const
    {
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(slots, 0, 3 * stride(), 0x00020000);
        int o = (int)at(e, blk, blockIdx.x % EX_COPIES);
        asm volatile("" : "+v"(o)::"memory");  // a load each time
        if (TWO) {
            const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(r, o, 0, SC1);
            u = ((uint64_t)x[1] << 32) | x[0];
            v = ((uint64_t)x[3] << 32) | x[2];
        } else {
            const u32x2 x = __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, SC1);
            u = ((uint64_t)x[1] << 32) | x[0];
        }
    }
};

__device__ __forceinline__ uint64_t ex_bits(double v)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    return b == EX_NONE ? 0x7ff8000000000000ull : b;
}

// Publishes the sums of a (and, TWO, of b) over each block's work-items, waits
// for everybody's and returns their sums, formed as block_sum and sum_partials
// form them.  e: the exchange's number.  False: the wait went on for too long.
// The first four waves poll for all; a wait by every wave took three times as
// long at 243 blocks.
template <int VB, bool TWO>
__device__ __forceinline__ bool exchange(const Exchange &X, uint32_t e, double &a, double &b, double (*sh)[VB * SV_BLOCK / 64],
                                         double (*sum)[SV_BLOCK / 64], uint32_t *quit)
{
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    STORES_OUT();
    a = wave_sum(a);
    if (TWO) b = wave_sum(b);
    if (lane == 0) {
        sh[0][w] = a;
        if (TWO) sh[1][w] = b;
    }
    __syncthreads();
    // lanes of the first wave: block, partial, copy
    const int q = lane / (2 * EX_COPIES), two = lane / EX_COPIES % 2, copy = lane % EX_COPIES, blk = blockIdx.x * VB + q;
    const bool mine = w == 0 && q < VB && blk < X.G;
    if (mine && (TWO || two == 0)) {
        double s = 0.0;
        for (int k = 0; k < SV_BLOCK / 64; k++) s += sh[two][q * (SV_BLOCK / 64) + k];
        X.put(e, blk, copy, two, ex_bits(s));
    }
    if (tid < SV_BLOCK) {
        a = 0.0;
        b = 0.0;
        for (int i = tid; i < X.G; i += 4 * SV_BLOCK) {
            uint64_t u[4], v[4];
            int spin = X.limit;
            bool wait;
            do {
                wait = false;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    u[q] = v[q] = 0;
                    if (i + q * SV_BLOCK < X.G) X.get<TWO>(e, i + q * SV_BLOCK, u[q], v[q]);
                }
#pragma unroll
                for (int q = 0; q < 4; q++) wait |= u[q] == EX_NONE || v[q] == EX_NONE;
            } while (wait && --spin > 0);
            if (wait) *quit = 1u;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                if (i + q * SV_BLOCK >= X.G) break;
                a += __builtin_bit_cast(double, u[q]);
                if (TWO) b += __builtin_bit_cast(double, v[q]);
            }
        }
        a = wave_sum(a);
        if (TWO) b = wave_sum(b);
        if (lane == 0) {
            sum[0][w] = a;
            if (TWO) sum[1][w] = b;
        }
    }
    __syncthreads();
    a = 0.0;
    b = 0.0;
    for (int k = 0; k < SV_BLOCK / 64; k++) {
        a += sum[0][k];
        if (TWO) b += sum[1][k];
    }
    if (mine) X.put(e + 2, blk, copy, two, EX_NONE);
    return *quit == 0u;  // set before the barrier by whoever gave up
}

__global__ void k_cg_slots(uint64_t *__restrict__ slots, int n, double *__restrict__ sc)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) sc[S_LOST] = 0.0;
    if (i < n) slots[i] = EX_NONE;
}

// Groups of CHECK iterations from the state that k_cg_reset or this kernel left
// (r, z, p, r.z partials) until ||r||^2 <= goal2 or maxit; leaves the same state
// as k_cg_dir, the iteration count in sc[S_IT] and ||r||^2 in sc[S_RREC]; sc[S_LOST] is set by
// every workgroup that gave up a wait (another may have been through it).
template <typename T, typename TX, typename C, int VB>
__global__ __launch_bounds__(VB * SV_BLOCK) void k_cg_small(int64_t n, const uint32_t *__restrict__ off,
                                                       const C *__restrict__ col, const T *__restrict__ val,
                                                       const T *__restrict__ dinv, T *r_, T *z_, T *pa, T *pb, TX *xs_,
                                                       double *x_, const double *part_rz, Exchange X, double *sc,
                                                       double goal2, int it, int maxit)
{
    __shared__ double sh[2][VB * SV_BLOCK / 64], sum[2][SV_BLOCK / 64];
    __shared__ uint32_t quit;
    if (threadIdx.x == 0) quit = 0;
    const int64_t i = (int64_t)blockIdx.x * (VB * SV_BLOCK) + threadIdx.x;
    const bool live = i < n;
    const int64_t ic = live ? i : n - 1;
    const uint32_t s = (uint32_t)__builtin_amdgcn_readfirstlane((int)(ic >> 6));
    const uint32_t o = off[s], w = (off[s + 1] - o) >> 6;
    T v[SELL_UNROLL];
    int32_t cj[SELL_UNROLL];
#pragma unroll
    for (int k = 0; k < SELL_UNROLL; k++) {
        const int64_t at = sell_slot(o, w, k, (int)(ic & 63));
        v[k] = T(0);
        cj[k] = (int32_t)ic;
        if (at >= 0) {
            v[k] = val[at];
            cj[k] = sell_col<C>(col[at], ic);
        }
    }
    const T di = dinv[ic];
    T ri = r_[ic], zi = z_[ic], pi = pa[ic];
    TX xs = xs_[ic];
    double xd = sizeof(TX) == 4 ? x_[ic] : 0.0;
    // r.z of the state, summed as sum_partials does
    double rz = 0.0, rz_old = 0.0, rr = 0.0, none = 0.0;
    if (threadIdx.x < SV_BLOCK) {
        for (int k = threadIdx.x; k < X.G; k += SV_BLOCK) rz += part_rz[k];
        for (int d = 32; d > 0; d >>= 1) rz += __shfl_down(rz, d, 64);
        if ((threadIdx.x & 63) == 0) sum[0][threadIdx.x >> 6] = rz;
    }
    __syncthreads();
    rz = 0.0;
    for (int k = 0; k < SV_BLOCK / 64; k++) rz += sum[0][k];
    T *p_old = pa, *p_new = pb;
    uint32_t e = 0;
    bool dir = false, ok = true;
    rr = sc[S_RR];  // the state's
    while (ok && rr > goal2 && it < maxit) {
        for (int k = 0; k < CHECK && ok; k++) {
            T y[SELL_UNROLL];
            if (dir) {
                const T beta = (T)(rz_old != 0.0 ? rz / rz_old : 0.0);
#pragma unroll
                for (int q = 0; q < SELL_UNROLL; q++) y[q] = dev_load(z_ + cj[q]) + beta * dev_load(p_old + cj[q]);
                pi = zi + beta * pi;
                if (live) dev_store(p_new + i, pi);
                T *t = p_old;
                p_old = p_new;
                p_new = t;
            } else {
#pragma unroll
                for (int q = 0; q < SELL_UNROLL; q++) y[q] = dev_load(p_old + cj[q]);
                dir = true;
            }
            T qi = T(0);
#pragma unroll
            for (int q = 0; q < SELL_UNROLL; q++)
                if (q < (int)w) qi += v[q] * y[q];
            double pq = 0.0;
            if (live) pq += (double)pi * (double)qi;
            if (!(ok = exchange<VB, false>(X, e++, pq, none, sh, sum, &quit))) break;
            const double alpha64 = pq != 0.0 ? rz / pq : 0.0;
            const T alpha = (T)alpha64;
            double a = 0.0, b = 0.0;
            if (live) {
                ri = ri - alpha * qi;
                zi = di * ri;
                dev_store(z_ + i, zi);
                a += (double)ri * (double)zi;
                b += (double)ri * (double)ri;
                xs += (TX)alpha64 * (TX)pi;
            }
            if (!(ok = exchange<VB, true>(X, e++, a, b, sh, sum, &quit))) break;
            rz_old = rz;
            rz = a;
            rr = b;
        }
        if constexpr (sizeof(TX) == 4) {
            xd += (double)xs;
            xs = TX(0);
        }
        it += CHECK;
    }
    // the state that the next reset continues from
    const T beta = (T)(rz_old != 0.0 ? rz / rz_old : 0.0);
    if (live && dir) {
        r_[i] = ri;
        p_old[i] = zi + beta * pi;
        if (p_old != pa) pa[i] = zi + beta * pi;
        xs_[i] = xs;
        if constexpr (sizeof(TX) == 4) x_[i] = xd;
    }
    // (every workgroup reads S_RR at its start: the result has its own word)
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc[S_RREC] = rr;
        sc[S_IT] = (double)it;
    }
    if (!ok && threadIdx.x == 0) sc[S_LOST] = 1.0;
}

// ---- systems that the register file holds -----------------------------------------
// The same one launch for larger systems on grid-like meshes (k_sell_rec): a
// workgroup a CU, R rows a work-item, with their entries in registers (R x 9 of
// them) and r, 1/diagonal, p and the iterate in LDS.  An iteration then reads
// and writes z and p alone where the streaming kernels move 80 bytes a row.
// Streaming -> resident, us an iteration: FP64 Q4 460x450 22.9 -> 8.7, T3
// 700x690 29.4 -> 10.9; mixed Q4 500^2 19.1 -> 7.6, 1000^2 30.5 -> 10.7,
// 1500x1300 (1.95 million rows) 44.3 -> 18.9.
// The rows, blocks and sums are those of the streaming kernels (block b's rows
// are b * 256 + t + k * 256 G): the same bits.
//
// What bounds it: up to 1 million rows the two exchanges, 3 us each (a store
// until it can be read, then a load of it, both past the L2s); beyond, z and p
// through the Infinity Cache.  A row's nine neighbours lie three by three.  The
// three on its own grid row come from p in LDS, with the two rows beside the
// block read extra.  Of the runs above and below every lane reads one word of z
// and of p, four lanes the two that follow the wave's 64, and the others come
// from the next lanes: 13 % faster at 1 million rows than six loads of three
// words (16 cycles each in the address unit, and a word fetched three times),
// two full loads a run 5 % slower than one (twice the lines).  Loads are
// device-scope, with bounds of their own: a word outside the vector reads zero,
// and the entry for it is zero.
#define RES_VB 4
#define RES_BLOCK (RES_VB * SV_BLOCK)
#define RES_GRID SV_BLOCK  // workgroups at most: block b's is b % RES_GRID
// a * b rounded, whatever it is added to
template <typename T>
__device__ __forceinline__ T product(T a, T b)
{
#pragma clang fp contract(off)
    return a * b;
}

// A vector's n words, device-coherent: a word outside reads zero, a store there
// is dropped (a negative number is one far past the end).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t words_rsrc(void *v, size_t word, int64_t n)
{
    return __builtin_amdgcn_make_buffer_rsrc(v, 0, (int)(n * word), 0x00020000);
}
template <int POLICY>
__device__ __forceinline__ void load1(__amdgpu_buffer_rsrc_t r, int32_t i, float &o)
{
    o = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, i * 4, 0, POLICY));
}
template <int POLICY>
__device__ __forceinline__ void load1(__amdgpu_buffer_rsrc_t r, int32_t i, double &o)
{
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, i * 8, 0, POLICY);
    o = __builtin_bit_cast(double, ((uint64_t)v[1] << 32) | v[0]);
}
__device__ __forceinline__ void store1(__amdgpu_buffer_rsrc_t r, int32_t i, float v)
{
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, i * 4, 0, SC1);
}
__device__ __forceinline__ void store1(__amdgpu_buffer_rsrc_t r, int32_t i, double v)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    __builtin_amdgcn_raw_buffer_store_b64(u32x2{(uint32_t)b, (uint32_t)(b >> 32)}, r, i * 8, 0, SC1);
}
// Lane l: the next lane's x; lane 63: last.
__device__ __forceinline__ float next_lane(float x, float last)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, last), __builtin_bit_cast(int, x), 0x130,
                                                                 0xf, 0xf, false));  // wave_shl:1
}
__device__ __forceinline__ double next_lane(double x, double last)
{
    const uint64_t a = __builtin_bit_cast(uint64_t, x), b = __builtin_bit_cast(uint64_t, last);
    const uint32_t l = (uint32_t)__builtin_amdgcn_update_dpp((int)b, (int)a, 0x130, 0xf, 0xf, false);
    const uint32_t h = (uint32_t)__builtin_amdgcn_update_dpp((int)(b >> 32), (int)(a >> 32), 0x130, 0xf, 0xf, false);
    return __builtin_bit_cast(double, (uint64_t)h << 32 | l);
}
__device__ __forceinline__ float of_lane(float x, int l)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), l));
}
__device__ __forceinline__ double of_lane(double x, int l)
{
    const uint64_t a = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)a, l), hi = (uint32_t)__builtin_amdgcn_readlane((int)(a >> 32), l);
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// exchange() for workgroups that hold the blocks w, w + RES_GRID, ...: these are
// the ones that one work-item of the sum over all blocks adds up, so the
// workgroup publishes what that work-item would have: a quarter of the slots.
template <bool TWO>
__device__ __forceinline__ bool exchange_res(const Exchange &X, uint32_t e, double &a, double &b,
                                             double (*sh)[RES_BLOCK / 64], double (*sum)[SV_BLOCK / 64], uint32_t *quit)
{
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, nw = gridDim.x;
    STORES_OUT();
    a = wave_sum(a);
    if (TWO) b = wave_sum(b);
    if (lane == 0) {
        sh[0][w] = a;
        if (TWO) sh[1][w] = b;
    }
    __syncthreads();
    const int two = lane / EX_COPIES, copy = lane % EX_COPIES;  // lanes of the first wave: partial, copy
    const bool mine = w == 0 && two < 2;
    if (mine && (TWO || two == 0)) {
        double t = 0.0;
        for (int q = 0; q < RES_VB && (int)blockIdx.x + q * RES_GRID < X.G; q++) {
            double s = 0.0;
            for (int k = 0; k < SV_BLOCK / 64; k++) s += sh[two][q * (SV_BLOCK / 64) + k];
            t += s;
        }
        X.put(e, blockIdx.x, copy, two, ex_bits(t));
    }
    if (tid < SV_BLOCK) {
        uint64_t u = 0, v = 0;
        if (tid < nw) {
            int spin = X.limit;
            do {
                X.get<TWO>(e, tid, u, v);
            } while ((u == EX_NONE || v == EX_NONE) && --spin > 0);
            if (u == EX_NONE || v == EX_NONE) *quit = 1u;
        }
        a = wave_sum(__builtin_bit_cast(double, u));
        if (TWO) b = wave_sum(__builtin_bit_cast(double, v));
        if (lane == 0) {
            sum[0][w] = a;
            if (TWO) sum[1][w] = b;
        }
    }
    __syncthreads();
    a = 0.0;
    b = 0.0;
    for (int k = 0; k < SV_BLOCK / 64; k++) {
        a += sum[0][k];
        if (TWO) b += sum[1][k];
    }
    if (mine) X.put(e + 2, blockIdx.x, copy, two, EX_NONE);
    return *quit == 0u;
}

// A row's nine entries out of its slice (v: zeros before).
template <typename T>
__device__ __forceinline__ void nine_entries(const uint32_t *__restrict__ off, const int16_t *__restrict__ col,
                                             const T *__restrict__ val, int32_t s, int lane, int32_t lo, int32_t hi, T *v)
{
    const uint32_t o = off[s], w = (off[s + 1] - o) >> 6;
    for (uint32_t q = 0; q < w; q++) {
        const size_t at = (size_t)o + (size_t)q * 64 + lane;
        const T x = val[at];  // zero in the padding of a short row, whose column is its own
        const int32_t d = col[at];
        if (x != T(0) || d != 0) nine_put(x, d, lo, hi, v);
    }
}

template <typename T, typename TX, int R>
__global__ __launch_bounds__(RES_BLOCK) void k_cg_resident(int64_t n, const uint32_t *__restrict__ off,
                                                           const int16_t *__restrict__ col, const T *__restrict__ val,
                                                           const int2 *__restrict__ rec, const T *__restrict__ dinv, T *r_,
                                                           T *z_, T *pa, T *pb, TX *xs_, double *x_, const double *part_rz,
                                                           Exchange X, double *sc, double goal2, int it, int maxit)
{
    // (z and p of more than a million rows are gone from an L2 before the next
    // row of the grid reads them: 3 to 7 % faster past them; fewer rows 2 % slower)
    constexpr int POLICY = R >= 6 ? SC1 | NT : SC1;
    constexpr int DEEP = R < 3 ? R : 3;  // rows in flight (1, 2, 3, 4, 6: 22.0, 20.5, 19.5, 19.8, 23.5 us at 1.95 million rows)
    __shared__ T sr[R][RES_BLOCK], sd[R][RES_BLOCK];
    __shared__ T sp[R][RES_VB][SV_BLOCK + 2];  // p, each block's between the two rows beside it
    __shared__ TX sx[R][RES_BLOCK];
    __shared__ double sh[2][RES_BLOCK / 64], sum[2][SV_BLOCK / 64];
    __shared__ uint32_t quit;
    const int tid = threadIdx.x, lane = tid & 63;
    if (tid == 0) quit = 0;
    const int bq = tid / SV_BLOCK, bt = tid % SV_BLOCK, blk = blockIdx.x + bq * RES_GRID;
    const int32_t stride = X.G * SV_BLOCK, nn = (int32_t)n;
    const int32_t i0 = blk < X.G ? blk * SV_BLOCK + bt : ((nn + 63) & ~63) + bt;  // no such block: rows past the last
    const int32_t s0 = __builtin_amdgcn_readfirstlane(i0 >> 6), sstride = stride >> 6;
    const int32_t slast = (nn - 1) >> 6;
    // row k's number, formed anew (kept for all rows, with what follows from it,
    // it would take the registers that hold the matrix)
    auto row = [&](int k) -> int32_t {
        int32_t i = i0 + k * stride;
        asm volatile("" : "+v"(i));
        return i;
    };
    T v[R][RES_W], qv[R];
    int32_t lo[R], hi[R];  // of the wave's slices
#pragma unroll
    for (int k = 0; k < R; k++) {
        const int32_t i = row(k), ic = min(i, nn - 1), s = s0 + k * sstride;
        qv[k] = T(0);
        lo[k] = hi[k] = 0;
#pragma unroll
        for (int q = 0; q < RES_W; q++) v[k][q] = T(0);
        if (s <= slast) {
            lo[k] = __builtin_amdgcn_readfirstlane(rec[s].x);
            hi[k] = __builtin_amdgcn_readfirstlane(rec[s].y);
            nine_entries(off, col, val, s, lane, lo[k], hi[k], v[k]);
        }
        // zeros past the last row, and so all that follows from them
        sr[k][tid] = i < nn ? r_[ic] : T(0);
        sd[k][tid] = i < nn ? dinv[ic] : T(0);
        sp[k][bq][bt + 1] = i < nn ? pa[ic] : T(0);
        sx[k][tid] = i < nn ? xs_[ic] : TX(0);
        if (i >= nn) {
#pragma unroll
            for (int q = 0; q < RES_W; q++) v[k][q] = T(0);
        }
    }
    double rz = 0.0, rz_old = 0.0, rr = 0.0, none = 0.0;
    if (tid < SV_BLOCK) {
        for (int k = tid; k < X.G; k += SV_BLOCK) rz += part_rz[k];
        for (int d = 32; d > 0; d >>= 1) rz += __shfl_down(rz, d, 64);
        if (lane == 0) sum[0][tid >> 6] = rz;
    }
    __syncthreads();
    rz = 0.0;
    for (int k = 0; k < SV_BLOCK / 64; k++) rz += sum[0][k];
    const __amdgpu_buffer_rsrc_t bz = words_rsrc(z_, sizeof(T), n);
    T *p_old = pa, *p_new = pb;
    uint32_t e = 0;
    bool dir = false, ok = true;
    rr = sc[S_RR];
    const int32_t past = lane < 4 ? 64 - (lane & 2) : 1 << 28;  // lanes 4 ..: outside the vector, nothing is fetched
    while (ok && rr > goal2 && it < maxit) {
        for (int c = 0; c < CHECK && ok; c++) {
            const T beta = dir ? (T)(rz_old != 0.0 ? rz / rz_old : 0.0) : T(0);
            const __amdgpu_buffer_rsrc_t bp = words_rsrc(p_old, sizeof(T), n), bn = words_rsrc(p_new, sizeof(T), n);
            // DEEP rows in flight: their lower and upper run's first words, and
            // (lanes 0, 1 the lower's, 2, 3 the upper's) the two past the wave's
            T zz[DEEP][3], pp[DEEP][3];
            auto load = [&](int k) {
                const int32_t i = row(k);
                int32_t l = lo[k], h = hi[k];
                asm volatile("" : "+s"(l), "+s"(h));
                load1<POLICY>(bp, i + l, pp[k % DEEP][0]);
                load1<POLICY>(bz, i + l, zz[k % DEEP][0]);
                load1<POLICY>(bp, i + h, pp[k % DEEP][1]);
                load1<POLICY>(bz, i + h, zz[k % DEEP][1]);
                const int32_t j = i + past + (lane < 2 ? l : h);
                load1<POLICY>(bp, j, pp[k % DEEP][2]);
                load1<POLICY>(bz, j, zz[k % DEEP][2]);
            };
            if (tid < 2 * RES_VB * R) {  // the rows beside the blocks
                const int k = tid / (2 * RES_VB), q = (tid >> 1) % RES_VB, right = tid & 1;
                const int32_t i = (int32_t)(blockIdx.x + q * RES_GRID) * SV_BLOCK + k * stride + (right ? SV_BLOCK : -1);
                T z1, p1;
                load1<POLICY>(bp, i, p1);
                load1<POLICY>(bz, i, z1);
                sp[k][q][right ? SV_BLOCK + 1 : 0] = dir ? z1 + beta * p1 : p1;
            }
#pragma unroll
            for (int k = 0; k < DEEP; k++) load(k);
            __builtin_amdgcn_sched_barrier(0);
            if (dir) {
#pragma unroll
                for (int k0 = 0; k0 < R; k0 += 4) {
                    T pk[4];
#pragma unroll
                    for (int k = k0; k < k0 + 4 && k < R; k++)
                        pk[k - k0] = product(sd[k][tid], sr[k][tid]) + beta * sp[k][bq][bt + 1];
#pragma unroll
                    for (int k = k0; k < k0 + 4 && k < R; k++) {
                        sp[k][bq][bt + 1] = pk[k - k0];
                        store1(bn, row(k), pk[k - k0]);
                    }
                }
            }
            __syncthreads();
            double pq = 0.0;
#pragma unroll
            for (int k = 0; k < R; k++) {
                T y[RES_W];
#pragma unroll
                for (int g = 0; g < 3; g++) {
                    const T zg = zz[k % DEEP][g], pg = pp[k % DEEP][g], yg = dir ? zg + beta * pg : pg;
                    if (g < 2) y[6 * g] = yg;
                    else y[4] = yg;
                }
                y[1] = next_lane(y[0], of_lane(y[4], 0));
                y[2] = next_lane(y[1], of_lane(y[4], 1));
                y[7] = next_lane(y[6], of_lane(y[4], 2));
                y[8] = next_lane(y[7], of_lane(y[4], 3));
#pragma unroll
                for (int j = 0; j < 3; j++) y[3 + j] = sp[k][bq][bt + j];
                __builtin_amdgcn_sched_barrier(0);
                if (k + DEEP < R) load(k + DEEP);
                __builtin_amdgcn_sched_barrier(0);
                T acc = T(0);
#pragma unroll
                for (int j = 0; j < RES_W; j++) acc += v[k][j] * y[j];
                qv[k] = acc;
                pq += (double)y[4] * (double)acc;
                __builtin_amdgcn_sched_barrier(0);
            }
            if (dir) {
                T *t = p_old;
                p_old = p_new;
                p_new = t;
            }
            dir = true;
            if (!(ok = exchange_res<false>(X, e++, pq, none, sh, sum, &quit))) break;
            const double alpha64 = pq != 0.0 ? rz / pq : 0.0;
            const T alpha = (T)alpha64;
            const TX alphax = (TX)alpha64;
            double a = 0.0, b = 0.0;
#pragma unroll
            for (int k0 = 0; k0 < R; k0 += 4) {
                T ri[4], zi[4];
                TX xi[4];
#pragma unroll
                for (int k = k0; k < k0 + 4 && k < R; k++) {
                    ri[k - k0] = sr[k][tid] - alpha * qv[k];
                    zi[k - k0] = sd[k][tid] * ri[k - k0];
                    xi[k - k0] = sx[k][tid] + alphax * (TX)sp[k][bq][bt + 1];
                }
#pragma unroll
                for (int k = k0; k < k0 + 4 && k < R; k++) {
                    store1(bz, row(k), zi[k - k0]);
                    sr[k][tid] = ri[k - k0];
                    sx[k][tid] = xi[k - k0];
                    a += (double)ri[k - k0] * (double)zi[k - k0];
                    b += (double)ri[k - k0] * (double)ri[k - k0];
                }
            }
            if (!(ok = exchange_res<true>(X, e++, a, b, sh, sum, &quit))) break;
            rz_old = rz;
            rz = a;
            rr = b;
        }
        if constexpr (sizeof(TX) == 4) {
#pragma unroll
            for (int k = 0; k < R; k++) {
                const int32_t i = row(k);
                if (i >= nn) break;
                x_[i] += (double)sx[k][tid];
                sx[k][tid] = TX(0);
            }
        }
        it += CHECK;
    }
    // the state that the next reset continues from
    if (dir) {
        const T beta = (T)(rz_old != 0.0 ? rz / rz_old : 0.0);
#pragma unroll
        for (int k = 0; k < R; k++) {
            const int32_t i = row(k);
            if (i >= nn) break;
            r_[i] = sr[k][tid];
            pa[i] = product(sd[k][tid], sr[k][tid]) + beta * sp[k][bq][bt + 1];
            xs_[i] = sx[k][tid];
        }
    }
    if (blockIdx.x == 0 && tid == 0) {
        sc[S_RREC] = rr;
        sc[S_IT] = (double)it;
    }
    if (!ok && threadIdx.x == 0) sc[S_LOST] = 1.0;
}

// The same for at most 2048 FP64 or 4096 FP32 rows, by one workgroup: p in LDS,
// R rows a work-item (row tid + 1024 k: block 4 k + tid / 256), the sums over
// waves in LDS and over the blocks by every wave for itself.  Three barriers are
// left of the waits for other workgroups, which are most of an iteration of the
// small systems above.  Whole solves, one launch of many workgroups -> of one:
// FP64 T3 33x32 775 -> 421 us, T3 46x45 (1980 rows) 977 -> 642; mixed Q4 30^2
// 959 -> 539, Q4 64^2 (3969) 1602 -> 1441.  Four FP64 rows a work-item spill
// (Q4 64x63 1399 -> 1825).
#define ONE_ROWS(T) (sizeof(T) == 8 ? 2 * RES_BLOCK : 4 * RES_BLOCK)
template <typename T, typename TX, int R>
__global__ __launch_bounds__(RES_BLOCK) void k_cg_one(int n, int G, const uint32_t *__restrict__ off,
                                                      const int16_t *__restrict__ col, const T *__restrict__ val,
                                                      const int2 *__restrict__ rec, const T *__restrict__ dinv, T *r_, T *pa,
                                                      TX *xs_, double *x_, const double *part_rz, double *sc, double goal2,
                                                      int it, int maxit)
{
    constexpr int N = R * RES_BLOCK, EDGE = 3;
    __shared__ T sp[N + 2 * EDGE];  // p between zeros
    __shared__ double sh[3][R * (RES_BLOCK / 64)];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    T v[R][RES_W], ri[R], di[R], pi[R], qi[R];
    TX xi[R];
    int lo[R], hi[R];  // where the row's runs begin in sp
    if (tid < EDGE) sp[tid] = sp[N + EDGE + tid] = T(0);
#pragma unroll
    for (int k = 0; k < R; k++) {
        const int i = k * RES_BLOCK + tid, s = i >> 6;
#pragma unroll
        for (int q = 0; q < RES_W; q++) v[k][q] = T(0);
        lo[k] = hi[k] = 0;
        if (i < n) {
            const int2 m = rec[s];
            nine_entries(off, col, val, s, lane, m.x, m.y, v[k]);
            lo[k] = EDGE + min(max(i + m.x, -EDGE), N);  // beyond: entries of nothing but zeros
            hi[k] = EDGE + min(max(i + m.y, -EDGE), N);
        }
        ri[k] = i < n ? r_[i] : T(0);
        di[k] = i < n ? dinv[i] : T(0);
        pi[k] = i < n ? pa[i] : T(0);
        xi[k] = i < n ? xs_[i] : TX(0);
    }
    // sums over all blocks, the same in every lane; lane l adds up block l's waves
    auto total = [&](const double *part) {
        double s = 0.0;
        if (lane < 4 * R)
            for (int k = 0; k < SV_BLOCK / 64; k++) s += part[lane * (SV_BLOCK / 64) + k];
        return 0.0 + of_lane(wave_sum(0.0 + s), 0);
    };
    double rz = 0.0 + of_lane(wave_sum(lane < G ? 0.0 + part_rz[lane] : 0.0), 0), rz_old = 0.0, rr = sc[S_RR];
    bool dir = false;
    while (rr > goal2 && it < maxit) {
        for (int c = 0; c < CHECK; c++) {
            const T beta = dir ? (T)(rz_old != 0.0 ? rz / rz_old : 0.0) : T(0);
#pragma unroll
            for (int k = 0; k < R; k++) {
                if (dir) pi[k] = product(di[k], ri[k]) + beta * pi[k];
                sp[EDGE + k * RES_BLOCK + tid] = pi[k];
            }
            dir = true;
            __syncthreads();
            double pq[R];
#pragma unroll
            for (int k = 0; k < R; k++) {
                T acc = T(0);
#pragma unroll
                for (int j = 0; j < RES_W; j++)
                    acc += v[k][j] * sp[j < 3 ? lo[k] + j : j < 6 ? EDGE - 4 + k * RES_BLOCK + tid + j : hi[k] + j - 6];
                qi[k] = acc;
                pq[k] = 0.0;
                pq[k] += (double)pi[k] * (double)acc;
                pq[k] = wave_sum(pq[k]);
            }
            if (lane == 0) {
#pragma unroll
                for (int k = 0; k < R; k++) sh[0][k * (RES_BLOCK / 64) + w] = pq[k];
            }
            __syncthreads();
            const double pqs = total(sh[0]);
            const double alpha64 = pqs != 0.0 ? rz / pqs : 0.0;
            const T alpha = (T)alpha64;
            const TX alphax = (TX)alpha64;
            double a[R], b[R];
#pragma unroll
            for (int k = 0; k < R; k++) {
                ri[k] = ri[k] - alpha * qi[k];
                const T zi = product(di[k], ri[k]);
                a[k] = b[k] = 0.0;
                a[k] += (double)ri[k] * (double)zi;
                b[k] += (double)ri[k] * (double)ri[k];
                a[k] = wave_sum(a[k]);
                b[k] = wave_sum(b[k]);
                xi[k] += alphax * (TX)pi[k];
            }
            if (lane == 0) {
#pragma unroll
                for (int k = 0; k < R; k++) {
                    sh[1][k * (RES_BLOCK / 64) + w] = a[k];
                    sh[2][k * (RES_BLOCK / 64) + w] = b[k];
                }
            }
            __syncthreads();
            rz_old = rz;
            rz = total(sh[1]);
            rr = total(sh[2]);
        }
        if constexpr (sizeof(TX) == 4) {
#pragma unroll
            for (int k = 0; k < R; k++) {
                const int i = k * RES_BLOCK + tid;
                if (i < n) x_[i] += (double)xi[k];
                xi[k] = TX(0);
            }
        }
        it += CHECK;
    }
    // the state that the next reset continues from
    if (dir) {
        const T beta = (T)(rz_old != 0.0 ? rz / rz_old : 0.0);
#pragma unroll
        for (int k = 0; k < R; k++) {
            const int i = k * RES_BLOCK + tid;
            if (i >= n) break;
            r_[i] = ri[k];
            pa[i] = product(di[k], ri[k]) + beta * pi[k];
            xs_[i] = xi[k];
        }
    }
    if (tid == 0) {
        sc[S_RREC] = rr;
        sc[S_IT] = (double)it;
        sc[S_LOST] = 0.0;
    }
}

// r = (T) r64, z = M r (p = z when `restart`); partials r.z (into rz_out) and r.r
template <typename T>
__global__ __launch_bounds__(SV_BLOCK) void k_cg_reset(int64_t n, const double *__restrict__ r64,
                                                       const T *__restrict__ dinv, T *__restrict__ r,
                                                       T *__restrict__ z, T *__restrict__ p, int restart,
                                                       double *__restrict__ rz_out, double *__restrict__ part_rr)
{
    __shared__ double sh[SV_BLOCK / 64];
    double a = 0.0, b = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * SV_BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * SV_BLOCK) {
        const T ri = (T)r64[i];
        const T zi = dinv[i] * ri;
        r[i] = ri;
        z[i] = zi;
        if (restart) p[i] = zi;
        a += (double)ri * (double)zi;
        b += (double)ri * (double)ri;
    }
    a = block_sum(a, sh);
    b = block_sum(b, sh);
    if (threadIdx.x == 0) { rz_out[blockIdx.x] = a; part_rr[blockIdx.x] = b; }
}

// Words into pinned host memory (read after a wait, without a copy).
__global__ void k_tell(const uint32_t *__restrict__ u, uint32_t *__restrict__ hu)
{
    if (threadIdx.x < 4) hu[threadIdx.x] = u[threadIdx.x];
}

// One workgroup: sc[slot] = sum of g partials (and sc[slot2] of a second set).
__global__ void k_reduce(const double *__restrict__ p, int g, double *sc, int slot,
                         const double *__restrict__ p2, int slot2, double *__restrict__ hsc)
{
    __shared__ double sh[1024 / 64];
    const double a = sum_partials(p, g, sh);
    const double b = p2 ? sum_partials(p2, g, sh) : 0.0;
    if (threadIdx.x == 0) {
        sc[slot] = a;
        if (p2) sc[slot2] = b;
        if (hsc)  // all scalars to pinned host memory
            for (int k = 0; k < S_NS; k++) hsc[k] = k == slot ? a : p2 && k == slot2 ? b : sc[k];
    }
}


// r = b - A x over the free block (SELL, FP64); partial ||r||^2
template <typename C>
__global__ __launch_bounds__(SV_BLOCK) void k_sell_resid(int64_t n, const uint32_t *__restrict__ off,
                                                         const C *__restrict__ col,
                                                         const double *__restrict__ val, SellU U,
                                                         const double *__restrict__ x, const double *__restrict__ b,
                                                         double *__restrict__ r, double *__restrict__ part)
{
    __shared__ double sh[SV_BLOCK / 64];
    double rr = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * SV_BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * SV_BLOCK) {
        const double v = b[i] - sell_row<double, C>(i, col, val, VecGather<double>{x}, U, slice_meta(i, off, U));
        r[i] = v;
        rr += v * v;
    }
    const double s = block_sum(rr, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// b = F_f - K_fd x_d with the CSR matrix (data columns only); partial ||b||^2
__global__ __launch_bounds__(SV_BLOCK) void k_rhs(int64_t nfree, const int32_t *__restrict__ ptr,
                                                  const int32_t *__restrict__ ind, const double *__restrict__ val,
                                                  const double *__restrict__ xfull, const double *F, double *b,
                                                  double *__restrict__ part)
{
    __shared__ double sh[SV_BLOCK / 64];
    double bb = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * SV_BLOCK + threadIdx.x; i < nfree; i += (int64_t)gridDim.x * SV_BLOCK) {
        double acc = 0.0;
        for (int32_t j = ptr[i]; j < ptr[i + 1]; j++)
            if (ind[j] >= nfree) acc += val[j] * xfull[ind[j]];
        const double v = F[i] - acc;
        b[i] = v;
        bb += v * v;
    }
    const double s = block_sum(bb, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ void k_diag_inv(int64_t n, const int32_t *__restrict__ ptr, const int32_t *__restrict__ ind,
                           const double *__restrict__ val, double *__restrict__ d64, float *__restrict__ d32)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double d = 0.0;
    int32_t lo = ptr[i], hi = ptr[i + 1];
    while (lo < hi) {  // sorted indices: binary search for the diagonal
        const int32_t m = (lo + hi) >> 1;
        if (ind[m] < i) lo = m + 1;
        else hi = m;
    }
    if (lo < ptr[i + 1] && ind[lo] == i) d = val[lo];
    const double inv = d != 0.0 ? 1.0 / d : 1.0;
    d64[i] = inv;
    if (d32) d32[i] = (float)inv;
}

template <typename T>
__global__ void k_fill(int64_t n, T *__restrict__ a, T v)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = v;
}

template <typename T>
struct Vecs {
    double *x;  // the iterate: FP64 in both solves
    T *r, *z, *p, *p2, *q, *dinv;
    float *xlo;  // mixed solve: the steps since the last k_cg_dir (null: x updated directly)
};

struct Sell {
    const uint32_t *off;
    const void *col;  // int32 columns, or int16 offsets from the row when c16
    bool c16;
    const double *v64;
    const float *v32;
    SellU U;
    const int2 *rec;  // per slice, for the resident solve (null: not made)
    bool fused;       // the mixed solve's product forms the direction
};

template <typename T>
const T *sell_vals(const Sell &S);
template <>
const double *sell_vals<double>(const Sell &S) { return S.v64; }
template <>
const float *sell_vals<float>(const Sell &S) { return S.v32; }

struct Parts {
    double *pq, *rz, *rr, *aux;
    int G;
};

template <typename T, typename TX, typename C>
void cg_group_as(hipStream_t st, int64_t n, const Sell &S, Vecs<T> &v, TX *xs, const Parts &P, double *sc, double *hsc)
{
    const dim3 g(P.G), b(SV_BLOCK);
    const C *col = (const C *)S.col;
    const T *val = sell_vals<T>(S);
    for (int k = 0; k < CHECK; k++) {
        const bool form = k > 0 && S.fused && sizeof(T) == 4;
        if (k > 0 && !form)
            hipLaunchKernelGGL((k_cg_dir<T, TX, false>), g, b, 0, st, n, P.rz, P.rr, (const T *)v.z, v.p, xs, v.x, sc,
                               (k - 1) & 1, hsc);
        hipLaunchKernelGGL((form ? k_cg_spmv<T, TX, C, sizeof(T) == 4, true>
                                 : k > 0 ? k_cg_spmv<T, TX, C, false, false> : k_cg_spmv<T, TX, C, false, true>),
                           g, b, 0, st, n, S.off, col, val, S.U, (const T *)v.z, (const T *)v.p, v.p2, v.q, xs, P.rz, sc, k & 1,
                           P.pq);
        if (form) std::swap(v.p, v.p2);
        hipLaunchKernelGGL((k_cg_update<T>), g, b, 0, st, n, (const T *)v.dinv, v.r, v.z, (const T *)v.q, P.pq, sc, k & 1,
                           P.rz, P.rr);
    }
    hipLaunchKernelGGL((k_cg_dir<T, TX, true>), g, b, 0, st, n, P.rz, P.rr, (const T *)v.z, v.p, xs, v.x, sc,
                       (CHECK - 1) & 1, hsc);
}

// CHECK PCG iterations on the stream; ||r||^2 goes to hsc[S_RR] (host) too.
void cg_group(hipStream_t st, int64_t n, const Sell &S, Vecs<double> &v, const Parts &P, double *sc, double *hsc)
{
    if (S.c16) cg_group_as<double, double, int16_t>(st, n, S, v, v.x, P, sc, hsc);
    else cg_group_as<double, double, int32_t>(st, n, S, v, v.x, P, sc, hsc);
}
void cg_group(hipStream_t st, int64_t n, const Sell &S, Vecs<float> &v, const Parts &P, double *sc, double *hsc)
{
    if (S.c16) cg_group_as<float, float, int16_t>(st, n, S, v, v.xlo, P, sc, hsc);
    else cg_group_as<float, float, int32_t>(st, n, S, v, v.xlo, P, sc, hsc);
}

// (a small number makes waits give up, for the tests of what follows then)
int ex_limit() { return std::max(1, env_int("ELFEL_HIP_PCG_POLLS", EX_LIMIT)); }

// Groups of iterations until ||r||^2 <= goal2 or maxit, in one launch; *it is
// carried on.  1: the device cannot run the launch (nothing has run).
template <typename T, typename TX, typename C>
int cg_small_as(hipStream_t st, int64_t n, const Sell &S, Vecs<T> &v, TX *xs, const Parts &P, uint64_t *slots, double *sc,
                double goal2, int it, int maxit)
{
    constexpr int VB = sizeof(T) == 8 ? SM_VB8 : SM_VB4;
    const int grid = (P.G + VB - 1) / VB;
    Exchange X{slots, P.G, ex_limit()};
    hipLaunchKernelGGL(k_cg_slots, dim3(ceil_div(3 * X.stride() / 8, 256)), dim3(256), 0, st, slots, 3 * X.stride() / 8, sc);
    const uint32_t *off = S.off;
    const C *col = (const C *)S.col;
    const T *val = sell_vals<T>(S);
    const T *dinv = v.dinv;
    const double *prz = P.rz;
    double *x = v.x;
    void *args[] = {&n, &off, &col, &val, &dinv, &v.r, &v.z, &v.p, &v.p2, &xs, &x, &prz, &X, &sc, &goal2, &it, &maxit};
    const hipError_t e = hipLaunchCooperativeKernel(reinterpret_cast<const void *>(&k_cg_small<T, TX, C, VB>), dim3(grid),
                                                    dim3(VB * SV_BLOCK), args, 0, st);
    if (e == hipSuccess) return 0;
    (void)hipGetLastError();
    return 1;
}
int cg_small(hipStream_t st, int64_t n, const Sell &S, Vecs<double> &v, const Parts &P, uint64_t *slots, double *sc,
             double goal2, int it, int maxit)
{
    return S.c16 ? cg_small_as<double, double, int16_t>(st, n, S, v, v.x, P, slots, sc, goal2, it, maxit)
                 : cg_small_as<double, double, int32_t>(st, n, S, v, v.x, P, slots, sc, goal2, it, maxit);
}
int cg_small(hipStream_t st, int64_t n, const Sell &S, Vecs<float> &v, const Parts &P, uint64_t *slots, double *sc,
             double goal2, int it, int maxit)
{
    return S.c16 ? cg_small_as<float, float, int16_t>(st, n, S, v, v.xlo, P, slots, sc, goal2, it, maxit)
                 : cg_small_as<float, float, int32_t>(st, n, S, v, v.xlo, P, slots, sc, goal2, it, maxit);
}

template <typename T, typename TX, int R>
int cg_resident_as(hipStream_t st, int64_t n, const Sell &S, Vecs<T> &v, TX *xs, const Parts &P, uint64_t *slots, double *sc,
                   double goal2, int it, int maxit)
{
    if (P.G < RES_GRID || P.G > RES_VB * RES_GRID) return 1;  // every block's work-items
    Exchange X{slots, P.G, ex_limit()};
    hipLaunchKernelGGL(k_cg_slots, dim3(ceil_div(3 * X.stride() / 8, 256)), dim3(256), 0, st, slots, 3 * X.stride() / 8, sc);
    const uint32_t *off = S.off;
    const int16_t *col = (const int16_t *)S.col;
    const T *val = sell_vals<T>(S);
    const int2 *rec = S.rec;
    const T *dinv = v.dinv;
    const double *prz = P.rz;
    double *x = v.x;
    void *args[] = {&n, &off, &col, &val, &rec, &dinv, &v.r, &v.z, &v.p, &v.p2, &xs, &x, &prz, &X, &sc, &goal2, &it, &maxit};
    const hipError_t e = hipLaunchCooperativeKernel(reinterpret_cast<const void *>(&k_cg_resident<T, TX, R>),
                                                    dim3(std::min(P.G, RES_GRID)), dim3(RES_BLOCK), args, 0, st);
    if (e == hipSuccess) return 0;
    (void)hipGetLastError();
    return 1;
}
template <typename T, typename TX>
void cg_one_as(hipStream_t st, int64_t n, const Sell &S, Vecs<T> &v, TX *xs, const Parts &P, double *sc, double goal2, int it,
            int maxit)
{
    auto kern = n <= RES_BLOCK ? k_cg_one<T, TX, 1> : n <= 2 * RES_BLOCK ? k_cg_one<T, TX, 2> : k_cg_one<T, TX, ONE_ROWS(T) / RES_BLOCK>;
    hipLaunchKernelGGL(kern, dim3(1), dim3(RES_BLOCK), 0, st, (int)n, P.G, S.off, (const int16_t *)S.col, sell_vals<T>(S), S.rec,
                       (const T *)v.dinv, v.r, v.p, xs, v.x, (const double *)P.rz, sc, goal2, it, maxit);
}
void cg_one(hipStream_t st, int64_t n, const Sell &S, Vecs<double> &v, const Parts &P, double *sc, double goal2, int it, int maxit)
{
    cg_one_as(st, n, S, v, v.x, P, sc, goal2, it, maxit);
}
void cg_one(hipStream_t st, int64_t n, const Sell &S, Vecs<float> &v, const Parts &P, double *sc, double goal2, int it, int maxit)
{
    cg_one_as(st, n, S, v, v.xlo, P, sc, goal2, it, maxit);
}
// Rows a work-item of the resident solve that n rows in G blocks need; most: 3
// FP64 (786 000 rows on 256 CUs), 8 mixed (2.1 million).
int cg_resident(hipStream_t st, int64_t n, const Sell &S, Vecs<double> &v, const Parts &P, uint64_t *slots, double *sc,
                double goal2, int it, int maxit)
{
    const int64_t r = (n + (int64_t)P.G * SV_BLOCK - 1) / ((int64_t)P.G * SV_BLOCK);
    if (r <= 1) return cg_resident_as<double, double, 1>(st, n, S, v, v.x, P, slots, sc, goal2, it, maxit);
    if (r <= 2) return cg_resident_as<double, double, 2>(st, n, S, v, v.x, P, slots, sc, goal2, it, maxit);
    if (r <= 3) return cg_resident_as<double, double, 3>(st, n, S, v, v.x, P, slots, sc, goal2, it, maxit);
    return 1;
}
int cg_resident(hipStream_t st, int64_t n, const Sell &S, Vecs<float> &v, const Parts &P, uint64_t *slots, double *sc,
                double goal2, int it, int maxit)
{
    const int64_t r = (n + (int64_t)P.G * SV_BLOCK - 1) / ((int64_t)P.G * SV_BLOCK);
    // (5 and 7 of their own gain less than 1 % on the next)
    if (r <= 1) return cg_resident_as<float, float, 1>(st, n, S, v, v.xlo, P, slots, sc, goal2, it, maxit);
    if (r <= 2) return cg_resident_as<float, float, 2>(st, n, S, v, v.xlo, P, slots, sc, goal2, it, maxit);
    if (r <= 4) return cg_resident_as<float, float, 4>(st, n, S, v, v.xlo, P, slots, sc, goal2, it, maxit);
    if (r <= 6) return cg_resident_as<float, float, 6>(st, n, S, v, v.xlo, P, slots, sc, goal2, it, maxit);
    if (r <= 8) return cg_resident_as<float, float, 8>(st, n, S, v, v.xlo, P, slots, sc, goal2, it, maxit);
    return 1;
}

}  // namespace

int pcg_solve(elfel_hip_ctx *c, int64_t nfree, const double *F, double *x, int precision, double tol, int maxit,
              int *iters, int *outer, double *relres)
{
    const int64_t n = nfree, N = c->nrow;
    const int32_t *ptr = result_ptr(c);
    const int32_t *ind = result_ind(c);
    const double *val = (const double *)c->val.p;
    if (n == 0) {
        if (iters) *iters = 0;
        if (outer) *outer = 0;
        if (relres) *relres = 0;
        return 0;
    }
    const bool mixed = precision == ELFEL_MIXED;
    const int64_t nslices = (n + 63) / 64;
    hipStream_t st = c->stream;
    int cus = 0;
    HIPCHK(c, hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device));
    // the CG grid: 4 workgroups per CU (grid-stride loops), fewer for small
    // systems (8 and 16 per CU measured slower on heat Q4 4096^2: 407 and 412
    // against 381 us per mixed iteration; every workgroup of the next kernel
    // sums G partials)
    const int G = (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div(n, SV_BLOCK), 4 * (int64_t)cus));

    // ---- scratch layout (8-byte words first, then 4-byte) -----------------
    // doubles: xfull[N], b[n], r64[n], dinv64[n], parts[4 G], slots, sc[S_NS],
    //          FP64 vectors r z p p2 q [5 m] (FP64 solve only)
    // floats:  r z p p2 q dinv xlo [7 m] (mixed solve only; its iterate is the FP64 xfull + xlo)
    // uint32:  off[nslices + 1], len[max(n, nslices)], total[4]
    // The vectors and the slots begin on 256 bytes: a wave's stores fill whole lines.
    const size_t m = ((size_t)n + 63) & ~(size_t)63;
    const size_t nd = (size_t)N + 3 * (size_t)n + 4 * (size_t)G + 3 * EX_STRIDE((size_t)G) / 8 + S_NS + 64 + (mixed ? 0 : 5 * m);
    const size_t nf = mixed ? 7 * m : 0;
    const size_t nu32 = (size_t)nslices + 1 + (size_t)std::max<int64_t>(n, nslices) + 4;
    int rc = ensure(c, c->pcg, 8 * nd + 4 * nf + 4 * nu32 + 256);
    if (rc) return rc;
    double *dp = (double *)c->pcg.p;
    double *xfull = dp; dp += N;
    double *b = dp; dp += n;
    double *r64 = dp; dp += n;
    double *dinv64 = dp; dp += n;
    Parts P;
    P.G = G;
    P.pq = dp; dp += G; P.rz = dp; dp += G; P.rr = dp; dp += G; P.aux = dp; dp += G;
    double *sc = dp; dp += S_NS;
    dp = (double *)(((uintptr_t)dp + 255) & ~(uintptr_t)255);
    uint64_t *slots = (uint64_t *)dp; dp += 3 * EX_STRIDE((size_t)G) / 8;
    dp = (double *)(((uintptr_t)dp + 255) & ~(uintptr_t)255);
    Vecs<double> v64{};
    if (!mixed) {
        v64.x = xfull;  // the free part of the full vector is the iterate
        v64.r = dp; dp += m; v64.z = dp; dp += m; v64.p = dp; dp += m; v64.p2 = dp; dp += m; v64.q = dp; dp += m;
        v64.dinv = dinv64;
    }
    float *fp = (float *)dp;
    Vecs<float> v32{};
    if (mixed) {
        v32.x = xfull;  // the free part of the full vector is the iterate (FP64)
        v32.r = fp; fp += m; v32.z = fp; fp += m; v32.p = fp; fp += m; v32.p2 = fp; fp += m; v32.q = fp; fp += m;
        v32.dinv = fp; fp += m;
        v32.xlo = fp; fp += m;
    }
    uint32_t *up = (uint32_t *)fp;
    uint32_t *off = up; up += nslices + 1;
    uint32_t *len = up; up += std::max<int64_t>(n, nslices);
    uint32_t *total = up;

    const HostIn in[2] = {{x, xfull, N, false, 0, 0}, {F, b, n, false, 0, 0}};
    if ((rc = to_device(c, in, 2, nullptr))) return rc;

    // ---- SELL-64 of the free block ------------------------------------------
    hipLaunchKernelGGL(k_fill<uint32_t>, dim3(1), dim3(64), 0, st, (int64_t)4, total, 0u);
    hipLaunchKernelGGL(k_sell_rowlen, dim3(ceil_div(n, 256)), dim3(256), 0, st, n, ptr, ind, len, total + 1);
    hipLaunchKernelGGL(k_sell_width, dim3(ceil_div(nslices * 64, 256)), dim3(256), 0, st, n, nslices, len, off, total + 2);
    if ((rc = exclusive_scan_u32(c, off, nslices, total))) return rc;
    volatile const uint32_t *tot = (const uint32_t *)c->told + 8;
    hipLaunchKernelGGL(k_tell, dim3(1), dim3(64), 0, st, (const uint32_t *)total, (uint32_t *)c->told + 8);
    HIPCHK(c, hipStreamSynchronize(st));
    const bool narrow = tot[2] == 0;  // no row of more than SELL_UNROLL entries
    const uint32_t nnzp = tot[0];
    const bool c16 = tot[1] == 0;  // every free column within a 16-bit offset of its row
    HIPCHK(c, hipMemcpyAsync(off + nslices, total, 4, hipMemcpyDeviceToDevice, st));
    // SELL arrays in a buffer of their own (the size is known only now)
    const size_t cbytes = (size_t)nnzp * (c16 ? 2 : 4);
    const size_t nslots = (size_t)nnzp / 64;
    const size_t vbytes = (size_t)nnzp * (8 + (mixed ? 4 : 0));
    const size_t sbytes = ((cbytes + 15) & ~(size_t)15) + vbytes + 4 * (size_t)(nslices + 1) + 4 * (nslots + SELL_UNROLL) +
                          16 * (size_t)(nslices + 1) + 256;
    if ((rc = ensure(c, c->pcg_sell, sbytes))) return rc;
    void *scol = c->pcg_sell.p;
    double *sv64 = (double *)((char *)c->pcg_sell.p + ((cbytes + 15) & ~(size_t)15));
    float *sv32 = mixed ? (float *)(sv64 + nnzp) : nullptr;
    uint32_t *uflag = (uint32_t *)((char *)sv64 + vbytes);
    int32_t *uoff = (int32_t *)(uflag + nslices + (nslices & 1));
    if (c16)
        hipLaunchKernelGGL((k_sell_fill<int16_t>), dim3(ceil_div(nslices * 64, 256)), dim3(256), 0, st, n, ptr, ind, val,
                           off, (int16_t *)scol, sv64, sv32);
    else
        hipLaunchKernelGGL((k_sell_fill<int32_t>), dim3(ceil_div(nslices * 64, 256)), dim3(256), 0, st, n, ptr, ind, val,
                           off, (int32_t *)scol, sv64, sv32);
    const bool uniform_slots = env_int("ELFEL_HIP_SELL_UNIFORM", 1) != 0;
    if (uniform_slots) {
        if (c16)
            hipLaunchKernelGGL((k_sell_uniform<int16_t>), dim3(ceil_div(nslices * 64, 256)), dim3(256), 0, st, n,
                               nslices, (const uint32_t *)off, (const int16_t *)scol, uflag, uoff, total + 3);
        else
            hipLaunchKernelGGL((k_sell_uniform<int32_t>), dim3(ceil_div(nslices * 64, 256)), dim3(256), 0, st, n,
                               nslices, (const uint32_t *)off, (const int32_t *)scol, uflag, uoff, total + 3);
    } else {
        hipLaunchKernelGGL(k_sell_empty, dim3(ceil_div(nslices, 256)), dim3(256), 0, st, nslices, (const uint32_t *)off, uflag);
    }
    hipLaunchKernelGGL(k_diag_inv, dim3(ceil_div(n, 256)), dim3(256), 0, st, n, ptr, ind, val, dinv64,
                       mixed ? v32.dinv : nullptr);
    HIPCHK(c, hipGetLastError());
    // records for the resident solve where rows are narrow and columns near
    const bool near9 = c16 && narrow;
    int2 *rec = (int2 *)(((uintptr_t)(uoff + nslots + SELL_UNROLL) + 15) & ~(uintptr_t)15);
    if (near9)
        hipLaunchKernelGGL(k_sell_rec, dim3(ceil_div(nslices * 64, 256)), dim3(256), 0, st, n, nslices,
                           (const uint32_t *)off, (const int16_t *)scol, (const uint32_t *)len, rec, total + 1);
    hipLaunchKernelGGL(k_tell, dim3(1), dim3(64), 0, st, (const uint32_t *)total, (uint32_t *)c->told + 8);
    Sell S{off, scol, c16, sv64, sv32, SellU{uflag, uoff}, near9 ? rec : nullptr, false};

    // the scalars as the last reduction left them, in pinned memory
    double *hsc = (double *)c->told + 8;
    // b = F_f - K_fd x_d, ||b||
    hipLaunchKernelGGL(k_rhs, dim3(G), dim3(SV_BLOCK), 0, st, n, ptr, ind, val, (const double *)xfull,
                       (const double *)b, b, P.aux);
    hipLaunchKernelGGL(k_reduce, dim3(1), dim3(1024), 0, st, (const double *)P.aux, G, sc, (int)S_BB,
                       (const double *)nullptr, 0, (double *)nullptr);
    // r64 = b - A x (FP64), its norm; waits
    auto true_residual = [&](double *out_norm) -> int {
        if (S.c16)
            hipLaunchKernelGGL((k_sell_resid<int16_t>), dim3(G), dim3(SV_BLOCK), 0, st, n, S.off,
                               (const int16_t *)S.col, S.v64, S.U, (const double *)xfull, (const double *)b, r64,
                               P.aux);
        else
            hipLaunchKernelGGL((k_sell_resid<int32_t>), dim3(G), dim3(SV_BLOCK), 0, st, n, S.off,
                               (const int32_t *)S.col, S.v64, S.U, (const double *)xfull, (const double *)b, r64,
                               P.aux);
        hipLaunchKernelGGL(k_reduce, dim3(1), dim3(1024), 0, st, (const double *)P.aux, G, sc, (int)S_RR64,
                           (const double *)nullptr, 0, hsc);
        HIPCHK(c, hipGetLastError());
        HIPCHK(c, hipStreamSynchronize(st));
        *out_norm = sqrt(std::max(hsc[S_RR64], 0.0));
        return 0;
    };
    // r = (T) r64, z = M r (p = z on restart); sc gets rz and ||r||^2
    auto reset = [&](auto &v, int restart) {
        using T = typename std::remove_pointer<decltype(v.r)>::type;
        hipLaunchKernelGGL((k_cg_reset<T>), dim3(G), dim3(SV_BLOCK), 0, st, n, (const double *)r64,
                           (const T *)v.dinv, v.r, v.z, v.p, restart, P.rz, P.rr);
        hipLaunchKernelGGL(k_reduce, dim3(1), dim3(1024), 0, st, (const double *)P.rr, G, sc, (int)S_RR,
                           (const double *)P.rz, (int)S_RZ, hsc);
    };

    int it = 0, nupd = 0;
    double rn = 0.0;
    if ((rc = true_residual(&rn))) return rc;
    const bool resident = near9 && tot[1] == 0;
    S.fused = env_int("ELFEL_HIP_PCG_FUSED", 2 * tot[3] >= (nslices + UNI_STEP - 1) / UNI_STEP) != 0;
    bool lost = false;  // a one-launch solve's workgroups did not all run: several launches an iteration from then on
    const double bnorm = hsc[S_BB] > 0 ? sqrt(hsc[S_BB]) : 1.0;
    const double target = tol * bnorm;
    // Iterations until ||r||^2 <= goal2 or maxit from the state of the last reset,
    // then the true residual (waits): *rrec the recurrence's ||r||^2, *norm the
    // true residual's norm.  One launch of one workgroup where all slices have
    // records and there are few rows; of many where every row has its own
    // work-item, the rows fit its registers and there are few enough workgroups,
    // or where all slices have records and the rows fit the chip's registers.
    const bool one_launch = env_int("ELFEL_HIP_PCG_ONE_LAUNCH", 1) != 0;
    auto solve_to = [&](auto &v, double goal2, double *rrec, double *norm) -> int {
        using T = typename std::remove_pointer<decltype(v.r)>::type;
        constexpr int VB = sizeof(T) == 8 ? SM_VB8 : SM_VB4;
        const bool small = narrow && n <= (int64_t)P.G * SV_BLOCK && (P.G + VB - 1) / VB <= SM_GRID;
        bool one = one_launch && resident && n <= ONE_ROWS(T);
        if (one) cg_one(st, n, S, v, P, sc, goal2, it, maxit);
        else one = one_launch && !lost && ((small && cg_small(st, n, S, v, P, slots, sc, goal2, it, maxit) == 0) ||
                                            (resident && cg_resident(st, n, S, v, P, slots, sc, goal2, it, maxit) == 0));
        if (one) {
            if ((rc = true_residual(norm))) return rc;
            lost = hsc[S_LOST] != 0.0;
            it = (int)hsc[S_IT];
            *rrec = lost ? 0.0 : hsc[S_RREC];  // 0: the next reset restarts from p = z
            return 0;
        }
        for (;;) {
            HIPCHK(c, hipStreamSynchronize(st));
            *rrec = hsc[S_RR];
            if (!(*rrec > goal2) || it >= maxit) break;
            cg_group(st, n, S, v, P, sc, hsc);
            HIPCHK(c, hipGetLastError());
            it += CHECK;
        }
        return true_residual(norm);
    };
    double rrec = 0.0;  // recurrence residual norm^2 at the last check
    if (!mixed) {
        reset(v64, 1);
        nupd = 1;
        while (rn > target && it < maxit) {
            // iterate until the recurrence residual reaches the target, then
            // check the true residual and continue from it if needed
            if ((rc = solve_to(v64, target * target, &rrec, &rn))) return rc;
            if (rn > target && it < maxit) {
                reset(v64, !(sqrt(std::max(rrec, 0.0)) >= RU_KEEP * rn));
                nupd++;
            }
        }
    } else {
        hipLaunchKernelGGL(k_fill<float>, dim3(ceil_div(n, 256)), dim3(256), 0, st, n, v32.xlo, 0.f);
        reset(v32, 1);
        double rlast = rn;
        while (rn > target && it < maxit) {
            const double goal = std::max(target, RU_DROP * rlast);
            // reliable update: the FP64 residual b - A x replaces the FP32 one
            if ((rc = solve_to(v32, goal * goal, &rrec, &rn))) return rc;
            nupd++;
            rlast = rn;
            // The search direction is kept while the recurrence still tracks the true residual; once
            // it has run far below it (FP32 round-off, or a tiny system solved exactly) p no longer
            // belongs to the new residual and the iteration restarts from p = z.
            if (rn > target && it < maxit) reset(v32, !(sqrt(std::max(rrec, 0.0)) >= RU_KEEP * rn));
        }
    }
    HIPCHK(c, hipGetLastError());
    const HostOut o{x, xfull, n, false, 0};
    if ((rc = to_host(c, &o, 1))) return rc;
    if (iters) *iters = it;
    if (outer) *outer = nupd;
    if (relres) *relres = rn / bnorm;
    return 0;
}
