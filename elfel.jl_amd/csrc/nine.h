// nine.h -- how the one-launch solves (solve.hip) take the rows of a slice of 64
// into registers: the slots that a row of any narrow slice reads, and, for rows
// of nine entries in three runs, which slices have them and which register an
// entry takes.
//
// Slots 0-2 are the entries at lo, lo + 1, lo + 2 from the diagonal, 3-5 those at
// -1, 0, 1, and 6-8 those at hi, hi + 1, hi + 2, with lo the slice's smallest
// offset below -1 and hi its smallest above 1.  The lower run of a narrow band
// reaches the centre (lo of -3 or -2: two nodes across a grid), so an entry's
// own offset says which of the three runs it belongs to; the slots that the
// centre takes from the lower run stay zero.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define RES_W 9
#define NINE_NONE (1 << 20)  // a run without entries: no offset is so large

// Where entry k of lane's row is read in a slice that begins at o and is w
// entries wide: past its width the first once more (it adds nothing), and in a
// slice of no entries (64 rows of dofs of no element) nowhere: -1.
__host__ __device__ __forceinline__ int64_t sell_slot(uint32_t o, uint32_t w, uint32_t k, int lane)
{
    return w == 0 ? -1 : (int64_t)o + (int64_t)(k < w ? k : 0) * 64 + lane;
}

// The ends of a slice's lower and upper runs.
struct NineRuns {
    int32_t lo = NINE_NONE, lo_end = -NINE_NONE, hi = NINE_NONE, hi_end = -NINE_NONE;
    __host__ __device__ __forceinline__ void add(int32_t d)
    {
        if (d < -1) {
            lo = d < lo ? d : lo;
            lo_end = d > lo_end ? d : lo_end;
        } else if (d > 1) {
            hi = d < hi ? d : hi;
            hi_end = d > hi_end ? d : hi_end;
        }
    }
    __host__ __device__ __forceinline__ bool fit() const { return lo_end - lo <= 2 && hi_end - hi <= 2; }
};

// Entry x at offset d of a slice that fits, into its slot of v.
template <typename T>
__host__ __device__ __forceinline__ void nine_put(T x, int32_t d, int32_t lo, int32_t hi, T *v)
{
    const int32_t slot = d < -1 ? d - lo : d <= 1 ? d + 4 : d - hi + 6;
#pragma unroll
    for (int j = 0; j < RES_W; j++)  // (v is in registers: no index that is not a constant)
        if (j == slot) v[j] = x;
}

// The offset of the row that slot j is multiplied with.
__host__ __device__ __forceinline__ int32_t nine_offset(int j, int32_t lo, int32_t hi)
{
    return (j < 3 ? lo : j < 6 ? -1 : hi) + j % 3;
}
