// Host-only check of the slots that a row of the small one-launch solve reads
// (sell_slot in elfel.jl_amd/csrc/nine.h), built and run by
// tests/test_small_slots.py: over matrices with runs of empty rows (dofs of no
// element) at the front, in the middle and at the end, stored in slices of 64
// rows as the solver stores them, every slot that is read lies in the row's own
// slice, holds its entry (or, past the row's entries, one that adds nothing),
// and its column is a row of the system, for 16-bit offsets and 32-bit columns;
// a slice without entries is not read at all.
#include <cstdio>
#include <random>
#include <string>
#include <vector>

#include "nine.h"

static int fails = 0, empty = 0, checked = 0;

struct Sell {
    std::vector<uint32_t> off;
    std::vector<int32_t> col;  // absolute columns, or offsets from the row
    std::vector<double> val;
};

static Sell store(const std::vector<std::vector<int>> &A, bool offsets)
{
    const int n = (int)A.size(), ns = (n + 63) / 64;
    Sell S;
    for (int s = 0; s < ns; s++) {
        size_t w = 0;
        for (int i = s * 64; i < n && i < s * 64 + 64; i++) w = std::max(w, A[i].size());
        S.off.push_back((uint32_t)S.col.size());
        for (size_t k = 0; k < w; k++)
            for (int i = s * 64; i < s * 64 + 64; i++) {
                const bool real = i < n && k < A[i].size();
                const int c = real ? A[i][k] : i < n ? i : 0;
                S.col.push_back(offsets ? (i < n ? c - i : 0) : c);
                S.val.push_back(real ? 1.0 + c : 0.0);
            }
    }
    S.off.push_back((uint32_t)S.col.size());
    return S;
}

// block: rows of a workgroup; the rows past the last read the last row's slots
static void check(const std::vector<std::vector<int>> &A, int block, const std::string &what)
{
    const int n = (int)A.size();
    for (int offsets = 0; offsets < 2; offsets++) {
        const Sell S = store(A, offsets != 0);
        for (int64_t i = 0; i < (int64_t)((n + block - 1) / block) * block; i++) {
            const int ic = (int)std::min<int64_t>(i, n - 1);
            const uint32_t s = (uint32_t)ic >> 6, o = S.off[s], w = (S.off[s + 1] - o) >> 6;
            for (int k = 0; k < 12; k++) {
                const int64_t at = sell_slot(o, w, k, ic & 63);
                if (at < 0) {
                    empty++;
                    if (w != 0) {
                        printf("FAIL %s: row %d is not read\n", what.c_str(), ic);
                        fails++;
                        return;
                    }
                    continue;
                }
                checked++;
                const bool inside = at >= (int64_t)o && at < (int64_t)S.off[s + 1] && at < (int64_t)S.col.size();
                const int c = inside ? S.col[at] + (offsets ? ic : 0) : -1;
                const bool own = k < (int)w ? (k < (int)A[ic].size() ? c == A[ic][k] : S.val[at] == 0.0) : true;
                if (!inside || c < 0 || c >= n || !own) {
                    printf("FAIL %s: row %d entry %d slot %lld\n", what.c_str(), ic, k, (long long)at);
                    fails++;
                    return;
                }
            }
        }
    }
}

int main()
{
    std::mt19937 rng(4);
    for (int n : {1, 63, 64, 65, 200, 513, 769, 1600, 5000})
        for (int front : {0, 64, 130})
            for (int back : {0, 63, 64, 65, 200, 700})
                for (int middle : {0, 128}) {
                    std::vector<std::vector<int>> A(front + n + middle + back);
                    for (int i = 0; i < n; i++) {
                        const int row = front + i + (i >= n / 2 ? middle : 0);
                        for (int d = -3; d <= 3; d++)
                            if (i + d >= 0 && i + d < n && (d == 0 || rng() % 3)) {
                                const int j = i + d;
                                A[row].push_back(front + j + (j >= n / 2 ? middle : 0));
                            }
                    }
                    const std::string what = std::to_string(front) + " + " + std::to_string(n) + " + " + std::to_string(back) +
                                             " rows, " + std::to_string(middle) + " empty between";
                    check(A, 512, what);
                    check(A, 768, what);
                }
    check(std::vector<std::vector<int>>(300), 512, "no entries");
    if (!empty || !checked) {
        printf("FAIL nothing was checked\n");
        fails++;
    }
    if (!fails) printf("OK\n");
    return fails;
}
