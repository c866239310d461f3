// Host-only check of the nine-entry rows of the one-launch solves
// (elfel.jl_amd/csrc/nine.h), built and run by tests/test_nine_slots.py: over
// narrow grids of triangles (both diagonals) and quadrilaterals and over bands,
// in slices of 64 rows, the operator that the slots hold equals the matrix that
// was put into them wherever a slice fits, and the slices of three runs fit.
// Prints one line per failed check and exits with their number.
#include <cstdio>
#include <map>
#include <string>
#include <vector>

#include "nine.h"

typedef std::vector<std::map<int, double>> Matrix;  // a row: column -> value

static int fails = 0, checked = 0;

// rows of a grid of w x h nodes, the short side first; kind 0, 1: triangles with
// either diagonal, 2: quadrilaterals
static Matrix grid(int w, int h, int kind)
{
    Matrix A(w * h);
    for (int y = 0; y < h; y++)
        for (int x = 0; x < w; x++)
            for (int dy = -1; dy <= 1; dy++)
                for (int dx = -1; dx <= 1; dx++) {
                    if (x + dx < 0 || x + dx >= w || y + dy < 0 || y + dy >= h) continue;
                    if (kind < 2 && dx * dy == (kind ? -1 : 1)) continue;
                    const int i = y * w + x, j = (y + dy) * w + x + dx;
                    A[i][j] = 1.0 + i + 0.001 * j;
                }
    return A;
}

static Matrix band(int n, const std::vector<int> &offsets)
{
    Matrix A(n);
    for (int i = 0; i < n; i++)
        for (int d : offsets)
            if (i + d >= 0 && i + d < n) A[i][i + d] = 1.0 + i + 0.001 * (i + d);
    return A;
}

// three: whether the matrix has three runs everywhere, so that all slices fit
static void check(const Matrix &A, bool three, const std::string &what)
{
    const int n = (int)A.size();
    for (int s = 0; s * 64 < n; s++) {
        NineRuns R;
        for (int i = s * 64; i < n && i < s * 64 + 64; i++)
            for (auto &e : A[i]) R.add(e.first - i);
        if (three && !R.fit()) {
            printf("FAIL %s: slice %d does not fit\n", what.c_str(), s);
            fails++;
        }
        if (!R.fit()) continue;
        for (int i = s * 64; i < n && i < s * 64 + 64; i++) {
            double v[RES_W] = {0};
            for (auto &e : A[i]) nine_put(e.second, e.first - i, R.lo, R.hi, v);
            std::map<int, double> row;
            for (int j = 0; j < RES_W; j++)
                if (v[j] != 0.0) row[i + nine_offset(j, R.lo, R.hi)] += v[j];
            checked++;
            if (row != A[i]) {
                printf("FAIL %s: row %d\n", what.c_str(), i);
                fails++;
                return;
            }
        }
    }
}

int main()
{
    for (int w = 1; w <= 6; w++)
        for (int h : {2, 3, 60, 130})
            for (int kind = 0; kind < 3; kind++)
                check(grid(w, h, kind), true, "grid " + std::to_string(w) + " x " + std::to_string(h) + " kind " + std::to_string(kind));
    for (int k = 2; k <= 9; k++) check(band(300, {-k, -1, 0, 1, k}), true, "band of offset " + std::to_string(k));
    check(band(300, {-2, -1, 0, 1, 2}), true, "pentadiagonal");
    check(band(300, {-3, -2, -1, 0, 1, 2, 3}), true, "seven diagonals");
    check(band(300, {-4, -3, -2, -1, 0, 1, 2, 3, 4}), true, "nine diagonals");
    check(band(300, {-1, 0, 1}), true, "tridiagonal");
    check(band(300, {0}), true, "diagonal");
    check(band(300, {-7, -2, 0, 2, 7}), false, "five runs");
    check(band(300, {-5, -4, -3, -2, -1, 0, 1, 2, 3, 4, 5}), false, "eleven diagonals");
    if (checked < 5000) {
        printf("FAIL only %d rows\n", checked);
        fails++;
    }
    if (!fails) printf("OK\n");
    return fails;
}
