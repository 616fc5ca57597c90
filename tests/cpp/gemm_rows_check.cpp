// CPU check of the rows that the 128 x 128 GEMM's loads read (mx_kernels.hpp: gemm_load_row): for every operand height
// from 1 row up, every tile and every load of it stays inside the operand, and loads of rows that exist read those rows.
// (An offset formed from a clamped base had read up to 16 rows ahead of the operand at heights of 9 to 16.)
#include <cstdio>

#include "mx_kernels.hpp"

int main() {
    constexpr int kTile = 128;
    for (int rows = 1; rows <= 600; rows++)
        for (int first = 0; first < rows; first += kTile)
            for (int row = 0; row < kTile; row++) {
                const int r = mx::gemm_load_row(first, row, rows);
                const int want = first + row < rows ? first + row : rows - 1;
                if (r != want) {
                    std::printf("rows %d: load %d of the tile at %d reads row %d, not %d\n", rows, row, first, r, want);
                    return 1;
                }
            }
    return 0;
}
