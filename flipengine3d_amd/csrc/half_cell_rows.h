// The rows of half-cells around a corner of the half-cell grid, nearest first,
// for searches of the nearest particle.
#pragma once

#include <hip/hip_runtime.h>

namespace flipmi {

constexpr int kCellRows = 100;  // 10 x 10 rows of half-cells around a cell
static_assert(kCellRows % 4 == 0, "rows are walked four at a time");

// Rows (oy, oz), half-cells relative to the cell's first, by their distance
// from the cell's centre: half-cells 0 and 1 touch it, -1 and 2 lie half a
// cell away, and so on to two cells (ring 4).
struct CellRow {
    signed char oy, oz, ry, rz;  // offsets and rings
};
struct CellRows {
    CellRow r[kCellRows];
};
constexpr CellRows make_cell_rows() {
    CellRows t{};
    int n = 0;
    for (int d = 0; d <= 32; d++)
        for (int oz = -4; oz <= 5; oz++)
            for (int oy = -4; oy <= 5; oy++) {
                const int ry = oy < 1 ? -oy : oy - 1, rz = oz < 1 ? -oz : oz - 1;
                if (ry * ry + rz * rz == d)
                    t.r[n++] = CellRow{(signed char)oy, (signed char)oz, (signed char)ry, (signed char)rz};
            }
    return t;
}
static __constant__ CellRows c_cell_rows = make_cell_rows();

}  // namespace flipmi
