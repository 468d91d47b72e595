// gf_stage.hpp -- the arithmetic of a staged box: which of its cells a query's
// ball can meet.  The same functions on host and device: every conversion to
// an integer is of a value already inside the integer's range, so none depends
// on how the target converts values outside it.
#pragma once

#include "gf_internal.hpp"

namespace gf {

// A box staged in LDS: its faces and its cells (counts and 1 / edges).
struct StageBox {
    double X0 = 0, X1 = 0, Y0 = 0, Y1 = 0, Z0 = 0, Z1 = 0;
    float hx = 0, hy = 0, hz = 0;
    int nx = 1, ny = 1, nz = 1;
};

// Cells [x0, x1] of rows [y0, y1] of layers [z0, z1]; no row when y0 > y1.
struct CellRange {
    int x0, x1, y0, y1, z0, z1;
};

// The cell, of n along an axis with 1 / edge h, at offset v from the face.
__host__ __device__ inline int stage_cell(float v, float h, int n)
{
    return static_cast<int>(fminf(fmaxf(v * h, 0.0f), static_cast<float>(n - 1)));
}

// The cells within e of a query at offset (fx, fy, fz) from the box's low
// faces.  A lane without an active query gets no cell: its offset is of no
// point in the box, and may be so many cells away that a walk from there would
// not end.
__host__ __device__ inline CellRange stage_range(const StageBox& B, bool act, float fx, float fy,
                                                 float fz, float e)
{
    if (!act) return CellRange{0, 0, 0, -1, 0, -1};
    return CellRange{stage_cell(fx - e, B.hx, B.nx), stage_cell(fx + e, B.hx, B.nx),
                     stage_cell(fy - e, B.hy, B.ny), stage_cell(fy + e, B.hy, B.ny),
                     stage_cell(fz - e, B.hz, B.nz), stage_cell(fz + e, B.hz, B.nz)};
}

} // namespace gf
