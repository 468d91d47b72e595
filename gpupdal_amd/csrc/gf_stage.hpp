// gf_stage.hpp -- the arithmetic of a staged box: its cells, which of them a
// query's ball can meet, and the coarse keys of its candidates.  The same
// functions on host and device: every conversion to an integer is of a value
// already inside the integer's range, so none depends on how the target
// converts values outside it.
#pragma once

#include "gf_internal.hpp"

#include <cfloat>

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

// The FP32 arithmetic of staged boxes serves coordinates and radii below this:
// a box reaches at most 1.3 of it beyond its queries, so that squared distances
// are at most 3 (2 + 1.3)^2 kStageFar^2 = 3.3e37, below FLT_MAX.  Other rows are
// searched in FP64 alone.
constexpr double kStageFar = 1e18;

// Whether the query-per-lane search takes the queries of a grid whose search
// radius is bounded by `reach` (before the margin is taken off it).
__host__ __device__ inline bool stage_takes(double reach, double margin)
{
    return reach < kStageFar && reach > 4.0 * margin;
}

__host__ __device__ inline bool stage_takes_point(double x, double y, double z)
{
    return fabs(x) < kStageFar && fabs(y) < kStageFar && fabs(z) < kStageFar;
}

// Cells of a box for searches of radius r: a third of it along x (runs are
// cut there), half of it along y, the radius along z when the box is tall;
// larger until they are at most `cells`.  False where no edge serves.
__host__ __device__ inline bool stage_size(StageBox& B, float r, int cells)
{
    const float Lx = static_cast<float>(B.X1 - B.X0), Ly = static_cast<float>(B.Y1 - B.Y0),
                Lz = static_cast<float>(B.Z1 - B.Z0);
    const bool tall = Lz > 4.0f * r;
    float cx = r * 0.34f, cy = r * 0.5f, cz = r;
    // (a bounded number of steps, whatever r and the faces: 1.3^128 = 4e14)
    for (int step = 0; step < 128; ++step) {
        B.nx = static_cast<int>(fminf(Lx / cx, 1000.0f)) + 1;
        B.ny = static_cast<int>(fminf(Ly / cy, 1000.0f)) + 1;
        B.nz = tall ? static_cast<int>(fminf(Lz / cz, 1000.0f)) + 1 : 1;
        if (B.nx * B.ny * B.nz <= cells) {
            B.hx = 1.0f / cx;
            B.hy = 1.0f / cy;
            B.hz = tall ? 1.0f / cz : 0.0f;
            return true;
        }
        cx *= 1.3f;
        cy *= 1.3f;
        cz *= 1.3f;
    }
    return false;
}

// A candidate's 32-bit key: its squared distance as FP32 without the low bits,
// the candidate's slot in their place.
constexpr uint32_t kSlotMask = 0x3FFu;

__host__ __device__ inline uint32_t list_key(double d2, uint32_t slot)
{
    const float f = static_cast<float>(d2);
    uint32_t u;
    __builtin_memcpy(&u, &f, sizeof(u));
    return (u & ~kSlotMask) | slot;
}

__host__ __device__ inline double key_value(uint32_t u)
{
    float f;
    __builtin_memcpy(&f, &u, sizeof(f));
    return static_cast<double>(f);
}

// Candidates whose d2 is at or above this have larger keys than `key` has.
__host__ __device__ inline double key_above(uint32_t key)
{
    return key_value((key | kSlotMask) + 1u);
}

// No candidate of this key or a larger one has a smaller d2.  (The float
// rounds a double by 6e-8; below FLT_MIN by an absolute amount, and nothing is
// claimed there.)
__host__ __device__ inline double key_below(uint32_t key)
{
    const double v = key_value(key & ~kSlotMask);
    return v >= static_cast<double>(FLT_MIN) ? v * (1.0 - 1.2e-7) : 0.0;
}

} // namespace gf
