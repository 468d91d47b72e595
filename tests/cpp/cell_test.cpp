// cell_test.cpp -- the arithmetic of the search kernels' staged boxes, on the
// host (the kernels call the same functions).
#include "gf_stage.hpp"

#include <cmath>
#include <random>

#include "mini_test.hpp"

using namespace gf;

namespace {

// The kernels' row loops: steps until no row is left, at most `cap`.
int row_steps(int y0, int y1, int cap)
{
    int steps = 0;
    for (int dy = 0; steps < cap; ++dy, ++steps) {
        const int y = static_cast<int>(static_cast<unsigned>(y0) + static_cast<unsigned>(dy));
        if (!(y <= y1)) break;
    }
    return steps;
}

struct Offset {
    float x, y, z;
};

// Offsets of points from the low faces of boxes at large negative coordinates
// (what a lane without a query, at the origin, has) and cell edges of fine or
// coincident clouds.
const Offset kFar[] = {{-1.0f, 5.0f, 0.0f}, {3e6f, 4e6f, 2e5f}, {1e18f, 1e18f, 1e18f},
                       {-4e6f, 4e6f, 1e-9f}, {0.0f, 1e30f, 0.0f}};
const float kEdges[] = {1e-18f, 1.2e-10f, 4e-4f, 0.5f, 1e6f};

} // namespace

TEST(Cells, IdleLanesHaveNoRow)
{
    for (const Offset& o : kFar)
        for (float edge : kEdges) {
            StageBox B;
            B.nx = 7;
            B.ny = 11;
            B.nz = 3;
            B.hx = B.hy = B.hz = 1.0f / edge;
            const CellRange w = stage_range(B, false, o.x, o.y, o.z, edge);
            EXPECT_EQ(row_steps(w.y0, w.y1, 100), 0);
            EXPECT_EQ(row_steps(w.z0, w.z1, 100), 0);
        }
}

TEST(Cells, RangesStayInsideTheBox)
{
    for (const Offset& o : kFar)
        for (float edge : kEdges)
            for (int n : {1, 2, 512}) {
                StageBox B;
                B.nx = B.ny = B.nz = n;
                B.hx = B.hy = B.hz = 1.0f / edge;
                const CellRange w = stage_range(B, true, o.x, o.y, o.z, edge);
                EXPECT_TRUE(w.x0 >= 0 && w.x0 <= w.x1 && w.x1 < n);
                EXPECT_TRUE(w.y0 >= 0 && w.y0 <= w.y1 && w.y1 < n);
                EXPECT_TRUE(w.z0 >= 0 && w.z0 <= w.z1 && w.z1 < n);
                EXPECT_EQ(row_steps(w.y0, w.y1, 1000), w.y1 - w.y0 + 1);
            }
}

TEST(Cells, RangeHoldsEveryPointInReach)
{
    // Points of a box within e of a query are in cells of its range.
    std::mt19937 rng(7);
    std::uniform_real_distribution<float> u(0.0f, 1.0f);
    for (float scale : {1e-15f, 1e-3f, 1.0f, 1e17f})
        for (int t = 0; t < 20000; ++t) {
            StageBox B;
            B.nx = B.ny = B.nz = 1 + t % 40;
            const float L = scale, edge = L / static_cast<float>(B.nx);
            B.hx = B.hy = B.hz = 1.0f / edge;
            const float q[3] = {L * u(rng), L * u(rng), L * u(rng)};
            const float p[3] = {L * u(rng), L * u(rng), L * u(rng)};
            float far = 0.0f;
            for (int d = 0; d < 3; ++d) far = std::fmax(far, std::fabs(p[d] - q[d]));
            const CellRange w = stage_range(B, true, q[0], q[1], q[2],
                                            far * 1.0001f + 1e-6f * (q[0] + q[1] + q[2]));
            const int c[3] = {stage_cell(p[0], B.hx, B.nx), stage_cell(p[1], B.hy, B.ny),
                              stage_cell(p[2], B.hz, B.nz)};
            EXPECT_TRUE(w.x0 <= c[0] && c[0] <= w.x1);
            EXPECT_TRUE(w.y0 <= c[1] && c[1] <= w.y1);
            EXPECT_TRUE(w.z0 <= c[2] && c[2] <= w.z1);
        }
}

int main(int argc, char** argv) { return mini::run_all(argc, argv); }
