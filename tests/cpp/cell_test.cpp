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

TEST(Cells, SizingEndsForAnyBox)
{
    const float inf = INFINITY;
    for (double L : {0.0, 1e-300, 1e-9, 1.0, 1e18, 1e30, 1e40, 1e300})
        for (float r : {0.0f, 1e-45f, 1e-18f, 2.4e-10f, 1.0f, 1e18f, 3e38f, inf})
            for (double flat : {0.0, 1.0}) {
                StageBox B;
                B.X0 = B.Y0 = B.Z0 = -L;
                B.X1 = B.Y1 = L;
                B.Z1 = flat * L - (1.0 - flat) * L;
                const bool ok = stage_size(B, r, 512);
                if (ok) EXPECT_TRUE(B.nx * B.ny * B.nz <= 512 && B.nx > 0 && B.ny > 0 && B.nz > 0);
                // Where radius and box are of comparable size it succeeds.
                if (r >= 1e-18f && r <= 1e18f && L < 1e12 * r) EXPECT_TRUE(ok);
            }
}

TEST(Keys, OrderIsThatOfTheDistances)
{
    // key_above and key_below bound the distances left out after a cut, at
    // every scale the search takes and below FLT_MIN.
    std::mt19937_64 rng(9);
    std::uniform_real_distribution<double> e(-330.0, std::log10(3.3e37)), u(1.0, 1.0 + 1e-3);
    for (int t = 0; t < 200000; ++t) {
        const double a = std::pow(10.0, e(rng));
        const double b = t % 3 ? a * u(rng) : std::pow(10.0, e(rng));
        const uint32_t ka = list_key(a, 1023u), kb = list_key(b, 0u);
        EXPECT_TRUE(std::isfinite(key_value(ka & ~kSlotMask)));
        if (b >= key_above(ka)) EXPECT_TRUE(kb > ka);
        if (kb >= ka) EXPECT_TRUE(b >= key_below(ka));
        EXPECT_TRUE(a < key_above(ka) || a <= 0.0);
    }
}

TEST(Keys, RowsTakenHaveFiniteDistances)
{
    // The largest coordinate difference of a row the search takes: queries a
    // kStageFar apart on either side of the origin, and the box's growth.
    const double reach = kStageFar * (1.0 - 1e-9), margin = reach * 0.2499;
    EXPECT_TRUE(stage_takes(reach, margin));
    EXPECT_TRUE(stage_takes_point(-kStageFar * (1.0 - 1e-9), 0.0, 0.0));
    const double d = 2.0 * kStageFar + reach + 3e-7 * 4.0 * kStageFar + margin;
    EXPECT_TRUE(std::isfinite(static_cast<float>(3.0 * d * d)));
    // Spacings whose squares leave FP32's range are refused: the first cells
    // of clouds 1e20 and 1e40 across, and coordinates that far out.
    EXPECT_TRUE(!stage_takes(8.0 * 3e19, 1e5));
    EXPECT_TRUE(!stage_takes(8.0 * 3e39, 1e25));
    EXPECT_TRUE(!stage_takes_point(0.0, 1e18, 0.0));
    EXPECT_TRUE(!stage_takes_point(0.0, 0.0, -INFINITY));
    EXPECT_TRUE(!stage_takes_point(NAN, 0.0, 0.0));
    EXPECT_TRUE(!stage_takes(1.0, 0.25));
}

int main(int argc, char** argv) { return mini::run_all(argc, argv); }
