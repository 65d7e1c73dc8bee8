// knots_harness.cpp -- C entry points over the table code's knots (test
// infrastructure; host code only).
#include "tables.hpp"
extern "C" {
// coefficient rows [nr][4] of a spline over the knot values y, and its FP32
// knots [nr][2] for a derivative times scale; 0 where the rows are not the
// knots' Hermite cubics
int emu_slope_knots(const double* y, int nr, double scale, double* rows, float* knots)
{
    for (int m = 0; m < nr; ++m) rows[4 * m] = y[m];
    mapp::spline_coefficients(nr, rows, 4);
    std::vector<double> ys;
    if (!mapp::hermite_knots(rows, nr, ys)) return 0;
    mapp::slope_knots(ys, nr, scale, knots);
    return 1;
}
}
