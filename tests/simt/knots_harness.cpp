// knots_harness.cpp -- C entry points over the table code's knots and the
// device helpers that read them, as the CPU SIMT emulation compiles them (test
// infrastructure).
#include "tables.hpp"
#include "kern.hpp"
extern "C" {
// values at offset p[k] of the cubics with end values and slopes (y0, s0, y1, s1)[k]
void emu_hermite(int n, const double* knots, const double* p, double* out)
{
    for (int k = 0; k < n; ++k) {
        const double* c = knots + 4 * k;
        out[k] = mapp::hermite_eval(c[0], c[1], c[2], c[3], mapp::hermite_basis<double>(p[k]));
    }
}
// the root of x[k] and its inverse
void emu_root_inv(int n, const double* x, double* r, double* r_inv)
{
    for (int k = 0; k < n; ++k) mapp::root_inv(x[k], r[k], r_inv[k]);
}
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
