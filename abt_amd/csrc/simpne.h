// simpne.h -- quadrature on uneven nodes.
//
// The reference's simpne (misc_submod.f90:2392-2531): 3-point Lagrange panels over x[m-1], x[m], x[m+1] for
// m = 1, 3, 5, ..., plus, for an even node count, the integral of the last three points' parabola over the
// final interval.  The result is linear in y; simpne_weights gives the weights w with
// simpne(y) = sum_i w_i y_i, which fold the phi and theta integrals into per-bin weights.
#pragma once
namespace abt {

// The quadrature weights of the nodes x (n >= 3), panel by panel, each in the reference's operations up to
// the factor y.
inline void simpne_weights(int n, const double* x, double* w)
{
#pragma clang fp contract(off)
    for (int i = 0; i < n; i++) w[i] = 0.0;
    const auto panel = [&](int m, double lo, double hi) {   // the parabola through x[m-1..m+1] over [lo, hi]
#pragma clang fp contract(off)
        const double x1 = x[m - 1], x2 = x[m], x3 = x[m + 1];
        const double e = hi * hi - lo * lo, f = hi * hi * hi - lo * lo * lo, fe = hi - lo;
        const double del[3] = {x3 - x2, x1 - x3, x2 - x1};
        const double g[3] = {x2 + x3, x1 + x3, x1 + x2};
        const double p[3] = {x2 * x3, x1 * x3, x1 * x2};
        for (int i = 0; i < 3; i++)
            w[m - 1 + i] -= del[i] * (f / 3.0 - g[i] * 0.5 * e + p[i] * fe) / (del[0] * del[1] * del[2]);
    };
    for (int m = 1; m < n - 1; m += 2) panel(m, x[m - 1], x[m + 1]);
    if (n % 2 == 0) panel(n - 2, x[n - 2], x[n - 1]);
}

}  // namespace abt
