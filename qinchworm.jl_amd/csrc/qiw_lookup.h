// qiw_lookup.h -- device lookups of grid-stored propagators and hybridization functions, and
// the times of a launch, shared by the evaluator kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

#include "qiw_device.h"

// ---------------------------------------------------------------------------------------
// Propagator lookups
// ---------------------------------------------------------------------------------------
// A grid-stored function of the time difference (the bold i*P table, a grid-stored i*Delta)
// at two contour times t1 >= t2, as Keldysh.jl's interpolate! evaluates a grid container
// (kd.interpolate! on expansion.P, src/topology_eval.jl:368; the call of an ImaginaryTimeGF
// pair propagator, :414): bilinear over the grid cell (i1, i2) holding (t1, t2), with the
// stored G[i1, i2] = g(i1 - i2), and linear in t1 - t2 inside a diagonal cell (i1 == i2).
// With a, b the fractions of t1, t2 in their grid intervals and d = i1 - i2 >= 0 both are
//     g(d) + a (1 - b) (g(d+1) - g(d)) - (1 - a) b (g(d) - g(d-1)),   g(-1) = 2 g(0) - g(1),
// i.e. row d plus wp times the forward and minus wm times the backward difference.
struct GridCell {
    int d;
    double wp, wm;  // a (1 - b), (1 - a) b
};
__device__ __forceinline__ GridCell grid_cell(double t1, double t2, double inv_h, int n_tau) {
    t1 = t1 > t2 ? t1 : t2;  // ordering clamp (src/topology_eval.jl:362-365, :408-411)
    const double x1 = t1 * inv_h, x2 = t2 * inv_h;
    int i1 = (int)floor(x1), i2 = (int)floor(x2);
    i1 = i1 < 0 ? 0 : (i1 > n_tau - 2 ? n_tau - 2 : i1);
    i2 = i2 < 0 ? 0 : (i2 > n_tau - 2 ? n_tau - 2 : i2);
    const double a = x1 - (double)i1, b = x2 - (double)i2;
    return GridCell{i1 - i2, a * (1.0 - b), (1.0 - a) * b};
}
// Value at cell c from g(d - 1) (any finite value when d = 0), g(d) and g(d + 1).
__device__ __forceinline__ double cell_value(const GridCell &c, double gm, double g0, double gp) {
    const double dm = c.d > 0 ? g0 - gm : gp - g0;
    return g0 + c.wp * (gp - g0) - c.wm * dm;
}

// Hybridization tables (QiwDeltaTables): per arc, the spline interval j and fraction u of
// the time difference, and the grid cell; a table is evaluated by its kind (grid_mask).
struct ArcPos {
    int j;
    double u;
    double z;  // the time difference itself (DLR tables)
    GridCell c;
};
__device__ __forceinline__ ArcPos arc_pos(double t_tail, double t_head, double inv_h, int n_tau) {
    ArcPos p;
    double z = t_tail - t_head;
    z = z > 0.0 ? z : 0.0;
    const double x = z * inv_h;
    int j = (int)floor(x);
    j = j < 0 ? 0 : (j > n_tau - 2 ? n_tau - 2 : j);
    p.j = j;
    p.u = x - (double)j;
    p.z = z;
    p.c = grid_cell(t_tail, t_head, inv_h, n_tau);
    return p;
}

// The fermionic kernel of the DLR, e^{-w tau} / (1 + e^{-w beta}) for 0 <= tau <= beta, in
// the form whose exponents are never positive.
__device__ __forceinline__ double dlr_kernel(double tau, double w, double beta) {
    return w >= 0.0 ? exp(-w * tau) / (1.0 + exp(-w * beta)) : exp(w * (beta - tau)) / (1.0 + exp(w * beta));
}
// i*Delta of table tab at arc position p: a natural cubic spline in the time difference
// (SplineInterpolatedGF, src/spline_gf.jl:194-219), coefficients (c0..c3) per interval, a
// grid container, (g(d), g(d+1) - g(d), g(d) - g(d-1), 0) per index d, or a DLR pole sum
// (keldysh_dlr.DLRImaginaryTimeGF, src/keldysh_dlr.jl:172-176).
// DLR = false leaves out the pole sums (a launch with no DLR table: fewer registers).
template <bool DLR = true>
__device__ __forceinline__ double delta_value(const QiwDeltaTables &dt, int tab, const ArcPos &p) {
    if (DLR && ((dt.dlr_mask >> tab) & 1)) {
        const double *c = dt.dlr + (int64_t)tab * dt.dlr_rank * 2;
        double s = 0.0;
        for (int k = 0; k < dt.dlr_rank; ++k) s = fma(c[2 * k + 1], dlr_kernel(p.z, c[2 * k], dt.beta), s);
        return s;
    }
    if ((dt.grid_mask >> tab) & 1) {
        const double *c = dt.coef + ((int64_t)tab * (dt.n_tau - 1) + p.c.d) * 4;
        return c[0] + p.c.wp * c[1] - p.c.wm * c[2];
    }
    const double *c = dt.coef + ((int64_t)tab * (dt.n_tau - 1) + p.j) * 4;
    return c[0] + p.u * (c[1] + p.u * (c[2] + p.u * c[3]));
}

// The fixed times of a group in a launch: tau_i = 0, tau_w, tau_f.
struct StepTimes {
    double tau_w, tau_f;
};
__device__ __forceinline__ StepTimes step_times(const EvalArgs &a, const QiwGroup &g, int tau_index) {
    StepTimes t;
    if (g.kind == QIW_G_BARE) {
        t.tau_w = 0.0;
        t.tau_f = a.h;
    } else if (g.kind == QIW_G_BOLD) {
        t.tau_w = a.step_w * a.h;
        t.tau_f = (a.step_w + 1) * a.h;
    } else if (g.kind == QIW_G_SIGMA) {  // tau_f_prev = grid[step_w]
        t.tau_w = a.step_w * a.h;
        t.tau_f = t.tau_w;
    } else {
        t.tau_w = tau_index * a.h;
        t.tau_f = a.beta;
    }
    return t;
}
