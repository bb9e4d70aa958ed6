// shake.h -- the constraint sweeps of LFIntegrator::shake
// (src/integrators/LFIntegrator.cpp:1499-1540) for one rigid 3-site molecule.
//
// The sweeps are Gauss-Seidel over the cyclic constraints (0,1), (1,2), (2,0)
// and take about 32 rounds for water at a 1e-8 tolerance, each constraint
// waiting for the one before: a serial chain that nothing else in the kernel
// hides.  Every move of constraint b is f o_b (o_b the old bond vector) on its
// two sites, so the bond vectors n_c, which the sweeps only read through
// |n_c|^2 and o_j . n_c, change by M_cb f o_b with constant M.  The sweeps
// therefore run on those twelve scalars instead of nine coordinates: per
// constraint the chain is one product, one or two FMAs, the quotient and a
// select, about a third of the dependent operations of differences, dot
// products and an IEEE division.  The quotients are those of the coordinate
// form to rounding (the same factors, in the same order, with the same stop),
// and the positions take one rounding instead of one per move: 1,021 waters, a
// step against the same sweeps in 80 bits, 6e-17 nm rms, 3.4e-16 for the
// coordinate sweeps.
// Measured on 4,096 waters: 31 sweeps take 7.6 us (0.25 us each); with the
// loads issued ahead of the chain and wave_store's transposed sums,
// k_shake_kinetics takes 17.4 us against 29.7 us for the coordinate sweeps,
// and the sheared replicas' k_shake (73,689 molecules) 36 us against 53 us.
#pragma once

#include "smd_internal.h"

namespace smd {

// q = n / d to about an ulp: hardware reciprocal, two Newton steps, then the
// quotient corrected by its residual.  d > 0 and normal; the sweeps drop the
// quotients of any other.
__device__ __forceinline__ double quotient(double n, double d) {
    double r = __builtin_amdgcn_rcp(d);
    r = fma(fma(-d, r, 1.0), r, r);
    r = fma(fma(-d, r, 1.0), r, r);
    const double q = n * r;
    return fma(fma(-d, q, n), r, q);
}

// od: old bond vectors o_b = r_b - r_b+1 (cyclic); n0: the unconstrained new
// ones; mr: inverse masses; bl: squared lengths.  On return rn, the
// unconstrained new positions, are the constrained ones and wv[b] holds the
// sum over b's moves of f n_b, so the constraint virial is sum_b wv[b] (x) o_b.
__device__ __forceinline__ void shake_sweeps(const double (&od)[3][3], const double (&n0)[3][3],
                                             const double (&mr)[3], const double (&bl)[3], double tol, int max_count,
                                             double (&rn)[3][3], double (&wv)[3][3], bool& done, bool& failed) {
    double g[3][3], len2[3], oo[3][3], M[3][3], hm[3], lam[3] = {0.0, 0.0, 0.0}, W[3][3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        len2[c] = n0[c][0] * n0[c][0] + n0[c][1] * n0[c][1] + n0[c][2] * n0[c][2];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            g[c][j] = od[j][0] * n0[c][0] + od[j][1] * n0[c][1] + od[j][2] * n0[c][2];
            oo[c][j] = od[j][0] * od[c][0] + od[j][1] * od[c][1] + od[j][2] * od[c][2];
            W[c][j] = 0.0;
        }
    }
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        const int nx = (b + 1) % 3, pv = (b + 2) % 3;
        M[b][b] = mr[b] + mr[nx];
        M[nx][b] = -mr[nx];
        M[pv][b] = -mr[b];
        hm[b] = 2.0 * M[b][b];
    }
    const double tol_2 = 2.0 * tol;
    int count = 0;
    done = failed = false;
    while (!done && count < max_count && !failed) {
        done = true;
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            const double diff = bl[b] - len2[b];
            const double rno = g[b][b];
            const bool act = fabs(diff) > bl[b] * tol_2;
            failed = failed || (act && rno < bl[b] * tol);
            const double q = quotient(diff, rno * hm[b]);
            // a failed molecule moves no further: its positions stay finite
            const double f = act && !failed ? q : 0.0;
            done = done && !act;
#pragma unroll
            for (int j = 0; j < 3; ++j) W[b][j] = fma(f, lam[j], W[b][j]);
            lam[b] += f;
            // the next constraint's scalars first: they are the chain
#pragma unroll
            for (int s = 1; s <= 3; ++s) {
                const int c = (b + s) % 3;
                const double t = M[c][b] * f;
                len2[c] = fma(t, fma(t, oo[b][b], 2.0 * g[c][b]), len2[c]);
#pragma unroll
                for (int u = 0; u < 3; ++u) {
                    const int j = (c + u) % 3;
                    g[c][j] = fma(t, oo[b][j], g[c][j]);
                }
            }
        }
        count++;
    }
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        const int pv = (b + 2) % 3;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            rn[b][d] += mr[b] * (lam[b] * od[b][d] - lam[pv] * od[pv][d]);
            wv[b][d] = lam[b] * n0[b][d] + M[b][0] * W[b][0] * od[0][d] + M[b][1] * W[b][1] * od[1][d] +
                       M[b][2] * W[b][2] * od[2][d];
        }
    }
}

}  // namespace smd
