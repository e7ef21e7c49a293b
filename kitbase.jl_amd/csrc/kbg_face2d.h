// kbg_face2d.h -- device helpers shared by the fused 2D step kernels (kbg_step2d.hip, kbg_tile2d.hip).
#pragma once

#include "kbg_device.h"
#include "kbg_types.h"

namespace kbg {

// FP64 slope of the conserved variables of cell c along dir (k_recon2d's sw)
KBG_D void wslope(const Solve2D& S, const double* w, int c, int dir, double* sw) {
    const int nx = S.nx, ny = S.ny;
    const int p = dir == 0 ? c % nx + 1 : c / nx + 1;
    const int n = dir == 0 ? nx : ny;
    const int step = dir == 0 ? 1 : nx;
    const double* d = dir == 0 ? S.dx : S.dy;
    if (!S.interp2) {
        for (int m = 0; m < 4; m++) sw[m] = 0.0;
    } else if (p == 1 || p == n) {
        const int a = p == 1 ? c : c - step, e = p == 1 ? c + step : c;
        const double D = 0.5 * (d[a] + d[e]);
        for (int m = 0; m < 4; m++) sw[m] = (w[(size_t)e * 4 + m] - w[(size_t)a * 4 + m]) / D;
    } else {
        const int a = c - step, e = c + step;
        const double dL = 0.5 * (d[a] + d[c]), dR = 0.5 * (d[c] + d[e]);
        for (int m = 0; m < 4; m++)
            sw[m] = limiter<double>(S.limiter, (w[(size_t)c * 4 + m] - w[(size_t)a * 4 + m]) / dL,
                                    (w[(size_t)e * 4 + m] - w[(size_t)c * 4 + m]) / dR);
    }
}

// index of the solve that owns global item g, from the prefix array start[0..n] (start[0] = 0)
KBG_D int owner(const int* start, int n, int g) {
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (g >= start[mid]) lo = mid;
        else hi = mid;
    }
    return lo;
}

// XCD-aware order: the workgroups of one XCD (ids congruent mod 8) take a contiguous run of items,
// so neighbouring faces and cells are read through the same L2
KBG_D int xcd_order() {
    const int G = gridDim.x, bx = blockIdx.x;
    const int x8 = bx & 7, q8 = G >> 3, r8 = G & 7;
    return x8 * q8 + (x8 < r8 ? x8 : r8) + (bx >> 3);
}

}  // namespace kbg
