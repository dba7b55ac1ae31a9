// Device functions shared by the HHO assembly kernels (affine and general
// cells): the exact solutions and their sources, and the position of an
// entry of a cell matrix in the element layout.
#pragma once
#include "fh_hho_dev.h"

namespace fh {
namespace {

// position of entry (r, s) of a cell matrix of n unknowns stored by cyclic
// diagonals (diagonal t = (s - r) mod n, position r; diagonal 0 first, then
// diagonals 2p + 1 and 2p + 2 interleaved), or -1 when the entry is stored
// as its transpose (t > n / 2)
__device__ __forceinline__ int elem_entry(int n, int r, int s) {
    const int t = s >= r ? s - r : s - r + n;
    if (t > n / 2) return -1;
    return t == 0 ? r : n + 2 * n * ((t - 1) / 2) + 2 * r + (t - 1) % 2;
}

__device__ inline double source_at(const HhoDev& d, double x, double y, double z) {
    const double X[3] = {x, y, z};
    if (d.src == 2) {
        double f = 0;
        for (int m = 0; m < d.nmodes; m++) {
            const double* md = d.modes + 4 * m;
            double s = 1, k2 = 0;
            for (int a = 0; a < d.dim; a++) {
                s *= sin(md[1 + a] * M_PI * X[a]);
                k2 += md[1 + a] * md[1 + a];
            }
            f += md[0] * M_PI * M_PI * k2 * s;
        }
        return f;
    }
    const double w = d.src == 1 ? 4 * M_PI : M_PI;
    double s = 1;
    for (int a = 0; a < d.dim; a++) s *= sin(w * X[a]);
    return d.dim * w * w * s;
}

// Exact solution of the source (its Laplacian is -source_at).
__device__ inline double exact_at(const HhoDev& d, double x, double y, double z) {
    const double X[3] = {x, y, z};
    if (d.src == 2) {
        double u = 0;
        for (int m = 0; m < d.nmodes; m++) {
            const double* md = d.modes + 4 * m;
            double s = 1;
            for (int a = 0; a < d.dim; a++) s *= sin(md[1 + a] * M_PI * X[a]);
            u += md[0] * s;
        }
        return u;
    }
    const double w = d.src == 1 ? 4 * M_PI : M_PI;
    double s = 1;
    for (int a = 0; a < d.dim; a++) s *= sin(w * X[a]);
    return s;
}

}  // namespace
}  // namespace fh
