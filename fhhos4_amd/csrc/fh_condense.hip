// Batched static condensation of caller-supplied HHO element matrices and the
// recovery of the cell unknowns, on gfx950.
//
// Input per cell: the local matrix of the element (cell unknowns first, then
// its faces in element order; Diff_HHOElement::A, Diff_HHOElement.h:144,
// FirstDOFNumber :522-525) and the system number of each face (-1 for a
// face whose unknowns are eliminated, a Dirichlet face).  The face system is
//   A = sum over cells of (A_FF - A_TF^T A_TT^-1 A_TF),
//   b = B_F - sum over cells of A_TF^T A_TT^-1 B_T,
// the reference's A = A_ndF_ndF - A_T_ndF^T Solve_A_T_T(A_T_ndF) and
// CondensedRHS (Diffusion_HHO.h:624-637, :1026-1032) cell by cell, and the
// cell unknowns are x_T = A_TT^-1 (B_T - A_TF x_F) (SolveCellUnknowns,
// Diffusion_HHO.h:960-966).
//
// Cells of the usual shapes (nc cell unknowns of a polynomial degree 0..3 in
// 2-D or 3-D, at most 63 face unknowns) take one wavefront each, four cells to
// a workgroup, without a barrier: lane r holds row r of A_TT and lane c column
// c of [A_TF B_T] in registers, one pass over the columns factors A_TT = L L^T
// and forms L^-1 [A_TF B_T] with the same broadcasts, L^-T follows, and
// A_FF - A_TF^T X runs on v_mfma_f64_16x16x4f64 from the X left in LDS.  The
// input is read from memory once, row by row (the bound: the nl^2 values of a
// cell read and its blocks written).  The factor and the solves subtract their
// products one by one in ascending order (the recovery's last solve in
// descending order); A_TF^T X is summed first and then subtracted from A_FF.  A
// cell whose quotients leave the range of div_by (an infinite diagonal entry)
// is computed a second time with divisions.
// Other shapes take a workgroup per cell with the matrices in LDS.
//
// The block pattern is formed on the device for conforming meshes (a face in
// at most two cells, cells of at most 8 faces), else on the host.  A block
// with one contribution (every off-diagonal one of a conforming mesh) is
// stored; one with more is cleared and added to with FP64 atomics: at most two
// contributions on a conforming mesh, so the sums do not depend on the order
// of the additions.  The right-hand side is formed without atomics: every cell
// stores its A_TF^T A_TT^-1 B_T, and every face adds those of its cells in
// cell order.
//
// MI355X, hexahedra at k = 3 (nc = 20, 60 face unknowns), 13 824 cells, the
// condensation and the recovery of all cells: 0.74 ms, of which the cells'
// condensation 287 us and the recovery 80 us.  Bound by memory: 110 592 cells
// take 2.34 ms for 7.4 GB (3.2 TB/s), and the counters show 11.3 GB (4.9 TB/s):
// A_TF is read three times and does not stay in the caches; its registers
// leave three wavefronts per SIMD to cover the loads.  A workgroup per cell with a barrier per column and the
// pattern formed on the host by sorting took 6.2 ms.
#include <algorithm>
#include <cstdlib>
#include <type_traits>
#include <vector>

#include "fh_condense.h"
#include "fh_lane.h"

namespace fh {
namespace {

constexpr int kCondWG = 256;
constexpr int kCondWaves = kCondWG / 64;
constexpr int kPatFaces = 8;  // faces per cell of the device-built pattern

struct CondDev {
    int ncells, nfc, nc, nf, nl, m;
    const int* faces;     // ncells x nfc system face numbers, -1: eliminated
    // ncells x nfc x nfc: block of (face j1, face j2), -1: none; a block p with
    // more than one contribution is coded -2 - p (its values start at zero)
    const int* slot;
    const double* local;  // ncells x nl x nl
    const double* BT;     // ncells x nc, or null (zero)
    double* vals;         // block values (nf x nf row-major per block)
    double* cstage;       // ncells x m: A_TF^T A_TT^-1 B_T
    int* err;             // bit 0: an A_TT is not positive definite
};

// Entry o of the block coded s (not -1) takes the contribution v.
__device__ __forceinline__ void add_entry(double* vals, int s, int bsz, int o, double v) {
    if (s >= 0) vals[(int64_t)s * bsz + o] = v;
    else atomicAdd(vals + (int64_t)(-2 - s) * bsz + o, v);
}

// In-place lower Cholesky factor of the nc x nc matrix L (row-major, LDS).
// Returns false (the same on every thread) if a pivot is not positive.
__device__ bool chol_lds(double* L, int nc) {
    for (int j = 0; j < nc; j++) {
        __syncthreads();
        const double piv = L[j * nc + j];
        if (!(piv > 0.0)) return false;  // uniform: every thread read the same pivot
        const double d = sqrt(piv);
        __syncthreads();
        for (int r = j + 1 + (int)threadIdx.x; r < nc; r += blockDim.x) L[r * nc + j] /= d;
        if (threadIdx.x == 0) L[j * nc + j] = d;
        __syncthreads();
        const int w = nc - j - 1;  // trailing block, lower triangle
        for (int t = threadIdx.x; t < w * w; t += blockDim.x) {
            const int r = j + 1 + t / w, q = j + 1 + t % w;
            if (q <= r) L[r * nc + q] -= L[r * nc + j] * L[q * nc + j];
        }
    }
    __syncthreads();
    return true;
}

// Solves L L^T y = y for column col of the nc x ld array Y (row-major).
__device__ void chol_solve_col(const double* L, int nc, double* Y, int ld, int col) {
    for (int r = 0; r < nc; r++) {
        double s = Y[r * ld + col];
        for (int q = 0; q < r; q++) s -= L[r * nc + q] * Y[q * ld + col];
        Y[r * ld + col] = s / L[r * nc + r];
    }
    for (int r = nc - 1; r >= 0; r--) {
        double s = Y[r * ld + col];
        for (int q = r + 1; q < nc; q++) s -= L[q * nc + r] * Y[q * ld + col];
        Y[r * ld + col] = s / L[r * nc + r];
    }
}

// Schur entries A_FF - A_TF^T X of a workgroup's cell on the matrix cores: 16 x
// 16 output tiles dealt to the wavefronts, four cell unknowns per instruction
// (zero beyond nc and m).  T: A_TF (nc x m), X: nc x (m + 1), in LDS.
__device__ void schur_tiles(const CondDev& a, const double* T, const double* X, const double* loc, const int* slot) {
    const int nc = a.nc, m = a.m, nl = a.nl, nf = a.nf, nfc = a.nfc;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane >> 4, lc = lane & 15, tiles = (m + 15) / 16;
    for (int t = wave; t < tiles * tiles; t += kCondWaves) {
        const int ti = t / tiles, tj = t - ti * tiles, pa = 16 * ti + lc, q = 16 * tj + lc;
        lane_d4 acc = {0.0, 0.0, 0.0, 0.0};
        for (int k0 = 0; k0 < nc; k0 += 4) {
            const int k = k0 + lr;
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(k < nc && pa < m ? T[k * m + pa] : 0.0,
                                                       k < nc && q < m ? X[k * (m + 1) + q] : 0.0, acc, 0, 0, 0);
        }
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int p = 16 * ti + lr + 4 * v;
            if (p >= m || q >= m) continue;
            const int s = slot[(p / nf) * nfc + q / nf];
            if (s == -1) continue;
            add_entry(a.vals, s, nf * nf, (p % nf) * nf + q % nf, loc[(int64_t)(nc + p) * nl + nc + q] - acc[v]);
        }
    }
}

// Other shapes: a workgroup per cell, the matrices in LDS (nc^2 + nc m +
// nc (m + 1) doubles), the factorisation column by column with barriers, the
// triangular solves a column per thread, the Schur blocks by tiles (MFMA) or
// entry by entry.
template <bool MFMA>
__global__ __launch_bounds__(kCondWG) void k_condense(CondDev a) {
    extern __shared__ double lds[];
    const int nc = a.nc, m = a.m, nl = a.nl, nf = a.nf, nfc = a.nfc;
    const int cell = blockIdx.x;
    double* L = lds;
    double* T = L + nc * nc;  // A_TF, nc x m
    double* X = T + nc * m;   // A_TT^-1 [A_TF B_T], nc x (m + 1)
    const double* loc = a.local + (int64_t)cell * nl * nl;
    for (int t = threadIdx.x; t < nc * nc; t += blockDim.x) L[t] = loc[(int64_t)(t / nc) * nl + t % nc];
    for (int t = threadIdx.x; t < nc * m; t += blockDim.x) {
        const int r = t / m, q = t - r * m;
        const double v = loc[(int64_t)r * nl + nc + q];
        T[t] = v;
        X[r * (m + 1) + q] = v;
    }
    for (int r = threadIdx.x; r < nc; r += blockDim.x) X[r * (m + 1) + m] = a.BT ? a.BT[(int64_t)cell * nc + r] : 0.0;
    if (!chol_lds(L, nc)) {
        if (threadIdx.x == 0) atomicOr(a.err, 1);
        return;  // the whole workgroup leaves together
    }
    for (int col = threadIdx.x; col <= m; col += blockDim.x) chol_solve_col(L, nc, X, m + 1, col);
    __syncthreads();
    // Schur entries (p, q) of the cell's faces j1 = p / nf, j2 = q / nf
    const int* slot = a.slot + (int64_t)cell * nfc * nfc;
    if constexpr (MFMA) {
        schur_tiles(a, T, X, loc, slot);
    } else {
        for (int t = threadIdx.x; t < m * m; t += blockDim.x) {
            const int p = t / m, q = t - p * m;
            const int s = slot[(p / nf) * nfc + q / nf];
            if (s == -1) continue;
            double v = loc[(int64_t)(nc + p) * nl + nc + q];
            for (int r = 0; r < nc; r++) v -= T[r * m + p] * X[r * (m + 1) + q];
            add_entry(a.vals, s, nf * nf, (p % nf) * nf + q % nf, v);
        }
    }
    if (a.cstage) {
        for (int p = threadIdx.x; p < m; p += blockDim.x) {
            double v = 0;
            for (int r = 0; r < nc; r++) v += T[r * m + p] * X[r * (m + 1) + m];
            a.cstage[(int64_t)cell * m + p] = v;
        }
    }
}

// b_f = B_F[f] - sum over the cells of face f (cell order) of their stored
// A_TF^T A_TT^-1 B_T entries; thread per face unknown.  The cells of face f
// are entries fptr[f] .. fptr[f + 1] - 1 of fent, or, with counts cnt, the
// first cnt[f] of fent[2 f], fent[2 f + 1].
__global__ void k_condense_rhs(int nfaces, int nf, const int* fptr, const int* cnt, const int* fent,
                               const double* cstage, const double* BF, double* b) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)nfaces * nf) return;
    const int f = (int)(t / nf), i = (int)(t - (int64_t)f * nf);
    double v = BF ? BF[t] : 0.0;
    const int e0 = cnt ? 2 * f : fptr[f], e1 = cnt ? 2 * f + cnt[f] : fptr[f + 1];
    for (int e = e0; e < e1; e++) {
        const int cj = fent[e];  // cell * (faces per cell) + local face
        v -= cstage[(int64_t)cj * nf + i];
    }
    b[t] = v;
}

__global__ __launch_bounds__(kCondWG) void k_cell_recover(CondDev a, const double* xF, double* xT) {
    extern __shared__ double lds[];
    const int nc = a.nc, m = a.m, nl = a.nl, nf = a.nf;
    const int cell = blockIdx.x;
    double* L = lds;
    double* y = L + nc * nc;
    const double* loc = a.local + (int64_t)cell * nl * nl;
    const int* faces = a.faces + (int64_t)cell * a.nfc;
    for (int t = threadIdx.x; t < nc * nc; t += blockDim.x) L[t] = loc[(int64_t)(t / nc) * nl + t % nc];
    for (int r = threadIdx.x; r < nc; r += blockDim.x) {
        double v = a.BT ? a.BT[(int64_t)cell * nc + r] : 0.0;
        for (int p = 0; p < m; p++) {
            const int f = faces[p / nf];
            if (f >= 0) v -= loc[(int64_t)r * nl + nc + p] * xF[(int64_t)f * nf + p % nf];
        }
        y[r] = v;
    }
    if (!chol_lds(L, nc)) {
        if (threadIdx.x == 0) atomicOr(a.err, 1);
        return;
    }
    if (threadIdx.x == 0) chol_solve_col(L, nc, y, 1, 0);
    __syncthreads();
    for (int r = threadIdx.x; r < nc; r += blockDim.x) xT[(int64_t)cell * nc + r] = y[r];
}

// ---- one wavefront per cell ----------------------------------------------
// p / nf for p < 64
__device__ __forceinline__ int div_nf(int p, int rcp) { return (p * rcp) >> 16; }

// x = column c of A_TT^-1 [A_TF B_T] of a cell (lane c; column m: B_T).
// Returns whether A_TT is not positive definite or, without DIVIDE, whether a
// quotient may have left the range of div_by: such a quotient is NaN, and a NaN
// in a row of the factor or of x reaches x[0] or a pivot.
template <int NC, bool DIVIDE>
__device__ __forceinline__ bool condense_columns(const CondDev& a, const double* loc, int cell, int lane,
                                                 double (&x)[NC]) {
    const int m = a.m, nl = a.nl;
    double A[NC];
    {
        const double* row = loc + (int64_t)min(lane, NC - 1) * nl;
#pragma unroll
        for (int k = 0; k < NC; k++) A[k] = row[k];
#pragma unroll
        for (int i = 0; i < NC; i++) {
            x[i] = 0.0;
            if (lane < m) x[i] = loc[(int64_t)i * nl + NC + lane];
            else if (lane == m && a.BT) x[i] = a.BT[(int64_t)cell * NC + i];
        }
    }
    // A_TT = L L^T and L^-1 [A_TF B_T] with the same broadcasts; then L^-T,
    // products in ascending order.  Lane j keeps diagonal entry j and, in rd,
    // its reciprocal.
    bool bad = false;
    double rd = 1.0;
#pragma unroll
    for (int j = 0; j < NC; j++) {
        double dj = bcast(A[j], j);
        if (!(dj > 0.0)) {
            bad = true;  // wavefront-uniform
            dj = 1.0;
        }
        const double sj = sqrt(dj), rj = 1.0 / sj, l = quotient<DIVIDE>(A[j], sj, rj);
        x[j] = quotient<DIVIDE>(x[j], sj, rj);
        A[j] = lane == j ? sj : l;
        rd = lane == j ? rj : rd;
#pragma unroll
        for (int k = j + 1; k < NC; k++) {
            const double lk = bcast(l, k);
            A[k] = fma(-l, lk, A[k]);
            x[k] = fma(-lk, x[j], x[k]);
        }
#pragma unroll
        for (int k = j + 1; k < NC; k++) {
            pin(A[k]);
            pin(x[k]);
        }
    }
    if (bad) return true;
#pragma unroll
    for (int i = NC - 1; i >= 0; i--) {
        double s = x[i];
#pragma unroll
        for (int k = i + 1; k < NC; k++) s = fma(-bcast(A[i], k), x[k], s);
        x[i] = quotient<DIVIDE>(s, bcast(A[i], i), bcast(rd, i));
        pin(x[i]);
    }
    return !DIVIDE && __any(x[0] != x[0]);
}

// The condensation of a cell of NC cell unknowns and m <= 63 face unknowns
// (nfc <= 8 faces): lane r holds row r of A_TT, lane c column c of
// [A_TF B_T] (column m: B_T).  rcp = ceil(65536 / nf); ldx: row length of X
// in LDS, a multiple of 16 above m.
template <int NC>
__global__ __launch_bounds__(kCondWG, 3) void k_condense_wave(CondDev a, int rcp, int ldx) {
    extern __shared__ double lds[];
    const int m = a.m, nl = a.nl, nf = a.nf, nfc = a.nfc;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cell = blockIdx.x * kCondWaves + wave;
    if (cell >= a.ncells) return;  // wavefront-uniform; no barrier follows
    const double* loc = a.local + (int64_t)cell * nl * nl;
    const int sl = lane < nfc * nfc ? a.slot[(int64_t)cell * nfc * nfc + lane] : -1;
    double x[NC];
    if (condense_columns<NC, false>(a, loc, cell, lane, x) && condense_columns<NC, true>(a, loc, cell, lane, x)) {
        if (lane == 0) atomicOr(a.err, 1);
        return;
    }
    if (a.cstage) {
        double v = 0;
#pragma unroll
        for (int i = 0; i < NC; i++) v = fma(lane < m ? loc[(int64_t)i * nl + NC + lane] : 0.0, bcast(x[i], m), v);
        if (lane < m) a.cstage[(int64_t)cell * m + lane] = v;
    }
    double* X = lds + wave * NC * ldx;
    if (lane < ldx)
#pragma unroll
        for (int i = 0; i < NC; i++) X[i * ldx + lane] = x[i];
    lds_order();
    // A_FF - A_TF^T X by 16 x 16 tiles, A_TF read again; columns of
    // eliminated faces and beyond m reach entries that are not stored only
    const int lr = lane >> 4, lc = lane & 15, T = (m + 15) >> 4;
    constexpr int ST = (NC + 3) / 4;
    for (int ti = 0; ti < T; ti++) {
        double pa[ST];
#pragma unroll
        for (int s = 0; s < ST; s++) {
            const int k = 4 * s + lr;
            pa[s] = k < NC && 16 * ti + lc < m ? loc[(int64_t)k * nl + NC + 16 * ti + lc] : 0.0;
        }
        for (int tj = 0; tj < T; tj++) {
            const int q = 16 * tj + lc, fq = div_nf(q, rcp);
            double aff[4];
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int p = 16 * ti + lr + 4 * v;
                aff[v] = p < m && q < m ? loc[(int64_t)(NC + p) * nl + NC + q] : 0.0;
            }
            lane_d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int s = 0; s < ST; s++) {
                const int k = 4 * s + lr;
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(pa[s], k < NC ? X[k * ldx + q] : 0.0, acc, 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int p = 16 * ti + lr + 4 * v, fp = div_nf(p, rcp);
                const bool in = p < m && q < m;
                const int s = __shfl(sl, in ? fp * nfc + fq : 0, 64);
                if (in && s != -1) add_entry(a.vals, s, nf * nf, (p - fp * nf) * nf + q - fq * nf, aff[v] - acc[v]);
            }
        }
    }
}

// r <- A_TT^-1 r, r spread over the lanes; A: row `lane` of A_TT, P: NC^2
// entries of the wavefront's LDS.  Returns as condense_columns does.
template <int NC, bool DIVIDE>
__device__ __forceinline__ bool recover_solve(double (&A)[NC], int lane, double& r, double* P) {
    if (lane_chol<NC, false, DIVIDE>(A, 0, lane)) return true;
    // L^-1 r with the lane's own row of L, then L^-T with its column
    double d = 1.0;
#pragma unroll
    for (int j = 0; j < NC; j++)
        if (lane == j) d = A[j];
    const double rd = 1.0 / d;
#pragma unroll
    for (int j = 0; j < NC; j++) {
        const double yj = quotient<DIVIDE>(bcast(r, j), bcast(d, j), bcast(rd, j));
        if (lane == j) r = yj;
        else if (lane > j) r -= A[j] * yj;
    }
    if (lane < NC)
#pragma unroll
        for (int k = 0; k < NC; k++)
            if (k <= lane) P[lane * NC + k] = A[k];
    lds_order();
    r = wave_backward<NC, DIVIDE>(r, d, rd, [&](int i, int j) { return P[i * NC + j]; });
    return !DIVIDE && __any(lane < NC && r != r);
}

// Cell unknowns of a cell of NC cell unknowns and m <= 64 face unknowns:
// lane r holds row r of A_TT, lane p the face unknown p.
template <int NC>
__global__ __launch_bounds__(kCondWG) void k_recover_wave(CondDev a, int rcp, const double* xF, double* xT) {
    constexpr int kRow = 33;  // rows in different banks
    __shared__ double part[kCondWaves][NC * kRow + 64];
    const int m = a.m, nl = a.nl, nf = a.nf, nfc = a.nfc;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cell = blockIdx.x * kCondWaves + wave;
    if (cell >= a.ncells) return;  // wavefront-uniform; no barrier follows
    const double* loc = a.local + (int64_t)cell * nl * nl;
    const int fj = div_nf(min(lane, m - 1), rcp);
    const int f = lane < m ? a.faces[(int64_t)cell * nfc + fj] : -1;
    double A[NC], t[NC];
    {
        const double* row = loc + (int64_t)min(lane, NC - 1) * nl;
#pragma unroll
        for (int k = 0; k < NC; k++) A[k] = row[k];
#pragma unroll
        for (int i = 0; i < NC; i++) t[i] = f >= 0 ? loc[(int64_t)i * nl + NC + lane] : 0.0;
    }
    const double xf = f >= 0 ? xF[(int64_t)f * nf + lane - fj * nf] : 0.0;
    double r = lane < NC && a.BT ? a.BT[(int64_t)cell * NC + lane] : 0.0;
    double* P = part[wave];
    // row i of A_TF x_F by lane i, its products subtracted in ascending order;
    // half of the columns in LDS at a time (five workgroups fit a CU)
    P[NC * kRow + lane] = xf;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        if (lane >> 5 == h)
#pragma unroll
            for (int i = 0; i < NC; i++) P[i * kRow + (lane & 31)] = t[i];
        lds_order();
        const double *ti = P + min(lane, NC - 1) * kRow, *xp = P + NC * kRow + 32 * h;
        const int n = min(m - 32 * h, 32);
#pragma unroll 8
        for (int q = 0; q < n; q++) r = fma(-ti[q], xp[q], r);
        lds_order();
    }
    const double rhs = r;
    if (recover_solve<NC, false>(A, lane, r, P)) {
        // a quotient out of range: again with divisions
        const double* row = loc + (int64_t)min(lane, NC - 1) * nl;
#pragma unroll
        for (int k = 0; k < NC; k++) A[k] = row[k];
        r = rhs;
        lds_order();
        if (recover_solve<NC, true>(A, lane, r, P)) {
            if (lane == 0) atomicOr(a.err, 1);
            return;
        }
    }
    if (lane < NC) xT[(int64_t)cell * NC + lane] = r;
}

// ---- block pattern of a conforming mesh -----------------------------------
// (cell, local face) entries of every face: the first two in ent (ascending
// after k_pat_rows), their number in cnt; *flag is set if a face has more.
__global__ void k_pat_count(int n, const int* __restrict__ faces, int* __restrict__ cnt, int* __restrict__ ent,
                            int* __restrict__ flag) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int f = faces[t];
    if (f < 0) return;
    const int pos = atomicAdd(cnt + f, 1);
    if (pos < 2) ent[2 * (int64_t)f + pos] = t;
    else *flag = 1;
}

// Row f of the pattern: the distinct faces of its cells, ascending.  FILL
// false: their number into rlen (and the entries of the face in order); true:
// the columns, whether a block has several contributions, and the block of
// every face pair of the cells.
template <bool FILL>
__global__ void k_pat_rows(int nfaces, int nfc, const int* __restrict__ faces, const int* __restrict__ cnt,
                           int* __restrict__ ent, int* __restrict__ rlen, const int* __restrict__ rowptr,
                           int* __restrict__ colidx, unsigned char* __restrict__ multi, int* __restrict__ slot) {
    constexpr int W = 2 * kPatFaces;
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nfaces) return;
    const int n = min(cnt[f], 2);
    int e0 = n > 0 ? ent[2 * (int64_t)f] : -1, e1 = n > 1 ? ent[2 * (int64_t)f + 1] : -1;
    if (n > 1 && e0 > e1) {
        const int q = e0;
        e0 = e1;
        e1 = q;
    }
    if (!FILL && n > 1) {
        ent[2 * (int64_t)f] = e0;
        ent[2 * (int64_t)f + 1] = e1;
    }
    int g[W];
#pragma unroll
    for (int i = 0; i < W; i++) {
        const int e = i < kPatFaces ? e0 : e1, j = i % kPatFaces;
        g[i] = e >= 0 && j < nfc ? faces[(int64_t)(e / nfc) * nfc + j] : -1;
    }
    bool first[W];
    int len = 0;
#pragma unroll
    for (int i = 0; i < W; i++) {
        first[i] = g[i] >= 0;
#pragma unroll
        for (int k = 0; k < i; k++) first[i] = first[i] && g[k] != g[i];
        len += first[i];
    }
    if constexpr (!FILL) {
        rlen[f] = len;
    } else {
        const int base = rowptr[f];
#pragma unroll
        for (int i = 0; i < W; i++) {
            const int e = i < kPatFaces ? e0 : e1, j = i % kPatFaces;
            if (e < 0 || j >= nfc) continue;
            int code = -1;
            if (g[i] >= 0) {
                int rank = 0, times = 0;
#pragma unroll
                for (int k = 0; k < W; k++) {
                    rank += first[k] && g[k] < g[i];
                    times += g[k] == g[i];
                }
                const int p = base + rank;
                code = times > 1 ? -2 - p : p;
                if (first[i]) {
                    colidx[p] = g[i];
                    multi[p] = times > 1;
                }
            }
            slot[(int64_t)e * nfc + j] = code;
        }
    }
}

// out[0 .. n] = exclusive sums of in[0 .. n - 1]; one workgroup of 1024.
__global__ __launch_bounds__(1024) void k_scan(int n, const int* __restrict__ in, int* __restrict__ out) {
    __shared__ int wsum[16];
    __shared__ int carry;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    if (t == 0) carry = 0;
    __syncthreads();
    for (int base = 0; base < n; base += 4096) {
        int v[4], s = 0;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = base + 4 * t + u;
            v[u] = i < n ? in[i] : 0;
            s += v[u];
        }
        int inc = s;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int q = __shfl_up(inc, o, 64);
            if (lane >= o) inc += q;
        }
        if (lane == 63) wsum[w] = inc;
        __syncthreads();
        int off = carry;
        for (int k = 0; k < w; k++) off += wsum[k];
        int run = off + inc - s;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = base + 4 * t + u;
            if (i < n) out[i] = run;
            run += v[u];
        }
        __syncthreads();
        if (t == 1023) carry = run;
        __syncthreads();
    }
    if (t == 0) out[n] = carry;
}

// Clears the blocks with several contributions: 64 blocks per wavefront.
__global__ __launch_bounds__(kCondWG) void k_zero_multi(int64_t nnzb, int bsz, const unsigned char* __restrict__ multi,
                                                        double* __restrict__ vals) {
    const int lane = threadIdx.x & 63;
    const int64_t b0 = ((int64_t)blockIdx.x * kCondWaves + (threadIdx.x >> 6)) * 64;
    if (b0 >= nnzb) return;  // wavefront-uniform
    unsigned long long todo = __ballot(b0 + lane < nnzb && multi[min(b0 + lane, nnzb - 1)] != 0);
    while (todo) {
        const int i = __ffsll((long long)todo) - 1;
        todo &= todo - 1;
        for (int e = lane; e < bsz; e += 64) vals[(b0 + i) * bsz + e] = 0.0;
    }
}

// FHGPU_MFMA=0 keeps the Schur product on the vector ALUs.
bool mfma_enabled() {
    static const bool on = [] {
        const char* e = std::getenv("FHGPU_MFMA");
        return e ? std::atoi(e) != 0 : true;
    }();
    return on;
}

size_t cond_lds_bytes(int nc, int m) { return sizeof(double) * ((size_t)nc * nc + (size_t)nc * m + (size_t)nc * (m + 1)); }

void set_lds(const void* kernel, size_t bytes) {
    int dev = 0, maxb = 0;
    FH_HIP(hipGetDevice(&dev));
    FH_HIP(hipDeviceGetAttribute(&maxb, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    FH_CHECK(bytes <= (size_t)maxb, -3, "cell matrices do not fit the LDS of one workgroup");
    FH_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
}

void check_args(int ncells, int nfc, int nc, int nf, int nfaces, const int* cell_faces) {
    FH_CHECK(ncells > 0 && nfc > 0 && nc > 0 && nf > 0 && nfaces > 0, -2, "sizes must be positive");
    FH_CHECK(cell_faces != nullptr, -2, "null cell face array");
    const int64_t nl = nc + (int64_t)nfc * nf;
    FH_CHECK(nl * nl * ncells < ((int64_t)1 << 62), -2, "local matrices too large");
    for (int64_t t = 0; t < (int64_t)ncells * nfc; t++)
        FH_CHECK(cell_faces[t] >= -1 && cell_faces[t] < nfaces, -2, "cell face number out of range");
}

}  // namespace

// Shapes of one wavefront per cell: a compiled number of cell unknowns, the
// face unknowns and B_T in its 64 lanes.  FHGPU_MFMA=0 keeps the general
// kernel (vector ALUs only).
static bool wave_shape(int nc, int m, int nfc) {
    return mfma_enabled() && (nc == 1 || nc == 3 || nc == 4 || nc == 6 || nc == 10 || nc == 20) && m <= 63 &&
           nfc <= kPatFaces;
}

template <class F>
static void with_nc(int nc, F&& f) {
    switch (nc) {
        case 1: f(std::integral_constant<int, 1>()); break;
        case 3: f(std::integral_constant<int, 3>()); break;
        case 4: f(std::integral_constant<int, 4>()); break;
        case 6: f(std::integral_constant<int, 6>()); break;
        case 10: f(std::integral_constant<int, 10>()); break;
        default: f(std::integral_constant<int, 20>()); break;
    }
}

static void launch_condense(Ctx& c, const CondDev& d) {
    if (wave_shape(d.nc, d.m, d.nfc)) {
        const int ldx = (d.m + 16) / 16 * 16;  // above m, at most 64
        const size_t lds = sizeof(double) * kCondWaves * d.nc * ldx;
        with_nc(d.nc, [&](auto N) {
            hipLaunchKernelGGL(k_condense_wave<decltype(N)::value>, dim3((d.ncells + kCondWaves - 1) / kCondWaves),
                               dim3(kCondWG), lds, c.stream, d, (65536 + d.nf - 1) / d.nf, ldx);
        });
    } else {
        // on the matrix cores where the blocks fill 2 x 2 tiles and two steps of
        // four cell unknowns: 4096 cells of nc = 35, m = 90 take 1193 us (1347 us
        // entry by entry), of nc = 20, m = 80 348 us (414 us)
        const size_t lds = cond_lds_bytes(d.nc, d.m);
        auto kern = d.m >= 32 && d.nc >= 8 && mfma_enabled() ? k_condense<true> : k_condense<false>;
        set_lds((const void*)kern, lds);
        hipLaunchKernelGGL(kern, dim3(d.ncells), dim3(kCondWG), lds, c.stream, d);
    }
    FH_HIP(hipGetLastError());
}

namespace {

// The block pattern on the host: any cells, any number of cells per face.
struct HostPattern {
    std::vector<int> slot, fptr, fent;
    std::vector<unsigned char> multi;
};

// Face by face from the (cell, local face) entries of every face: one sorted
// list at a time, in place of a list per face (4096 cells of 12 faces: 6.9 ms a
// call with those and a separate search for every block).
void host_pattern(int ncells, int nfc, int nfaces, const int* cell_faces, Bcsr& A, HostPattern& H) {
    const int64_t nent = (int64_t)ncells * nfc;
    // entries of every face, in cell order
    std::vector<int64_t> ptr((size_t)nfaces + 1, 0);
    for (int64_t t = 0; t < nent; t++)
        if (cell_faces[t] >= 0) ptr[cell_faces[t] + 1]++;
    for (int f = 0; f < nfaces; f++) ptr[f + 1] += ptr[f];
    std::vector<int64_t> ent(ptr[nfaces]), fill(ptr.begin(), ptr.end() - 1);
    for (int64_t t = 0; t < nent; t++)
        if (cell_faces[t] >= 0) ent[fill[cell_faces[t]]++] = t;
    A.h_rowptr.assign((size_t)nfaces + 1, 0);
    A.h_colidx.clear();
    H.multi.clear();
    H.slot.assign((size_t)nent * nfc, -1);
    std::vector<int> row;
    for (int f = 0; f < nfaces; f++) {
        // the distinct faces of the cells of f, ascending
        row.clear();
        for (int64_t e = ptr[f]; e < ptr[f + 1]; e++)
            for (int j = 0; j < nfc; j++) {
                const int g = cell_faces[ent[e] / nfc * nfc + j];
                if (g >= 0) row.push_back(g);
            }
        std::sort(row.begin(), row.end());
        const size_t base = A.h_colidx.size();
        for (size_t i = 0; i < row.size(); i++) {
            if (i > 0 && row[i] == row[i - 1]) {
                H.multi.back() = 1;
            } else {
                A.h_colidx.push_back(row[i]);
                H.multi.push_back(0);
            }
        }
        FH_CHECK(A.h_colidx.size() < (size_t)INT32_MAX, -2, "too many blocks");
        A.h_rowptr[f + 1] = (int)A.h_colidx.size();
        // block of every face pair (f, g) of the cells
        const auto b0 = A.h_colidx.begin() + base;
        for (int64_t e = ptr[f]; e < ptr[f + 1]; e++)
            for (int j = 0; j < nfc; j++) {
                const int g = cell_faces[ent[e] / nfc * nfc + j];
                if (g < 0) continue;
                const int p = (int)(std::lower_bound(b0, A.h_colidx.end(), g) - A.h_colidx.begin());
                H.slot[(size_t)ent[e] * nfc + j] = H.multi[p] ? -2 - p : p;
            }
    }
    A.nnzb = A.h_rowptr[nfaces];
    A.h_colidx.resize(std::max<int64_t>(1, A.nnzb));
    H.fptr.assign(ptr.begin(), ptr.end());
    H.fent.assign(ent.begin(), ent.end());
    H.fent.resize(std::max<size_t>(1, H.fent.size()));
}

}  // namespace

std::unique_ptr<Bcsr> condense_batched(Ctx& c, int ncells, int nfc, int nc, int nf, int nfaces,
                                       const int* cell_faces, const double* local, const double* BT,
                                       const double* BF, double* b_out) {
    FH_CHECK(!c.host_only, -9, "batched condensation needs a device context");
    check_args(ncells, nfc, nc, nf, nfaces, cell_faces);
    FH_CHECK(local != nullptr, -2, "null local matrices");
    const int m = nfc * nf, nl = nc + m;
    auto A = std::make_unique<Bcsr>();
    A->nbr = A->nbc = nfaces;
    A->bs_r = A->bs_c = nf;
    A->prec = Prec::F64;
    const int64_t nent = (int64_t)ncells * nfc;
    // one allocation for everything that the call alone needs
    size_t bytes = 0;
    auto part = [&](size_t b) {
        const size_t o = bytes;
        bytes += (b + 255) / 256 * 256;
        return o;
    };
    const size_t oflag = part(2 * sizeof(int)), ocnt = part(sizeof(int) * nfaces),
                 oent = part(sizeof(int) * 2 * (size_t)nfaces), olen = part(sizeof(int) * nfaces),
                 ofaces = part(sizeof(int) * nent), oslot = part(sizeof(int) * nent * nfc),
                 ostage = part(b_out ? sizeof(double) * (size_t)ncells * m : 0),
                 omulti = part((size_t)nent * nfc);
    DevBuf work;
    work.alloc_kept(bytes);
    char* w = work.as<char>();
    int* flag = (int*)(w + oflag);  // [0] an A_TT not positive definite, [1] a face of more than two cells
    int* cnt = (int*)(w + ocnt);
    int* ent = (int*)(w + oent);
    int* slot = (int*)(w + oslot);
    int* faces = (int*)(w + ofaces);
    double* stage = b_out ? (double*)(w + ostage) : nullptr;
    unsigned char* multi = (unsigned char*)(w + omulti);
    A->rowptr.alloc(sizeof(int) * ((size_t)nfaces + 1));
    bool on_device = nfc <= kPatFaces && nent < INT32_MAX && (int64_t)nfaces * 2 * nfc < INT32_MAX;
    const dim3 fgrid((nfaces + 255) / 256);
    FH_HIP(hipMemsetAsync(w, 0, oent, c.stream));  // flags and counts
    if (on_device) {
        FH_HIP(hipMemcpyAsync(faces, cell_faces, sizeof(int) * nent, hipMemcpyHostToDevice, c.stream));
        hipLaunchKernelGGL(k_pat_count, dim3((unsigned)((nent + 255) / 256)), dim3(256), 0, c.stream, (int)nent, faces,
                           cnt, ent, flag + 1);
        hipLaunchKernelGGL(k_pat_rows<false>, fgrid, dim3(256), 0, c.stream, nfaces, nfc, faces, cnt, ent,
                           (int*)(w + olen), nullptr, nullptr, nullptr, nullptr);
        hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, c.stream, nfaces, (int*)(w + olen), A->rowptr.as<int>());
        FH_HIP(hipGetLastError());
        A->h_rowptr.resize((size_t)nfaces + 1);
        int more = 0;
        FH_HIP(hipMemcpyAsync(&more, flag + 1, sizeof(int), hipMemcpyDeviceToHost, c.stream));
        FH_HIP(hipMemcpyAsync(A->h_rowptr.data(), A->rowptr.p, sizeof(int) * A->h_rowptr.size(), hipMemcpyDeviceToHost,
                              c.stream));
        c.sync();
        on_device = !more;
    }
    HostPattern H;
    DevBuf dptr, dent;  // host pattern: cells of every face
    if (on_device) {
        A->nnzb = A->h_rowptr[nfaces];
    } else {
        host_pattern(ncells, nfc, nfaces, cell_faces, *A, H);
        FH_HIP(hipMemcpyAsync(A->rowptr.p, A->h_rowptr.data(), sizeof(int) * A->h_rowptr.size(), hipMemcpyHostToDevice,
                              c.stream));
        FH_HIP(hipMemcpyAsync(slot, H.slot.data(), sizeof(int) * H.slot.size(), hipMemcpyHostToDevice, c.stream));
        FH_HIP(hipMemcpyAsync(multi, H.multi.data(), H.multi.size(), hipMemcpyHostToDevice, c.stream));
        if (b_out) {
            dptr.alloc(sizeof(int) * H.fptr.size());
            dent.alloc(sizeof(int) * H.fent.size());
            FH_HIP(hipMemcpyAsync(dptr.p, H.fptr.data(), sizeof(int) * H.fptr.size(), hipMemcpyHostToDevice, c.stream));
            FH_HIP(hipMemcpyAsync(dent.p, H.fent.data(), sizeof(int) * H.fent.size(), hipMemcpyHostToDevice, c.stream));
        }
    }
    A->colidx.alloc_kept(sizeof(int) * std::max<int64_t>(1, A->nnzb));
    A->vals.alloc_kept(sizeof(double) * std::max<int64_t>(1, A->nnzb * nf * nf));
    if (on_device) {
        // rows of eliminated faces have no block
        FH_HIP(hipMemsetAsync(slot, 0xff, sizeof(int) * nent * nfc, c.stream));
        hipLaunchKernelGGL(k_pat_rows<true>, fgrid, dim3(256), 0, c.stream, nfaces, nfc, faces, cnt, ent, nullptr,
                           A->rowptr.as<int>(), A->colidx.as<int>(), multi, slot);
        FH_HIP(hipGetLastError());
    } else {
        FH_HIP(hipMemcpyAsync(A->colidx.p, A->h_colidx.data(), sizeof(int) * A->h_colidx.size(), hipMemcpyHostToDevice,
                              c.stream));
    }
    if (A->nnzb > 0) {
        hipLaunchKernelGGL(k_zero_multi, dim3((unsigned)((A->nnzb + kCondWG - 1) / kCondWG)), dim3(kCondWG), 0,
                           c.stream, A->nnzb, nf * nf, multi, A->vals.as<double>());
        FH_HIP(hipGetLastError());
    }
    launch_condense(c, CondDev{ncells, nfc, nc, nf, nl, m, nullptr, slot, local, BT, A->vals.as<double>(), stage, flag});
    if (b_out) {
        const int64_t n = (int64_t)nfaces * nf;
        hipLaunchKernelGGL(k_condense_rhs, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c.stream, nfaces, nf,
                           dptr.as<int>(), on_device ? cnt : nullptr, on_device ? ent : dent.as<int>(), stage, BF,
                           b_out);
        FH_HIP(hipGetLastError());
    }
    if (on_device) {
        A->h_colidx.resize(std::max<int64_t>(1, A->nnzb));
        FH_HIP(hipMemcpyAsync(A->h_colidx.data(), A->colidx.p, sizeof(int) * A->nnzb, hipMemcpyDeviceToHost, c.stream));
    }
    int err = 0;
    FH_HIP(hipMemcpyAsync(&err, flag, sizeof(int), hipMemcpyDeviceToHost, c.stream));
    c.sync();  // the work buffer is freed on return
    FH_CHECK(err == 0, -4, "a cell matrix A_TT is not positive definite");
    return A;
}

void cell_recover_batched(Ctx& c, int ncells, int nfc, int nc, int nf, int nfaces, const int* cell_faces,
                          const double* local, const double* BT, const double* xF, double* xT) {
    FH_CHECK(!c.host_only, -9, "cell recovery needs a device context");
    check_args(ncells, nfc, nc, nf, nfaces, cell_faces);
    FH_CHECK(local && xF && xT, -2, "null local matrices or vectors");
    const int m = nfc * nf, nl = nc + m;
    const size_t nent = (size_t)ncells * nfc;
    DevBuf work;  // face numbers, error flag
    work.alloc_kept(sizeof(int) * (nent + 1));
    int* faces = work.as<int>();
    int* flag = faces + nent;
    FH_HIP(hipMemcpyAsync(faces, cell_faces, sizeof(int) * nent, hipMemcpyHostToDevice, c.stream));
    FH_HIP(hipMemsetAsync(flag, 0, sizeof(int), c.stream));
    CondDev d{ncells, nfc, nc, nf, nl, m, faces, nullptr, local, BT, nullptr, nullptr, flag};
    if (wave_shape(nc, m, nfc)) {
        with_nc(nc, [&](auto N) {
            hipLaunchKernelGGL(k_recover_wave<decltype(N)::value>, dim3((ncells + kCondWaves - 1) / kCondWaves),
                               dim3(kCondWG), 0, c.stream, d, (65536 + nf - 1) / nf, xF, xT);
        });
    } else {
        const size_t lds = sizeof(double) * ((size_t)nc * nc + nc);
        set_lds((const void*)k_cell_recover, lds);
        hipLaunchKernelGGL(k_cell_recover, dim3(ncells), dim3(kCondWG), lds, c.stream, d, xF, xT);
    }
    FH_HIP(hipGetLastError());
    int err = 0;
    FH_HIP(hipMemcpyAsync(&err, flag, sizeof(int), hipMemcpyDeviceToHost, c.stream));
    c.sync();
    FH_CHECK(err == 0, -4, "a cell matrix A_TT is not positive definite");
}

}  // namespace fh
