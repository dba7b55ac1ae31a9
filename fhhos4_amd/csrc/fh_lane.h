// Wavefront-level dense factorisations shared by the cell kernels: a matrix
// row (or a right-hand side) per lane in registers, broadcasts instead of
// barriers.
#pragma once
#include <hip/hip_runtime.h>

namespace fh {
namespace {

typedef double lane_d4 __attribute__((ext_vector_type(4)));

// Wavefront-uniform broadcast of lane l's value.
__device__ __forceinline__ double bcast(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}

// Orders one wavefront's LDS accesses: its lanes run in lockstep and the LDS
// serves its requests in order, so only the compiler has to be kept from
// moving accesses across this point.
__device__ __forceinline__ void lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Pins a value at this place of the program: the unrolled factorisations and
// solves are computed step by step (else every load of a factor is moved
// before the first use, which spills).
__device__ __forceinline__ void pin(double& x) { asm volatile("" : "+v"(x)); }

// acc += sum over k < KD of a(k) b(k) for one 16 x 16 tile: a(k) is the
// lane's entry (k, lane % 16) of the left operand (transposed), b(k) its
// entry of the right one, k = 4 s + lane / 16; result element v of a lane is
// entry (lane / 16 + 4 v, lane % 16).
template <int KD, class FA, class FB>
__device__ __forceinline__ lane_d4 tile(lane_d4 acc, FA a, FB b) {
    const int kl = (threadIdx.x & 63) >> 4;
    constexpr int ST = (KD + 3) / 4;
#pragma unroll 8
    for (int s = 0; s < ST; s++) {
        const int k = 4 * s + kl;
        const bool ok = KD % 4 == 0 || k < KD;
        const int kk = ok ? k : 0;
        const double av = a(kk), bv = b(kk);
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(ok ? av : 0.0, ok ? bv : 0.0, acc, 0, 0, 0);
    }
    return acc;
}

// a / b with r = 1 / b correctly rounded, shared by the quotients of one
// divisor: P. Markstein's method (IBM J. Res. Dev. 34, 1990).  a r is corrected
// once to within a unit in the last place; correcting such a quotient by r
// times its residual rounds it correctly while the residual a - b q is exact.
// For the divisors met here (square roots, half-widths of cells: 2^-537 to
// 2^512) that is from |a| = 2^-960 on; below, the quotient is within one unit,
// and a zero is +0.  An infinite divisor, an infinite or NaN numerator and a
// quotient that overflows give NaN: kernels on matrices of the caller's look for
// NaN in their result and then start over with divisions (quotient<true>).
__device__ __forceinline__ double div_by(double a, double b, double r) {
    double q = a * r;
    q = fma(fma(-b, q, a), r, q);
    return fma(fma(-b, q, a), r, q);
}

template <bool DIVIDE>
__device__ __forceinline__ double quotient(double a, double b, double r) {
    return DIVIDE ? a / b : div_by(a, b, r);
}

// Cholesky factor of an N x N matrix held as row r = lane - base in a[0..r]
// of lanes base .. base + N - 1 (GROUPS: base differs by lane group, then the
// broadcast is a shuffle), in place.  Products are subtracted in ascending
// order and divided by the diagonal, as a column-by-column factorisation
// does.  Returns whether a pivot of this lane's matrix was not positive (the
// factorisation then goes on with 1 in its place).
template <int N, bool GROUPS, bool DIVIDE = false>
__device__ __forceinline__ bool lane_chol(double (&a)[N], int base, int r) {
    bool bad = false;
#pragma unroll
    for (int j = 0; j < N; j++) {
        double dj = GROUPS ? __shfl(a[j], base + j, 64) : bcast(a[j], j);
        if (!(dj > 0)) {
            bad = true;
            dj = 1.0;
        }
        const double sj = sqrt(dj), l = quotient<DIVIDE>(a[j], sj, 1.0 / sj);
        a[j] = r == j ? sj : l;
#pragma unroll
        for (int k = j + 1; k < N; k++) {
            const double lk = GROUPS ? __shfl(l, base + k, 64) : bcast(l, k);
            a[k] = fma(-l, lk, a[k]);
        }
#pragma unroll
        for (int k = j + 1; k < N; k++) pin(a[k]);
    }
    return bad;
}

// x <- L^-1 x, then x <- L^-T x, for a right-hand side per lane; l(i, j) is
// entry (i, j) of L, the diagonal included.
template <int N, class FL>
__device__ __forceinline__ void lane_solve(double (&x)[N], FL l) {
    double c[N];  // column (row of L^T) of the next step, loaded during this one
#pragma unroll
    for (int i = 0; i < N; i++) c[i] = l(i, 0);
#pragma unroll
    for (int j = 0; j < N; j++) {
        double n[N];
#pragma unroll
        for (int i = j + 1; i < N; i++) n[i] = l(i, j + 1 < N ? j + 1 : j);
        x[j] = x[j] / c[j];
#pragma unroll
        for (int i = j + 1; i < N; i++) x[i] = fma(-c[i], x[j], x[i]);
#pragma unroll
        for (int i = j + 1; i < N; i++) {
            pin(x[i]);
            c[i] = n[i];
        }
    }
    // row i of L^T below the diagonal, summed in ascending order
    c[N - 1] = l(N - 1, N - 1);
#pragma unroll
    for (int i = N - 1; i >= 0; i--) {
        double n[N];
#pragma unroll
        for (int k = i > 0 ? i - 1 : 0; k < N; k++) n[k] = l(k, i > 0 ? i - 1 : 0);
        double s = x[i];
#pragma unroll
        for (int k = i + 1; k < N; k++) s = fma(-c[k], x[k], s);
        x[i] = s / c[i];
        pin(x[i]);
#pragma unroll
        for (int k = i > 0 ? i - 1 : 0; k < N; k++) c[k] = n[k];
    }
}

// x <- L^-T x for one right-hand side spread over the lanes (lane i: x_i, the
// diagonal d of L and its reciprocal rd); l(j, i) is entry (j, i) of L.
template <int N, bool DIVIDE, class FL>
__device__ __forceinline__ double wave_backward(double x, double d, double rd, FL l) {
    const int i = threadIdx.x & 63;
    for (int j = N - 1; j >= 0; j--) {
        const double xj = quotient<DIVIDE>(bcast(x, j), bcast(d, j), bcast(rd, j));
        if (i == j) x = xj;
        else if (i < j) x = fma(-l(j, i), xj, x);
    }
    return x;
}

}  // namespace
}  // namespace fh
