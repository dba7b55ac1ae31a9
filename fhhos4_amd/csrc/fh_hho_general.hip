// HHO local operators and static condensation of general cells (bilinear
// quadrilaterals, trilinear hexahedra) on gfx950: per-cell quadrature through
// the cell and face maps, saddle-point reconstruction with the mean-value
// condition, the general "hho" stabilisation with the face and cell L2
// projections, condensation and scatter (Diff_HHOElement.h:104-150, 312-509;
// Diffusion_HHO.h:624-652).
//
// One workgroup of NW wavefronts per cell, every size a compile-time constant
// of the dimension and the degree, 80 KB of LDS at k = 3 in 3-D (two cells per
// CU).  Inner products run on v_mfma_f64_16x16x4f64: 16 x 16 output tiles
// dealt to the wavefronts, operands from LDS with consecutive lanes on
// consecutive entries, 1/8 of a value read from LDS per multiply-add where a
// thread per output entry reads two.  Factorisations keep a matrix row per lane in
// registers and broadcast with v_readlane, triangular solves keep a
// right-hand side per lane; neither takes a barrier inside, and independent
// ones run on different wavefronts.
//
// The values are those of a thread per output entry that adds its products
// one after the other, bit for bit: the matrix instruction is a chain of
// fused multiply-adds over ascending k (measured), the factorisations and
// solves subtract in ascending order and divide by the pivots, and sums over
// quadrature points are taken slice by slice.  An operator does not change
// with the kernel that assembles it.  The one product whose terms are sums
// themselves (grad psi_i . K grad psi_j) stays on the vector ALUs, T x T
// entries per lane.
//
// MI355X, hexahedra at k = 3: 13 824 cells in 4.84 ms (0.35 us per cell; the
// products alone would take 0.1 us at the rate of a large FP64 matrix
// product).  Bound by latency: of 397 000 cycles per cell, with two cells in
// flight per CU, 33% go to the gradient products, 14% to the face integrals,
// 12% to the factorisation of S and the solves with it.  A workgroup of 256
// threads per cell with an entry per thread and a barrier per column took
// 48 ms (146 KB of LDS: one cell per CU).  k = 2: 1.11 ms for 12 167 cells.
#include "fh_hho_eval.h"
#include "fh_lane.h"

#include <algorithm>
#include <string>

namespace fh {
namespace {

template <int DIM, int K>
struct Gen {
    static constexpr int poly(int p) { return DIM == 3 ? (p + 1) * (p + 2) * (p + 3) / 6 : (p + 1) * (p + 2) / 2; }
    static constexpr int NC = poly(K), NR = poly(K + 1);  // cell and reconstruction functions
    static constexpr int NFB = DIM == 3 ? (K + 1) * (K + 2) / 2 : K + 1;
    static constexpr int M = 2 * DIM, NF = M * NFB, NH = NC + NF, N1 = NR - 1;
    static constexpr int NVC = 1 << DIM, NVF = DIM == 3 ? 4 : 2;
    static constexpr int Q1 = K + 2, QS = Q1 * Q1, NSL = DIM == 3 ? Q1 : 1, NQ = QS * NSL;  // cell rule, by slices
    static constexpr int QF = DIM == 3 ? QS : Q1;                                           // face rule
    static constexpr int SL = NSL < 2 ? NSL : 2;  // slices in LDS at a time
    // T x T entries of S per lane
    static constexpr int T = DIM == 3 ? (K == 3 ? 5 : (K == 2 ? 4 : (K == 1 ? 2 : 1))) : (K >= 2 ? 2 : 1);
    static constexpr int GT = (NR + T - 1) / T, LS = GT * GT;
    static constexpr int SPW = LS * SL <= 64 ? SL : 1;  // slices per wavefront
    static constexpr int WS = SL / SPW;                 // wavefronts that form S
    // tables per point and direction: Legendre values of degree 1..K+1, then
    // their derivatives
    static constexpr int TB = 2 * (K + 1);
    static constexpr int mx(int a, int b) { return a > b ? a : b; }
    // LDS, in doubles.  Kept: S (rows and columns 1.. of the stiffness), MT
    // (NC x NR), Mf, TF (traces, then projections), P (right-hand sides, then
    // the reconstruction; row 0 first).
    static constexpr int oMf = 0, oS = oMf + M * NFB * NFB, oMT = oS + N1 * N1, oTF = oMT + NC * NR,
                         oP = oTF + NF * NR, oT = oP + NR * NH;
    // cell integrals (before the rest exists)
    static constexpr int cG = 0, cPs = cG + SL * DIM * QS * NR, cPt = cPs + SL * QS * NR, cTab = cPt + 2 * SL * QS,
                         cEnd = cTab + SL * QS * DIM * TB;
    // face integrals; row 0 of P does not exist yet
    static constexpr int fPs = oT, fKg = fPs + QF * NR, fPhi = fKg + QF * NR, fTab = fPhi + QF * NFB,
                         fW = fTab + QF * DIM * TB, fFV = fW + 2 * QF, fSg = fFV + M * NVF * 3,
                         fKn0 = fSg + M;
    static constexpr bool kKnInP = QF * DIM <= NH;  // QF x DIM, over row 0 of P where it fits
    static constexpr int fKn = kKnInP ? oP : fKn0, fEnd = kKnInP ? fKn0 : fKn0 + QF * DIM;
    // algebra: factors (rows of N x N or N x (N + 1) / 2, diagonal as is), W
    static constexpr int tri(int n) { return n * (n + 1) / 2; }
    static constexpr int aLS = oT, aLF = aLS + tri(N1), aLEnd = aLF + M * tri(NFB);
    static constexpr int aW = oT, aWEnd = aW + N1 * NH;
    static constexpr int aN = oT, aNEnd = aN + NC * NH + tri(NC);  // D_T and the factor of M_T
    // DF (NF x NH) and MD of half of the faces replace everything but Mf
    static constexpr int bDF = oS, bMD = bDF + NF * NH, bEnd = bMD + NF / 2 * NH;
    // condensation: [A_TT A_TF], X, the condensed matrix
    static constexpr int xA = 0, xX = xA + NC * NH, xL = xX + NC * (NF + 1), xS = xL + tri(NC), xEnd = xS + NF * NF;
    static constexpr int mCV = mx(mx(mx(cEnd, fEnd), mx(aLEnd, aWEnd)), mx(mx(aNEnd, bEnd), xEnd));
    static constexpr int mCtr = mCV + NVC * 3, mHw = mCtr + 3, mK = mHw + 3, mCf = mK + 9, mLm = mCf + M,
                         mBT = mLm + NR, mG = mBT + NC, mOne = mG + 2 * Q1, mEx = mOne + 2, mBlk = mEx + (NR + 1) / 2,
                         mRed = mBlk + (M * M + M + 1) / 2, total = mRed;
    // post-processing mode: P is kept, and two vectors and the reduction
    static constexpr int pP = total, pW = pP + NR * NH, pC = pW + NH, pRed = pC + NR, total_post = pRed + 16;
};
static_assert(2 * Gen<3, 3>::total * sizeof(double) <= 163840, "two cells per CU at k = 3");
// Legendre polynomials of degree 1..P at s into t[0..P-1], their derivatives
// into t[P..2P-1].
template <int P>
__device__ __forceinline__ void legendre_table(double s, double* t) {
    double L[P + 1], D[P + 1];
    L[0] = 1;
    D[0] = 0;
    L[1] = s;
    D[1] = 1;
#pragma unroll
    for (int q = 2; q <= P; q++) {
        L[q] = ((2 * q - 1) * s * L[q - 1] - (q - 1) * L[q - 2]) / q;
        D[q] = D[q - 2] + (2 * q - 1) * L[q - 1];
    }
#pragma unroll
    for (int q = 1; q <= P; q++) {
        t[q - 1] = L[q];
        t[P + q - 1] = D[q];
    }
}

__device__ inline double legendre_at(int p, double s) {
    double a = 1, b = s;
    if (p == 0) return a;
    for (int q = 2; q <= p; q++) {
        const double c = ((2 * q - 1) * s * b - (q - 1) * a) / q;
        a = b;
        b = c;
    }
    return b;
}

// Where the table holds the value (or derivative) of degree e: entry e - 1 of
// every point's run, or the constant one (zero) of stride 0.
struct TabRef {
    const double* p;
    int stride;
    __device__ double at(int q) const { return p[q * stride]; }
};

__device__ __forceinline__ double norm3(double x, double y, double z) { return sqrt(fma(z, z, fma(x, x, y * y))); }

// Cell map at xi: x and det J (corners CV[2^DIM][3], corner code x + 2y + 4z).
template <int DIM>
__device__ inline double gen_cell_map(const double* CV, const double (&xi)[3], double (&x)[3]) {
    double J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
    x[0] = x[1] = x[2] = 0;
#pragma unroll
    for (int cc = 0; cc < (1 << DIM); cc++) {
        double f[3] = {1, 1, 1}, df[3] = {0, 0, 0};
#pragma unroll
        for (int a = 0; a < DIM; a++) {
            const double sg = ((cc >> a) & 1) ? 1.0 : -1.0;
            f[a] = 0.5 * (1 + sg * xi[a]);
            df[a] = 0.5 * sg;
        }
        const double N = f[0] * f[1] * f[2];
        const double dN[3] = {df[0] * f[1] * f[2], f[0] * df[1] * f[2], f[0] * f[1] * df[2]};
#pragma unroll
        for (int r = 0; r < 3; r++) {
            x[r] += N * CV[cc * 3 + r];
#pragma unroll
            for (int q = 0; q < DIM; q++) J[r][q] += dN[q] * CV[cc * 3 + r];
        }
    }
    if (DIM == 2) J[2][2] = 1;
    return J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) - J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
           J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
}

// Face map at (s, t): x and the (unoriented) vector area element (FV: the
// face's corners a, b, c, d, or a, b in 2-D).
template <int DIM>
__device__ inline void gen_face_map(const double* FV, double s, double t, double (&x)[3], double (&nv)[3]) {
    double xs[3], xt[3];
    if (DIM == 2) {
        for (int a = 0; a < 3; a++) {
            x[a] = 0.5 * (1 - s) * FV[a] + 0.5 * (1 + s) * FV[3 + a];
            xs[a] = 0.5 * (FV[3 + a] - FV[a]);
        }
        nv[0] = xs[1];
        nv[1] = -xs[0];
        nv[2] = 0;
        return;
    }
    for (int a = 0; a < 3; a++) {
        const double A = FV[a], B = FV[3 + a], C = FV[6 + a], D = FV[9 + a];
        x[a] = 0.25 * ((1 - s) * (1 - t) * A + (1 + s) * (1 - t) * B + (1 + s) * (1 + t) * C + (1 - s) * (1 + t) * D);
        xs[a] = 0.25 * ((1 - t) * (B - A) + (1 + t) * (C - D));
        xt[a] = 0.25 * ((1 - s) * (D - A) + (1 + s) * (C - B));
    }
    nv[0] = xs[1] * xt[2] - xs[2] * xt[1];
    nv[1] = xs[2] * xt[0] - xs[0] * xt[2];
    nv[2] = xs[0] * xt[1] - xs[1] * xt[0];
}

template <int DIM, int K, int NW, int MW>
__global__ __launch_bounds__(NW * 64, MW) void k_hho_general(HhoDev d, int* err) {
    using G = Gen<DIM, K>;
    constexpr int NT = NW * 64, TB = G::TB, P1 = K + 1;
    constexpr int NC = G::NC, NR = G::NR, NFB = G::NFB, M = G::M, NF = G::NF, NH = G::NH, N1 = G::N1;
    constexpr int QS = G::QS, QF = G::QF, NVF = G::NVF, SL = G::SL, T = G::T, GT = G::GT, LS = G::LS;
    static_assert(NR <= NT && NF < 64, "a thread per basis function, a lane per face unknown");
    extern __shared__ double sm[];
    const int c = blockIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // thread, lane and tile entries (lr + 4 v, lc) of this thread, renewed
    // for every phase: indexes kept from one phase for the next cost the
    // registers that the factorisations need
    int t = threadIdx.x, lane = t & 63, lr = lane >> 4, lc = lane & 15;
    auto phase = [&] {
        __syncthreads();
        t = threadIdx.x;
        asm volatile("" : "+v"(t));
        lane = t & 63;
        lr = lane >> 4;
        lc = lane & 15;
    };
    if (c >= d.ncell) return;  // whole workgroup
    double* CV = sm + G::mCV;
    double* FV = sm + G::fFV;
    double* Sg = sm + G::fSg;
    double* ctr = sm + G::mCtr;
    double* hw = sm + G::mHw;
    double* Kc = sm + G::mK;
    double* Cf = sm + G::mCf;
    double* Lm = sm + G::mLm;
    double* BT = sm + G::mBT;
    double* gx = sm + G::mG;
    double* gw = gx + G::Q1;
    double* one = sm + G::mOne;  // 1, 0
    int* EX = (int*)(sm + G::mEx);
    int* blk = (int*)(sm + G::mBlk);  // block indices, then rows, of the cell's faces
    const lane_d4 zero4{0.0, 0.0, 0.0, 0.0};

    // ---- cell geometry
    for (int e = t; e < G::NVC * 3; e += NT) CV[e] = d.V[3 * (size_t)d.cv[(size_t)c * G::NVC + e / 3] + e % 3];
    for (int e = t; e < 2 * G::Q1; e += NT) gx[e] = d.g1[e];
    for (int e = t; e < NR; e += NT) EX[e] = d.rexp[3 * e] | d.rexp[3 * e + 1] << 8 | d.rexp[3 * e + 2] << 16;
    for (int e = t; e < M * M; e += NT) blk[e] = d.blk[(size_t)c * M * M + e];
    for (int e = t; e < M; e += NT) blk[M * M + e] = d.frow[(size_t)c * M + e];
    if (t < 9) {
        Kc[t] = d.K[(size_t)c * 9 + t];
        if (t % 4 != 0 && Kc[t] != 0) atomicOr(err, 4);  // S takes the tensor's diagonal
    }
    if (t < 2) one[t] = 1.0 - t;
    phase();
    if (t < 3) {
        double lo = 1e300, hi = -1e300, s = 0;
        for (int l = 0; l < G::NVC; l++) {
            const double v = CV[l * 3 + t];
            s += v;
            lo = fmin(lo, v);
            hi = fmax(hi, v);
        }
        ctr[t] = s / G::NVC;
        hw[t] = t < DIM ? 0.5 * (hi - lo) : 1.0;
    }
    // basis function bi at the points bq, bq + NT / NR, ..: its entries of the
    // tables at tab
    const int bi = t % NR, bq = t < NT / NR * NR ? t / NR : QS * SL;
    auto refs = [&](const double* tab, TabRef (&L)[3], TabRef (&D)[3]) {
        const int ex = EX[bi];
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const int e = a < DIM ? (ex >> (8 * a)) & 255 : 0;
            L[a] = e > 0 ? TabRef{tab + a * TB + e - 1, DIM * TB} : TabRef{one, 0};
            D[a] = e > 0 ? TabRef{tab + a * TB + P1 + e - 1, DIM * TB} : TabRef{one + 1, 0};
        }
    };
    phase();

    // ---- cell integrals, SL slices of the rule at a time: S (its terms are
    // sums, so it stays on the vector ALUs: T x T entries per lane, a
    // wavefront or part of one per slice) and [MT; mean values; source] (tiles;
    // left operand the weighted functions, the weights and the weighted source)
    {
        double* Gp = sm + G::cG;   // gradients, (slice, point, direction) x function
        double* Ps = sm + G::cPs;  // functions, (slice, point) x function
        double* pt = sm + G::cPt;  // weight, weighted source of every point
        double* tab = sm + G::cTab;
        constexpr int TN = (NR + 15) / 16, TMR = (NC + 2 + 15) / 16, TC = TMR * TN;
        // wavefronts that form S change with the cell: two cells share a CU
        const int w0 = NW > 1 ? (wave + NW / 2 * (c & 1)) % NW : 0;
        constexpr int NM = NW > G::WS ? NW - G::WS : NW;  // wavefronts of the tiles
        const int wm = NW > G::WS ? w0 - G::WS : w0;
        constexpr int UC = (TC + NM - 1) / NM;
        lane_d4 tot[UC];
#pragma unroll
        for (int u = 0; u < UC; u++) tot[u] = zero4;
        const int se = lane % LS, ssl = G::SPW > 1 ? lane / LS : w0;
        const bool sact = w0 < G::WS && lane < LS * G::SPW;
        const int si = se / GT * T, sj = se % GT * T;
        double S[T][T];
#pragma unroll
        for (int i = 0; i < T; i++)
#pragma unroll
            for (int j = 0; j < T; j++) S[i][j] = 0;
        for (int s0 = 0; s0 < G::NSL; s0 += SL) {
            const int ns = min(SL, G::NSL - s0);
            for (int e = t; e < ns * QS * DIM; e += NT) {
                const int ql = e / DIM, a = e - ql * DIM, q = s0 * QS + ql;
                const int i0 = q % G::Q1, i1 = (q / G::Q1) % G::Q1, i2 = DIM == 3 ? q / QS : 0;
                const double xi[3] = {gx[i0], gx[i1], DIM == 3 ? gx[i2] : 0.0};
                double x[3];
                const double det = gen_cell_map<DIM>(CV, xi, x);
                const double xa = a == 0 ? x[0] : (a == 1 ? x[1] : x[2]);
                legendre_table<P1>((xa - ctr[a]) / hw[a], tab + e * TB);
                if (a == 0) {
                    const double w = gw[i0] * gw[i1] * (DIM == 3 ? gw[i2] : 1.0);
                    if (!(det > 0)) atomicOr(err, 2);
                    pt[2 * ql] = w * det;
                    pt[2 * ql + 1] = w * det * source_at(d, x[0], x[1], x[2]);
                }
            }
            phase();
            {
                TabRef L[3], D[3];
                refs(tab, L, D);
                const double r0 = 1.0 / hw[0], r1 = 1.0 / hw[1], r2 = 1.0 / hw[2];
#pragma unroll 2
                for (int q = bq; q < ns * QS; q += NT / NR) {
                    const double L0 = L[0].at(q), L1 = L[1].at(q), L2 = DIM == 3 ? L[2].at(q) : 1.0;
                    const double D0 = D[0].at(q), D1 = D[1].at(q), D2 = DIM == 3 ? D[2].at(q) : 0.0;
                    Ps[q * NR + bi] = L0 * L1 * L2;
                    Gp[(q * DIM) * NR + bi] = div_by(D0, hw[0], r0) * L1 * L2;
                    Gp[(q * DIM + 1) * NR + bi] = div_by(L0 * D1, hw[1], r1) * L2;
                    if (DIM == 3) Gp[(q * DIM + 2) * NR + bi] = div_by(L0 * L1 * D2, hw[2], r2);
                }
            }
            phase();
            if (sact && ssl < ns) {
                double s[T][T];
#pragma unroll
                for (int i = 0; i < T; i++)
#pragma unroll
                    for (int j = 0; j < T; j++) s[i][j] = 0;
                const double k0 = Kc[0], k1 = Kc[4], k2 = Kc[8];
#pragma unroll 1
                for (int q = ssl * QS; q < (ssl + 1) * QS; q++) {
                    const double* g = Gp + q * DIM * NR;
                    const double w = pt[2 * q];
                    double gj[T][3];
#pragma unroll
                    for (int j = 0; j < T; j++) {
                        const int jj = min(sj + j, NR - 1);
                        gj[j][0] = g[jj];
                        gj[j][1] = g[NR + jj];
                        gj[j][2] = DIM == 3 ? g[(DIM == 3 ? 2 : 0) * NR + jj] : 0.0;
                    }
#pragma unroll
                    for (int i = 0; i < T; i++) {
                        const int ii = min(si + i, NR - 1);
                        const double a0 = k0 * g[ii], a1 = k1 * g[NR + ii];
                        const double a2 = DIM == 3 ? k2 * g[(DIM == 3 ? 2 : 0) * NR + ii] : 0.0;
#pragma unroll
                        for (int j = 0; j < T; j++) {
                            double v = fma(a0, gj[j][0], a1 * gj[j][1]);
                            if (DIM == 3) v = fma(a2, gj[j][2], v);
                            s[i][j] = fma(w, v, s[i][j]);
                        }
                    }
                }
                // the second slice's sums go to the lanes of the first, which
                // add the slices in order
                if (ssl == 0) {
#pragma unroll
                    for (int i = 0; i < T; i++)
#pragma unroll
                        for (int j = 0; j < T; j++) S[i][j] += s[i][j];
                } else {
#pragma unroll
                    for (int i = 0; i < T; i++)
#pragma unroll
                        for (int j = 0; j < T; j++) S[i][j] = s[i][j];
                }
            }
            if (wm >= 0)
                for (int sl = 0; sl < ns; sl++) {
                    const double* Pq = Ps + sl * QS * NR;
                    const double* pq = pt + 2 * sl * QS;
#pragma unroll
                    for (int u = 0; u < UC; u++) {
                        const int tt = wm + u * NM;
                        if (tt >= TC) continue;
                        const int ti = tt / TN, tj = tt - ti * TN;
                        const int i = 16 * ti + lc, j = min(16 * tj + lc, NR - 1);
                        // rows i < NC: weight times function; NC: weight; NC + 1: source
                        const double* pa = i < NC ? Pq + i : one;
                        const double* pw = pq + (i == NC + 1 ? 1 : 0);
                        const int la = i < NC ? NR : 0;
                        const double* pb = Pq + j;
                        tot[u] += tile<QS>(zero4, [&](int k) { return pw[2 * k] * pa[k * la]; },
                                           [&](int k) { return pb[k * NR]; });
                    }
                }
            phase();
            if (ns > 1) {
                double* tmp = Gp;  // GT T x GT T
                if (sact && ssl == 1)
#pragma unroll
                    for (int i = 0; i < T; i++)
#pragma unroll
                        for (int j = 0; j < T; j++) tmp[(si + i) * (GT * T) + sj + j] = S[i][j];
                phase();
                if (sact && ssl == 0)
#pragma unroll
                    for (int i = 0; i < T; i++)
#pragma unroll
                        for (int j = 0; j < T; j++) S[i][j] += tmp[(si + i) * (GT * T) + sj + j];
                phase();
            }
        }
        double* So = sm + G::oS;
        double* MT = sm + G::oMT;
        double* P = sm + G::oP;
        if (sact && ssl == 0)
#pragma unroll
            for (int i = 0; i < T; i++)
#pragma unroll
                for (int j = 0; j < T; j++) {
                    const int r = si + i, s = sj + j;
                    if (r < 1 || r >= NR || s >= NR) continue;
                    if (s >= 1) So[(r - 1) * N1 + s - 1] = S[i][j];
                    if (s < NC) P[r * NH + s] = S[i][j];
                }
        if (wm >= 0)
#pragma unroll
            for (int u = 0; u < UC; u++) {
                const int tt = wm + u * NM;
                if (tt >= TC) continue;
                const int ti = tt / TN, tj = tt - ti * TN, j = 16 * tj + lc;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int i = 16 * ti + lr + 4 * v;
                    if (j >= NR) continue;
                    if (i < NC) MT[i * NR + j] = tot[u][v];
                    else if (i == NC) Lm[j] = tot[u][v];
                    else if (i == NC + 1 && j < NC) BT[j] = tot[u][v];
                }
            }
    }
    phase();
    // ---- face geometry: corners, then orientation and stabilisation weight;
    // the face basis at the rule's points
    for (int e = t; e < M * NVF * 3; e += NT) {
        const int f = e / (NVF * 3), l = e - f * (NVF * 3);
        FV[e] = d.V[3 * (size_t)d.fv[(size_t)d.cf[(size_t)c * M + f] * NVF + l / 3] + l % 3];
    }
    for (int e = t; e < QF * NFB; e += NT) {
        const int q = e / NFB, j = e - q * NFB;
        sm[G::fPhi + e] = legendre_at(d.fexp[2 * j], gx[q % G::Q1]) *
                          (DIM == 3 ? legendre_at(d.fexp[2 * j + 1], gx[q / G::Q1]) : 1.0);
    }
    phase();
    for (int f = t; f < M; f += NT) {
        const double* F = FV + f * NVF * 3;
        double x0[3], nv[3];
        gen_face_map<DIM>(F, 0, 0, x0, nv);
        const double dd = nv[0] * (x0[0] - ctr[0]) + nv[1] * (x0[1] - ctr[1]) + nv[2] * (x0[2] - ctr[2]);
        const double sg = dd < 0 ? -1.0 : 1.0;
        Sg[f] = sg;
        const double l0 = norm3(nv[0], nv[1], nv[2]);
        const double nu[3] = {sg * nv[0] / l0, sg * nv[1] / l0, sg * nv[2] / l0};
        double Kn = 0;
        for (int r = 0; r < 3; r++)
            for (int q = 0; q < 3; q++) Kn += nu[r] * Kc[r * 3 + q] * nu[q];
        double hF = 0;
        for (int e = 0; e < (DIM == 3 ? 4 : 1); e++) {
            const int a1 = (e + 1) % NVF;
            const double e0 = F[3 * a1] - F[3 * e], e1 = F[3 * a1 + 1] - F[3 * e + 1], e2 = F[3 * a1 + 2] - F[3 * e + 2];
            hF = fmax(hF, norm3(e0, e1, e2));
        }
        Cf[f] = Kn / hF;
    }
    phase();

    // ---- face integrals: per face one product of the rows [w K grad psi . n |
    // w da phi] with the columns [phi | psi] over the face rule
    auto face_tables = [&](int f) {
        for (int e = t; e < QF * DIM; e += NT) {
            const int q = e / DIM, a = e - q * DIM;
            const int i0 = q % G::Q1, i1 = DIM == 3 ? q / G::Q1 : 0;
            double x[3], nv[3];
            gen_face_map<DIM>(FV + f * NVF * 3, gx[i0], DIM == 3 ? gx[i1] : 0.0, x, nv);
            const double sg = Sg[f];
            for (int b = 0; b < 3; b++) nv[b] *= sg;
            const double xa = a == 0 ? x[0] : (a == 1 ? x[1] : x[2]);
            legendre_table<P1>((xa - ctr[a]) / hw[a], sm + G::fTab + e * TB);
            sm[G::fKn + e] = Kc[3 * a] * nv[0] + Kc[3 * a + 1] * nv[1] + Kc[3 * a + 2] * nv[2];
            if (a == 0) {
                const double w = gw[i0] * (DIM == 3 ? gw[i1] : 1.0);
                sm[G::fW + (f & 1) * QF + q] = w * norm3(nv[0], nv[1], nv[2]);
            }
        }
    };
    double* P = sm + G::oP;
    double* Mf = sm + G::oMf;
    double* TF = sm + G::oTF;
    face_tables(0);
    phase();
    for (int f = 0; f < M; f++) {
        {
            TabRef L[3], D[3];
            refs(sm + G::fTab, L, D);
            const double r0 = 1.0 / hw[0], r1 = 1.0 / hw[1], r2 = 1.0 / hw[2];
#pragma unroll 2
            for (int q = bq; q < QF; q += NT / NR) {
                const double L0 = L[0].at(q), L1 = L[1].at(q), L2 = DIM == 3 ? L[2].at(q) : 1.0;
                const double D0 = D[0].at(q), D1 = D[1].at(q), D2 = DIM == 3 ? D[2].at(q) : 0.0;
                const double* kn = sm + G::fKn + q * DIM;
                sm[G::fPs + q * NR + bi] = L0 * L1 * L2;
                const double g0 = div_by(D0, hw[0], r0) * L1 * L2, g1 = div_by(L0 * D1, hw[1], r1) * L2;
                double kg = fma(g0, kn[0], g1 * kn[1]);
                if (DIM == 3) kg = fma(div_by(L0 * L1 * D2, hw[2], r2), kn[DIM == 3 ? 2 : 0], kg);
                sm[G::fKg + q * NR + bi] = gw[q % G::Q1] * (DIM == 3 ? gw[q / G::Q1] : 1.0) * kg;
            }
        }
        phase();
        constexpr int TFN = (NR + NFB + 15) / 16;
        int cnt = 0;
#pragma unroll
        for (int ti = 0; ti < TFN; ti++)
#pragma unroll
            for (int tj = 0; tj < TFN; tj++) {
                // rows of K grad psi need the columns of phi and of the cell basis only
                if (16 * ti + 15 < NR && 16 * tj >= NFB + NC) continue;
                // a tile stays with one wavefront for all faces: it alone
                // updates its entries of P
                if (cnt++ % NW != wave) continue;
                const int r = 16 * ti + lc, s = 16 * tj + lc;
                const bool kg = r < NR, ph = s < NFB;
                const double* pa = kg ? sm + G::fKg + r : sm + G::fPhi + min(r - NR, NFB - 1);
                const double* pb = ph ? sm + G::fPhi + s : sm + G::fPs + min(s - NFB, NR - 1);
                const int la = kg ? NR : NFB, lb = ph ? NFB : NR;
                const double* pw = sm + G::fW + (f & 1) * QF;
                const lane_d4 acc = tile<QF>(zero4, [&](int k) { return pa[k * la] * (kg ? 1.0 : pw[k]); },
                                             [&](int k) { return pb[k * lb]; });
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int i = 16 * ti + lr + 4 * v, j = 16 * tj + lc;
                    if (i < NR) {
                        if (i < 1) continue;
                        if (j < NFB) P[i * NH + NC + f * NFB + j] = acc[v];
                        else if (j < NFB + NC) P[i * NH + j - NFB] -= acc[v];
                    } else if (i < NR + NFB) {
                        if (j < NFB) Mf[(f * NFB + i - NR) * NFB + j] = acc[v];
                        else if (j < NFB + NR) TF[(f * NFB + i - NR) * NR + j - NFB] = acc[v];
                    }
                }
            }
        if (f + 1 < M) face_tables(f + 1);
        phase();
    }

    // ---- factors of S and the face masses (packed rows)
    const double* S = sm + G::oS;
    const double* MT = sm + G::oMT;
    double* LS_ = sm + G::aLS;
    double* LF = sm + G::aLF;
    auto put_rows = [](auto& a, int r, double* L) {
        constexpr int N = sizeof(a) / sizeof(a[0]);
#pragma unroll
        for (int k = 0; k < N; k++)
            if (k <= r) L[r * (r + 1) / 2 + k] = a[k];
    };
    if (wave == 0) {
        double a[N1];
        const int r = min(lane, N1 - 1);
#pragma unroll
        for (int k = 0; k < N1; k++) a[k] = S[r * N1 + k];
        if (lane_chol<N1, false>(a, 0, lane) && lane == 0) atomicOr(err, 1);
        if (lane < N1) put_rows(a, r, LS_);
    }
    if (wave == 1 % NW) {
        double a[NFB];
        const int rr = min(lane, NF - 1), base = rr / NFB * NFB, r = rr - base;
#pragma unroll
        for (int k = 0; k < NFB; k++) a[k] = Mf[rr * NFB + k];
        if (lane_chol<NFB, true>(a, base, r) && lane < NF) atomicOr(err, 1);
        if (lane < NF) put_rows(a, r, LF + rr / NFB * G::tri(NFB));
    }
    phase();
    // ---- solves: reconstruction rows 1.., face projections
    {
        constexpr int YT = (NH + 63) / 64, UT = (M * NR + 63) / 64;
        for (int task = wave; task < YT + UT; task += NW) {
            if (task < YT) {
                const int col = task * 64 + lane;
                if (col < NH) {
                    double x[N1];
#pragma unroll
                    for (int i = 0; i < N1; i++) x[i] = P[(i + 1) * NH + col];
                    lane_solve<N1>(x, [&](int i, int j) { return LS_[i * (i + 1) / 2 + j]; });
#pragma unroll
                    for (int i = 0; i < N1; i++) P[(i + 1) * NH + col] = x[i];
                }
            } else {
                const int e = (task - YT) * 64 + lane;
                if (e < M * NR) {
                    const int f = e / NR, i = e - f * NR;
                    const double* L = LF + f * G::tri(NFB);
                    double x[NFB];
#pragma unroll
                    for (int a = 0; a < NFB; a++) x[a] = TF[(f * NFB + a) * NR + i];
                    lane_solve<NFB>(x, [&](int i2, int j2) { return L[i2 * (i2 + 1) / 2 + j2]; });
#pragma unroll
                    for (int a = 0; a < NFB; a++) TF[(f * NFB + a) * NR + i] = x[a];
                }
            }
        }
    }
    phase();
    // row 0 from the mean value; W = S P (rows 1..)
    for (int j = t; j < NH; j += NT) {
        double v = j < NC ? Lm[j] : 0.0;
#pragma unroll 4
        for (int i = 1; i < NR; i++) v = fma(-Lm[i], P[i * NH + j], v);
        P[j] = v / Lm[0];
    }
    double* W = sm + G::aW;
    constexpr int TJ = (NH + 15) / 16;
    {
        constexpr int TI = (N1 + 15) / 16;
        for (int tt = wave; tt < TI * TJ; tt += NW) {
            const int ti = tt / TJ, tj = tt - ti * TJ, j = 16 * tj + lc;
            const double *pa = S + min(16 * ti + lc, N1 - 1) * N1, *pb = P + NH + min(j, NH - 1);
            const lane_d4 w = tile<N1>(zero4, [&](int k) { return pa[k]; }, [&](int k) { return pb[k * NH]; });
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int i = 16 * ti + lr + 4 * v;
                if (i < N1 && j < NH) W[i * NH + j] = w[v];
            }
        }
    }
    phase();
    // ---- A = P^T W, kept in registers (the tiles that hold A_TT, A_TF or
    // A_FF), and N_T P
    const auto need = [](int ti, int tj) { return 16 * ti < NC || 16 * tj + 15 >= NC; };
    constexpr int TA = TJ * TJ, UA = (TA + NW - 1) / NW;
    lane_d4 A[UA];
#pragma unroll
    for (int u = 0; u < UA; u++) {
        const int tt = wave + u * NW, ti = tt / TJ, tj = tt - ti * TJ;
        A[u] = zero4;
        if (tt >= TA || !need(ti, tj)) continue;
        const double *pa = P + NH + min(16 * ti + lc, NH - 1), *pb = W + min(16 * tj + lc, NH - 1);
        A[u] = tile<N1>(zero4, [&](int k) { return pa[k * NH]; }, [&](int k) { return pb[k * NH]; });
    }
    double* Dt = sm + G::aN;
    double* LM = Dt + NC * NH;
    {
        constexpr int TI = (NC + 15) / 16, UN = (TI * TJ + NW - 1) / NW;
        lane_d4 n[UN];
#pragma unroll
        for (int u = 0; u < UN; u++) {
            const int tt = wave + u * NW, ti = tt / TJ, tj = tt - ti * TJ;
            if (tt >= TI * TJ) continue;
            const double *pa = MT + min(16 * ti + lc, NC - 1) * NR, *pb = P + min(16 * tj + lc, NH - 1);
            n[u] = tile<NR>(zero4, [&](int k) { return pa[k]; }, [&](int k) { return pb[k * NH]; });
        }
        phase();
#pragma unroll
        for (int u = 0; u < UN; u++) {
            const int tt = wave + u * NW, ti = tt / TJ, tj = tt - ti * TJ, j = 16 * tj + lc;
            if (tt >= TI * TJ) continue;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int i = 16 * ti + lr + 4 * v;
                if (i < NC && j < NH) Dt[i * NH + j] = n[u][v];
            }
        }
    }
    if (wave == NW - 1) {
        double a[NC];
        const int r = min(lane, NC - 1);
#pragma unroll
        for (int k = 0; k < NC; k++) a[k] = MT[r * NR + k];
        if (lane_chol<NC, false>(a, 0, lane) && lane == 0) atomicOr(err, 1);
        if (lane < NC) put_rows(a, r, LM);
    }
    phase();
    // ---- D_T = M_T^-1 N_T P - [I 0]
    for (int col = wave * 64 + lane; col < NH; col += NT) {
        double x[NC];
#pragma unroll
        for (int i = 0; i < NC; i++) x[i] = Dt[i * NH + col];
        lane_solve<NC>(x, [&](int i, int j) { return LM[i * (i + 1) / 2 + j]; });
#pragma unroll
        for (int i = 0; i < NC; i++) Dt[i * NH + col] = i == col ? x[i] - 1.0 : x[i];
    }
    if (d.post)
        for (int e = t; e < NR * NH; e += NT) sm[G::pP + e] = P[e];
    phase();
    // ---- stabilisation: D_F = Pi_F (P - D_T) - I_F of all faces
    double* DF = sm + G::bDF;
    {
        constexpr int TI = (NF + 15) / 16, UD = (TI * TJ + NW - 1) / NW;
        lane_d4 x[UD];
#pragma unroll
        for (int u = 0; u < UD; u++) {
            const int tt = wave + u * NW, ti = tt / TJ, tj = tt - ti * TJ, j = 16 * tj + lc;
            if (tt >= TI * TJ) continue;
            const double *pa = TF + min(16 * ti + lc, NF - 1) * NR, *pb = P + min(j, NH - 1), *pc = Dt + min(j, NH - 1);
            x[u] = tile<NR>(zero4, [&](int k) { return pa[k]; }, [&](int k) { return pb[k * NH]; });
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (j == NC + 16 * ti + lr + 4 * v) x[u][v] -= 1.0;
            x[u] = tile<NC>(x[u], [&](int k) { return -pa[k]; }, [&](int k) { return pc[k * NH]; });
        }
        phase();
#pragma unroll
        for (int u = 0; u < UD; u++) {
            const int tt = wave + u * NW, ti = tt / TJ, tj = tt - ti * TJ, j = 16 * tj + lc;
            if (tt >= TI * TJ) continue;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int i = 16 * ti + lr + 4 * v;
                if (i < NF && j < NH) DF[i * NH + j] = x[u][v];
            }
        }
    }
    phase();
    // A += c_f D_F^T (M_F D_F), face by face, M / 2 faces' products at a time
    double* MD = sm + G::bMD;
    constexpr int FH = M / 2;
    static_assert(NFB <= 16, "a face's unknowns must fit one tile");
    for (int f0 = 0; f0 < M; f0 += FH) {
        for (int tt = wave; tt < FH * TJ; tt += NW) {
            const int fl = tt / TJ, tj = tt - fl * TJ, f = f0 + fl, j = 16 * tj + lc;
            const double *pa = Mf + (f * NFB + min(lc, NFB - 1)) * NFB, *pb = DF + f * NFB * NH + min(j, NH - 1);
            const lane_d4 m = tile<NFB>(zero4, [&](int k) { return pa[k]; }, [&](int k) { return pb[k * NH]; });
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int i = lr + 4 * v;
                if (i < NFB && j < NH) MD[(fl * NFB + i) * NH + j] = m[v];
            }
        }
        phase();
#pragma unroll
        for (int u = 0; u < UA; u++) {
            const int tt = wave + u * NW, ti = tt / TJ, tj = tt - ti * TJ;
            if (tt >= TA || !need(ti, tj)) continue;
            for (int fl = 0; fl < FH; fl++) {
                const double cf = Cf[f0 + fl];
                const double* pa = DF + (f0 + fl) * NFB * NH + min(16 * ti + lc, NH - 1);
                const double* pb = MD + fl * NFB * NH + min(16 * tj + lc, NH - 1);
                A[u] += tile<NFB>(zero4, [&](int k) { return cf * pa[k * NH]; }, [&](int k) { return pb[k * NH]; });
            }
        }
        phase();
    }
    // ---- static condensation: X = A_TT^-1 [A_TF B_T]
    double* AT = sm + G::xA;  // [A_TT A_TF]
    double* X = sm + G::xX;   // row length NF + 1
    double* LT = sm + G::xL;
#pragma unroll
    for (int u = 0; u < UA; u++) {
        const int tt = wave + u * NW, ti = tt / TJ, tj = tt - ti * TJ, j = 16 * tj + lc;
        if (tt >= TA || 16 * ti >= NC) continue;
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int i = 16 * ti + lr + 4 * v;
            if (i < NC && j < NH) AT[i * NH + j] = A[u][v];
        }
    }
    phase();
    if (wave == 0) {
        double a[NC];
        const int r = min(lane, NC - 1);
#pragma unroll
        for (int k = 0; k < NC; k++) a[k] = AT[r * NH + k];
        if (lane_chol<NC, false>(a, 0, lane) && lane == 0) atomicOr(err, 1);
        if (lane < NC) put_rows(a, r, LT);
        lds_order();
        if (lane <= NF) {
            double x[NC];
#pragma unroll
            for (int i = 0; i < NC; i++) x[i] = lane < NF ? AT[i * NH + NC + lane] : BT[i];
            lane_solve<NC>(x, [&](int i, int j) { return LT[i * (i + 1) / 2 + j]; });
#pragma unroll
            for (int i = 0; i < NC; i++) X[i * (NF + 1) + lane] = x[i];
        }
    }
    phase();
    if (d.post) {
        // ---- recovery v_T = X[:, NF] - X[:, :NF] v_F, reconstruction
        // P [v_T; v_F], L2 integrals
        double* wv = sm + G::pW;  // nh: [v_T; v_F]
        double* pc = sm + G::pC;  // nr
        const double* Pp = sm + G::pP;
        for (int r = t; r < NF; r += NT) {
            const int f = r / NFB, a = r - f * NFB, row = blk[M * M + f];
            wv[NC + r] = row >= 0 ? d.xsol[(size_t)row * NFB + a] : 0.0;
        }
        phase();
        for (int i = t; i < NC; i += NT) {
            double s = X[i * (NF + 1) + NF];
            for (int j = 0; j < NF; j++) s -= X[i * (NF + 1) + j] * wv[NC + j];
            wv[i] = s;
        }
        phase();
        for (int i = t; i < NR; i += NT) {
            double s = 0;
            for (int j = 0; j < NH; j++) s += Pp[i * NH + j] * wv[j];
            pc[i] = s;
        }
        phase();
        const int nl = d.nl1;
        const double* lx = d.l1;
        const double* lw = d.l1 + nl;
        const int nql = DIM == 3 ? nl * nl * nl : nl * nl;
        double e2 = 0, u2 = 0;
        for (int q = t; q < nql; q += NT) {
            const int i0 = q % nl, i1 = (q / nl) % nl, i2 = DIM == 3 ? q / (nl * nl) : 0;
            const double xi[3] = {lx[i0], lx[i1], DIM == 3 ? lx[i2] : 0.0};
            const double w = lw[i0] * lw[i1] * (DIM == 3 ? lw[i2] : 1.0);
            double x[3];
            const double det = gen_cell_map<DIM>(CV, xi, x);
            double tb[3][TB], Lv[3][P1 + 1];
#pragma unroll
            for (int a = 0; a < 3; a++) {
                if (a < DIM) legendre_table<P1>((x[a] - ctr[a]) / hw[a], tb[a]);
                Lv[a][0] = 1;
#pragma unroll
                for (int p = 1; p <= P1; p++) Lv[a][p] = a < DIM ? tb[a][p - 1] : 0.0;
            }
            double ph = 0;
            int i = 0;  // the graded order of the reconstruction functions
#pragma unroll
            for (int dg = 0; dg <= P1; dg++)
#pragma unroll
                for (int a = dg; a >= 0; a--) {
                    if (DIM == 2) {
                        ph += pc[i++] * (Lv[0][a] * Lv[1][dg - a]);
                    } else {
#pragma unroll
                        for (int b = dg - a; b >= 0; b--) ph += pc[i++] * (Lv[0][a] * Lv[1][b] * Lv[2][dg - a - b]);
                    }
                }
            const double u = exact_at(d, x[0], x[1], x[2]);
            e2 += w * det * (u - ph) * (u - ph);
            u2 += w * det * u * u;
        }
        // workgroup reduction in a fixed order (per wavefront, then wavefronts)
        for (int o = 32; o > 0; o >>= 1) {
            e2 += __shfl_xor(e2, o, 64);
            u2 += __shfl_xor(u2, o, 64);
        }
        double* red = sm + G::pRed;
        if (lane == 0) {
            red[2 * wave] = e2;
            red[2 * wave + 1] = u2;
        }
        phase();
        if (t == 0) {
            double se = 0, su = 0;
            for (int w = 0; w < NW; w++) {
                se += red[2 * w];
                su += red[2 * w + 1];
            }
            d.cell_err[2 * (size_t)c] = se;
            d.cell_err[2 * (size_t)c + 1] = su;
        }
        return;
    }
    // ---- condensed matrix A_FF - A_TF^T X (into LDS)
    double* Sc = sm + G::xS;
#pragma unroll
    for (int u = 0; u < UA; u++) {
        const int tt = wave + u * NW, ti = tt / TJ, tj = tt - ti * TJ;
        if (tt >= TA || 16 * ti + 15 < NC || 16 * tj + 15 < NC) continue;
        const int r = 16 * ti + lc, s = 16 * tj + lc;
        const double *pa = AT + min(r, NH - 1), *pb = X + min(max(s - NC, 0), NF);
        const lane_d4 x = tile<NC>(A[u], [&](int k) { return -pa[k * NH]; }, [&](int k) { return pb[k * (NF + 1)]; });
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int i = 16 * ti + lr + 4 * v - NC, j = s - NC;
            if (i >= 0 && i < NF && j >= 0 && j < NF) Sc[i * NF + j] = x[v];
        }
    }
    phase();
    // ---- blocks and right-hand side into the global system.  Two faces
    // share one cell, so an off-diagonal block is this cell's alone; a
    // diagonal block and an entry of b take at most two contributions, whose
    // sum does not depend on the order.
    constexpr int BSZ = NFB * NFB;
    for (int e = t; e < NF * NF; e += NT) {
        const int fg = e / BSZ, ab = e - fg * BSZ, f = fg / M, g = fg - f * M;
        const int p = blk[fg];
        if (p < 0) continue;
        const int a = ab / NFB, b = ab - a * NFB;
        const double v = Sc[(f * NFB + a) * NF + g * NFB + b];
        double* o = d.vals + (size_t)p * BSZ + ab;
        if (f == g) atomicAdd(o, v);
        else *o = v;
    }
    if (d.elem_vals != nullptr) {
        double* ev = d.elem_vals + (size_t)d.elem_pos[c] * d.elem_stride;
        for (int e = t; e < NF * (NF / 2 + 1); e += NT) {
            const int dt = e / NF, r = e - dt * NF, s = r + dt < NF ? r + dt : r + dt - NF;
            ev[elem_entry(NF, r, s)] = Sc[r * NF + s];
        }
    }
    for (int r = t; r < NF; r += NT) {
        const int f = r / NFB, a = r - f * NFB, row = blk[M * M + f];
        if (row < 0) continue;
        double v = 0;
#pragma unroll
        for (int i = 0; i < NC; i++) v = fma(-AT[i * NH + NC + r], X[i * (NF + 1) + NF], v);
        atomicAdd(d.b + (size_t)row * NFB + a, v);
    }
}

template <int DIM, int K, int NW, int MW>
void launch(Ctx& c, const HhoDev& d, int* err, int maxlds) {
    using G = Gen<DIM, K>;
    FH_CHECK(d.nc == G::NC && d.nr == G::NR && d.nfb == G::NFB && d.nfc == G::M && d.nvc == G::NVC &&
                 d.nvf == G::NVF && d.ng1 == G::Q1,
             -3, "general cells: sizes do not match the degree");
    const size_t lds = (size_t)(d.post ? G::total_post : G::total) * sizeof(double);
    FH_CHECK(lds <= (size_t)maxlds, -3,
             "cell matrices (" + std::to_string(lds) + " bytes) exceed the LDS of a workgroup (" + std::to_string(maxlds) + ")");
    auto kern = k_hho_general<DIM, K, NW, MW>;
    if (lds > 65536) FH_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3(d.ncell), dim3(NW * 64), lds, c.stream, d, err);
    FH_HIP(hipGetLastError());
}

}  // namespace

void launch_hho_general(Ctx& c, const HhoDev& d) {
    FH_CHECK(!d.post || (d.xsol && d.cell_err), -2, "post-processing needs the face solution and the cell output");
    FH_CHECK(d.nl1 <= 8, -3, "general cells: degree k <= 3");
    int dev = 0, maxlds = 0;
    FH_HIP(hipGetDevice(&dev));
    FH_HIP(hipDeviceGetAttribute(&maxlds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    DevBuf err(sizeof(int));
    FH_HIP(hipMemsetAsync(err.p, 0, sizeof(int), c.stream));
    int* e = err.as<int>();
    const int key = d.dim * 10 + d.ng1 - 2;  // degree k = ng1 - 2
    // Wavefronts per cell, and per SIMD.  Small cells are one wavefront each,
    // three to five to a SIMD: a few spilled registers cost less than the
    // latency that the other cells hide (12 167 hexahedra at k = 0: 109 us at
    // four, 121 us at three; k = 1: 317 us at three, 330 us at two, 354 us at
    // four; 10 000 quadrilaterals at k = 3: 281 us at two, 301 us at three; 282
    // and 249 us of the chosen ones since two points' tables are read at once).
    // At k = 2 and 3 in 3-D the tiles feed two and four wavefronts and the
    // factorisations need the registers of two per SIMD (k = 2: 1.11 ms with
    // two wavefronts, 1.67 ms with four; k = 3: 4.84 ms with four, 8.98 ms
    // with eight at four per SIMD, which spill).
    switch (key) {
        case 20: launch<2, 0, 1, 5>(c, d, e, maxlds); break;
        case 21: launch<2, 1, 1, 4>(c, d, e, maxlds); break;
        case 22: launch<2, 2, 1, 4>(c, d, e, maxlds); break;
        case 23: launch<2, 3, 1, 2>(c, d, e, maxlds); break;
        case 30: launch<3, 0, 1, 4>(c, d, e, maxlds); break;
        case 31: launch<3, 1, 1, 3>(c, d, e, maxlds); break;
        case 32: launch<3, 2, 2, 2>(c, d, e, maxlds); break;
        case 33: launch<3, 3, 4, 2>(c, d, e, maxlds); break;
        default: throw Error(-3, "general cells: degree k <= 3 in 2-D or 3-D");
    }
    int h = 0;
    FH_HIP(hipMemcpyAsync(&h, err.p, sizeof(int), hipMemcpyDeviceToHost, c.stream));
    FH_HIP(hipStreamSynchronize(c.stream));
    FH_CHECK(!(h & 2), -6, "a cell of the HHO assembly is inverted at a quadrature point");
    FH_CHECK(!(h & 4), -6, "general cells: the diffusion tensor must be diagonal");
    FH_CHECK(h == 0, -6, "a local matrix of the HHO assembly is not SPD");
}

}  // namespace fh
