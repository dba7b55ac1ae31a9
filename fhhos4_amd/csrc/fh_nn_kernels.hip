// gfx950 kernels of the learned post-smoother: a message-passing network over
// the face graph of the condensed operator (one node per block row, edges =
// off-diagonal blocks), hidden width 32.
//
// Layout: node features are row-major n x 32 FP32 arrays, one 128-byte row per
// face.  The message-passing layer (forward, inference and backward) gathers
// neighbour rows with 8 lanes of 16 bytes each and multiplies on the matrix
// cores: FP32 for training, BF16 operands (FP32 sums) for inference.  Weights
// are FP32 for training and BF16 for inference.
//
// Weight gradients are sums over nodes of outer products, formed for all
// layers in one launch on v_mfma_f64_16x16x4f64: FP64 sums per workgroup of a
// fixed-size grid, added in a fixed order by a second kernel, so gradients are
// deterministic.
#include <algorithm>

#include "fh_lane.h"
#include "fh_nn.h"

namespace fh {
namespace {

constexpr int H = kNnHidden;  // 32
constexpr int kNodesPerWG = 8;
constexpr int kOuterWGs = 128;
constexpr int kMaxDin = 12, kMaxNf = 10;
constexpr int kPrepWGs = 1024;  // partial sums of |v|^2

struct bf16w {
    uint16_t u;
};
__device__ __forceinline__ float wload(const float* p) { return *p; }
__device__ __forceinline__ float wload(const bf16w* p) { return __uint_as_float(((uint32_t)p->u) << 16); }

// v = D^-1 r1 (FP32) and the workgroup's share of |v|^2 (FP64), 256 / nf block
// rows at a time: their inverse blocks (one contiguous span) and entries of r1
// go through LDS, then thread t forms entry t of the tile.  Bound by reading
// the inverse blocks: 12.6 us for 95 232 blocks of 10 x 10 (38 MB) with the next
// tile's loads in flight, 25.5 us when a workgroup loads its tiles one after the
// other (a thread per unknown that reads its row of D strided took 21.5 us,
// without the norm).
__global__ __launch_bounds__(256) void k_nn_prep(int n, int nf, const double* __restrict__ r1,
                                                 const float* __restrict__ invD, float* __restrict__ v,
                                                 double* __restrict__ partials) {
    __shared__ float sD[256 * kMaxNf], sr[256];
    __shared__ double sw[4];
    const int t = threadIdx.x, R = 256 / nf, b = t / nf;
    double vv = 0;
    // the next tile's loads are in flight while this one is formed
    float nd[kMaxNf];
    double nr = 0;
    auto fetch = [&](int64_t r0) {
        const int nv = (int)min((int64_t)R, n - r0) * nf, ne = nv * nf;
        const float* D = invD + r0 * nf * nf;
#pragma unroll
        for (int u = 0; u < kMaxNf; u++)
            if (t + 256 * u < ne) nd[u] = __builtin_nontemporal_load(D + t + 256 * u);
        if (t < nv) nr = r1[r0 * nf + t];
    };
    const int64_t step = (int64_t)gridDim.x * R;
    fetch((int64_t)blockIdx.x * R);  // every workgroup has a tile
    for (int64_t r0 = (int64_t)blockIdx.x * R; r0 < n; r0 += step) {
        const int nv = (int)min((int64_t)R, n - r0) * nf, ne = nv * nf;
#pragma unroll
        for (int u = 0; u < kMaxNf; u++)
            if (t + 256 * u < ne) sD[t + 256 * u] = nd[u];
        if (t < nv) sr[t] = (float)nr;
        __syncthreads();
        if (r0 + step < n) fetch(r0 + step);
        if (t < nv) {
            float s = 0.f;
            for (int j = 0; j < nf; j++) s += sD[t * nf + j] * sr[b * nf + j];
            v[r0 * nf + t] = s;
            vv += (double)s * (double)s;
        }
        __syncthreads();
    }
    for (int o = 32; o > 0; o >>= 1) vv += __shfl_down(vv, o, 64);
    if ((t & 63) == 0) sw[t >> 6] = vv;
    __syncthreads();
    if (t == 0) partials[blockIdx.x] = ((sw[0] + sw[1]) + sw[2]) + sw[3];
}

// Encoder: sigma = sqrt(<v, v> / (n nf)) from the npart partial sums (added by
// every workgroup in the same order; the first one writes sigma to
// s[slot_sigma]), u = v / sigma, x = [u, feat] (stored when x0 is not null)
// and h = relu(We x + be).  Lane c keeps row c of We in registers; the inputs
// of 64 nodes at a time are staged in LDS.
constexpr int kEncodeNodes = 64, kEncodeMaxWGs = 1536;

template <class TW>
__global__ __launch_bounds__(256) void k_nn_encode(int n, int nf, int npart, const double* __restrict__ partials,
                                                    const float* __restrict__ v, const float* __restrict__ feat,
                                                    double* s, int slot_sigma, const TW* __restrict__ We,
                                                    const TW* __restrict__ be, float* __restrict__ u,
                                                    float* __restrict__ x0, float* __restrict__ h) {
    __shared__ float sx[kEncodeNodes * kMaxDin];
    __shared__ float sWe[H * kMaxDin + H];
    __shared__ double sw[4];
    const int t = threadIdx.x, din = nf + 2;
    double vv = 0;
    for (int i = t; i < npart; i += 256) vv += partials[i];
    for (int o = 32; o > 0; o >>= 1) vv += __shfl_down(vv, o, 64);
    if ((t & 63) == 0) sw[t >> 6] = vv;
    for (int e = t; e < H * din; e += 256) sWe[e] = wload(We + e);
    if (t < H) sWe[H * kMaxDin + t] = wload(be + t);
    __syncthreads();
    const double sig = sqrt((((sw[0] + sw[1]) + sw[2]) + sw[3]) / ((double)n * nf));
    const float inv = sig > 0 ? (float)(1.0 / sig) : 0.f;
    if (blockIdx.x == 0 && t == 0) s[slot_sigma] = sig;
    const int c = t & (H - 1), q = t >> 5;
    float wr[kMaxDin];
#pragma unroll
    for (int k = 0; k < kMaxDin; k++) wr[k] = k < din ? sWe[c * din + k] : 0.f;
    const float bias = sWe[H * kMaxDin + c];
    for (int64_t i0 = (int64_t)blockIdx.x * kEncodeNodes; i0 < n; i0 += (int64_t)gridDim.x * kEncodeNodes) {
        const int nn = (int)min((int64_t)kEncodeNodes, n - i0);
        for (int e = t; e < nn * nf; e += 256) {
            const int i = e / nf, a = e - i * nf;
            const float val = v[i0 * nf + e] * inv;
            u[i0 * nf + e] = val;
            sx[i * kMaxDin + a] = val;
        }
        for (int e = t; e < nn * 2; e += 256) sx[(e >> 1) * kMaxDin + nf + (e & 1)] = feat[i0 * 2 + e];
        __syncthreads();
        if (x0)
            for (int e = t; e < nn * din; e += 256) x0[i0 * din + e] = sx[e / din * kMaxDin + e % din];
        for (int i = q; i < nn; i += kNodesPerWG) {
            float acc = bias;
#pragma unroll
            for (int k = 0; k < kMaxDin; k++)
                if (k < din) acc += wr[k] * sx[i * kMaxDin + k];
            h[(i0 + i) * H + c] = acc > 0.f ? acc : 0.f;
        }
        __syncthreads();
    }
}

// Message-passing layer of 16 nodes per wavefront:
//   m_i = sum_j w_ij h_j (edge order, FP32);  y_i = S h_i + N m_i + c
//   LAYER_TRAIN  out = relu(y), m stored for the backward pass (FP32 products)
//   LAYER_INFER  out = relu(y), h and m rounded to BF16 for the products
//   LAYER_BACK   h, w, c: the gradient at the layer's output, the weights of
//                the reverse edges, none; S and N transposed; out = y where
//                the layer's input (mask) is positive, else 0: the gradient at
//                the previous layer's output.  (N^T m with m gathered first is
//                the sum of the neighbours' N^T h.)
// 8 lanes of 16 bytes read a 128-byte row, so one load instruction fetches 8
// neighbour rows; the lane group g sums the edges of nodes g and g + 8, their
// next kGather rows each in flight together (column indexes and weights of 8
// edges come in one load and are passed on by shuffles).  The 16 x 64 operand
// [h m] goes through LDS to the matrix cores: v_mfma_f32_16x16x4f32 or
// v_mfma_f32_16x16x32_bf16, lane l supplying row (column) l % 16 and receiving
// rows 4 (l / 16) + v of column l % 16.  Bound by the latency of the gather:
// 16 nodes instead of 32 per wavefront and 16-byte lanes halve the number of
// dependent loads (95 232 nodes, 1.02 M edges, BF16: 13.4 us; 36.5 us with 4-byte
// lanes and 32 nodes).  Workgroups of one XCD take a contiguous range of nodes, whose
// neighbour rows its L2 then holds.
enum { LAYER_TRAIN = 0, LAYER_INFER = 1, LAYER_BACK = 2 };
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
constexpr int kLTile = 16, kLWaves = 4;
constexpr int kGather = 6;

__device__ __forceinline__ __bf16 to_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return __builtin_bit_cast(__bf16, (uint16_t)(u >> 16));
}

template <int MODE>
__global__ __launch_bounds__(kLWaves * 64) void k_nn_layer(int n, const int* __restrict__ rp,
                                                            const int* __restrict__ ci, const float* __restrict__ w,
                                                            const float* __restrict__ hin, const void* Sv,
                                                            const void* Nv, const void* cv,
                                                            const float* __restrict__ mask, float* __restrict__ hout,
                                                            float* __restrict__ m_out) {
    constexpr bool BF = MODE == LAYER_INFER, BACK = MODE == LAYER_BACK;
    using TW = std::conditional_t<BF, bf16w, float>;
    using TT = std::conditional_t<BF, __bf16, float>;
    constexpr int PITCH = BF ? 2 * H + 8 : 2 * H + 4;  // rows 16 bytes apart in their banks
    __shared__ __align__(16) TT tiles[kLWaves][kLTile * PITCH];
    const TW *S = (const TW*)Sv, *N = (const TW*)Nv;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int wg = blockIdx.x;
    {
        const int nwg = gridDim.x, xcd = wg & 7, per = nwg >> 3, rem = nwg & 7;
        wg = xcd * per + (xcd < rem ? xcd : rem) + (wg >> 3);
    }
    const int64_t i0 = ((int64_t)wg * kLWaves + wave) * kLTile;
    if (i0 >= n) return;  // wavefront-uniform; no barrier follows
    const int nt = (int)min((int64_t)kLTile, n - i0);
    TT* tl = tiles[wave];
    // edges: lane group g (8 lanes) sums nodes g and g + 8
    const int g = lane >> 3, c4 = lane & 7, gl = lane & 56;
    const int rpv = rp[i0 + min(lane, nt)];
    int beg[2], deg[2];
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const int k = g + 8 * r;
        beg[r] = __shfl(rpv, min(k, nt), 64);
        deg[r] = __shfl(rpv, min(k + 1, nt), 64) - beg[r];
    }
    floatx4 own[2], m[2];
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const int k = g + 8 * r;
        own[r] = k < nt ? *(const floatx4*)(hin + (i0 + k) * H + 4 * c4) : floatx4{0.f, 0.f, 0.f, 0.f};
        m[r] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    int dmax = max(deg[0], deg[1]);
#pragma unroll
    for (int o = 8; o < 64; o <<= 1) dmax = max(dmax, __shfl_xor(dmax, o, 64));
    int colv[2];
    float wv[2];
    auto load_edges = [&](int e0) {
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const bool ok = c4 < kGather && e0 + c4 < deg[r];
            colv[r] = ok ? ci[beg[r] + e0 + c4] : 0;
            wv[r] = ok ? w[beg[r] + e0 + c4] : 0.f;
        }
    };
    load_edges(0);
    for (int e0 = 0; e0 < dmax; e0 += kGather) {
        floatx4 x[2][kGather];
        float we[2][kGather];
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int k = 0; k < kGather; k++) {
                const int col = __shfl(colv[r], gl + k, 64);
                we[r][k] = __shfl(wv[r], gl + k, 64);
                if (e0 + k < deg[r]) x[r][k] = *(const floatx4*)(hin + (int64_t)col * H + 4 * c4);
            }
        load_edges(e0 + kGather);
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int k = 0; k < kGather; k++)
                if (e0 + k < deg[r]) {
#pragma unroll
                    for (int a = 0; a < 4; a++) m[r][a] += we[r][k] * x[r][k][a];
                }
    }
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const int k = g + 8 * r;
        if (MODE == LAYER_TRAIN && k < nt) *(floatx4*)(m_out + (i0 + k) * H + 4 * c4) = m[r];
        if constexpr (BF) {
            bf16x4_t hb, mb;
#pragma unroll
            for (int a = 0; a < 4; a++) {
                hb[a] = to_bf16(own[r][a]);
                mb[a] = to_bf16(m[r][a]);
            }
            *(bf16x4_t*)(tl + k * PITCH + 4 * c4) = hb;
            *(bf16x4_t*)(tl + k * PITCH + H + 4 * c4) = mb;
        } else {
            *(floatx4*)(tl + k * PITCH + 4 * c4) = own[r];
            *(floatx4*)(tl + k * PITCH + H + 4 * c4) = m[r];
        }
    }
    lds_order();
    // [h m] (16 x 64) times [S N]^T (64 x 32); rows >= nt are zero
    const int lr = lane >> 4, lc = lane & 15;
    floatx4 acc[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const float b = BACK ? 0.f : wload((const TW*)cv + 16 * j + lc);
        acc[j] = floatx4{b, b, b, b};
    }
    if constexpr (BF) {
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const bf16x8_t a = *(const bf16x8_t*)(tl + lc * PITCH + 32 * t + 8 * lr);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                // entries k = 8 lr .. 8 lr + 7 of row 16 j + lc of S (t = 0) or N
                const bf16x8_t b = *(const bf16x8_t*)((t == 0 ? S : N) + (16 * j + lc) * H + 8 * lr);
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[j], 0, 0, 0);
            }
        }
    } else {
        // four chains per tile, added pairwise: shorter ones round less, and
        // their instructions do not wait for each other
        floatx4 part[3][2];
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
            for (int j = 0; j < 2; j++) part[q][j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 16; t++) {
            const int k = (4 * t + lr) & (H - 1);
            const float* W = (const float*)(t < 8 ? Sv : Nv);
            const float a = tl[lc * PITCH + 4 * t + lr];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const float b = BACK ? W[k * H + 16 * j + lc] : W[(16 * j + lc) * H + k];
                floatx4& to = t % 4 == 0 ? acc[j] : part[(t + 3) % 4 % 3][j];
                to = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, to, 0, 0, 0);
            }
        }
#pragma unroll
        for (int j = 0; j < 2; j++) acc[j] = (acc[j] + part[0][j]) + (part[1][j] + part[2][j]);
    }
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int k = 4 * lr + v;
        if (k >= nt) continue;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int64_t o = (i0 + k) * H + 16 * j + lc;
            const float y = acc[j][v];
            if constexpr (BACK) hout[o] = mask[o] > 0.f ? y : 0.f;
            else hout[o] = y > 0.f ? y : 0.f;
        }
    }
}

// Output: delta_i = sigma (u_i + Wo h_i + bo), thread per unknown (nf <= kMaxNf);
// with e1 the error left, e1 - delta, in its place.
template <class TW>
__global__ void k_nn_out(int n, int nf, const float* __restrict__ h, const float* __restrict__ u,
                         const TW* __restrict__ Wo, const TW* __restrict__ bo, const double* s, int slot_sigma,
                         const double* __restrict__ e1, double* __restrict__ delta) {
    __shared__ float sWo[kMaxNf * H + kMaxNf];
    for (int e = threadIdx.x; e < nf * H; e += blockDim.x) sWo[e] = wload(Wo + e);
    if (threadIdx.x < nf) sWo[kMaxNf * H + threadIdx.x] = wload(bo + threadIdx.x);
    __syncthreads();
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)n * nf) return;
    const int i = (int)(t / nf), a = (int)(t - (int64_t)i * nf);
    const float* hi = h + (int64_t)i * H;
    float y = sWo[kMaxNf * H + a];
#pragma unroll 8
    for (int k = 0; k < H; k++) y += sWo[a * H + k] * hi[k];
    const double dl = s[slot_sigma] * (double)(u[t] + y);
    delta[t] = e1 ? e1[t] - dl : dl;
}

// ---------------------------------------------------------------- backward
// g = (-2 / s[slot_e0]) Adiff, gy = sigma g (FP32), and dh = Wo^T gy where the
// last layer's output h is positive; thread per (node, channel).
__global__ __launch_bounds__(256) void k_nn_out_back(int n, int nf, const double* __restrict__ Adiff,
                                                      const double* s, int slot_e0, int slot_sigma,
                                                      const float* __restrict__ Wo, const float* __restrict__ h,
                                                      float* __restrict__ gy, float* __restrict__ dh) {
    const int c = threadIdx.x & (H - 1);
    const int64_t i = (int64_t)blockIdx.x * kNodesPerWG + (threadIdx.x >> 5);
    if (i >= n) return;
    const double scale = -2.0 / s[slot_e0], sig = s[slot_sigma];
    float acc = 0.f;
    for (int a = 0; a < nf; a++) {
        const float ga = (float)(sig * (scale * Adiff[i * nf + a]));
        if (c == 0) gy[i * nf + a] = ga;
        acc += Wo[a * H + c] * ga;
    }
    dh[i * H + c] = h[i * H + c] > 0.f ? acc : 0.f;
}

// Weight gradients of every layer: for job j (blockIdx.y) the sums over nodes
// of A_i [B1_i B2_i]^T and of A_i, into the workgroup's share of the
// parameters.  A has da <= 32 channels, B1 db1 <= 32, B2 none or 32.  A
// wavefront takes 4 nodes per v_mfma_f64_16x16x4f64 step (lane l: channel
// l % 16 of node l / 16; the products of FP32 values are exact in FP64), the
// workgroup's wavefronts add their tiles in LDS in order.  One launch for all
// layers: per layer and parameter matrix it was 22 us, plus 58 us for adding
// 256 shares one after the other (11 520 nodes).
struct NnOuterJob {
    const float *A, *B1, *B2;
    int da, db1;
    int64_t o1, o2, ob;  // parameter offsets of the two matrices and the bias
};
constexpr int kMaxOuter = kNnMaxLayers + 2;
struct NnOuterArgs {
    NnOuterJob job[kMaxOuter];
};

__global__ __launch_bounds__(256) void k_nn_outer(int n, int64_t np, NnOuterArgs args, double* __restrict__ partials) {
    __shared__ double red[16 * 16];
    const NnOuterJob J = args.job[blockIdx.y];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane >> 4, lc = lane & 15;
    const int TB1 = (J.db1 + 15) / 16, TB2 = J.B2 ? 2 : 0, TA = (J.da + 15) / 16;
    lane_d4 acc[2][4];
    double sum[2] = {0.0, 0.0};
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 4; b++) acc[a][b] = lane_d4{0.0, 0.0, 0.0, 0.0};
    const int64_t step = (int64_t)gridDim.x * 4 * 4;
#pragma unroll 2
    for (int64_t i0 = ((int64_t)blockIdx.x * 4 + wave) * 4; i0 < n; i0 += step) {
        const int64_t i = i0 + lr;
        const bool ok = i < n;
        double av[2], bv[4];
#pragma unroll
        for (int a = 0; a < 2; a++) {
            const int ch = 16 * a + lc;
            av[a] = ok && ch < J.da ? (double)J.A[i * J.da + ch] : 0.0;
            sum[a] += av[a];
        }
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const int ch = 16 * b + lc;
            bv[b] = ok && ch < J.db1 ? (double)J.B1[i * J.db1 + ch] : 0.0;
            bv[2 + b] = ok && J.B2 ? (double)J.B2[i * H + ch] : 0.0;
        }
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int b = 0; b < 4; b++)
                if (a < TA && (b < 2 ? b < TB1 : b - 2 < TB2))  // wavefront-uniform
                    acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[a], bv[b], acc[a][b], 0, 0, 0);
    }
    double* out = partials + (int64_t)blockIdx.x * np;
    const int t = threadIdx.x;
    // tile by tile: the wavefronts' sums in order
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 4; b++) {
            if (a >= TA || (b < 2 ? b >= TB1 : b - 2 >= TB2)) continue;  // workgroup-uniform
            for (int w = 0; w < 4; w++) {
                if (wave == w)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        double* p = red + (lr + 4 * v) * 16 + lc;
                        *p = (w > 0 ? *p : 0.0) + acc[a][b][v];
                    }
                __syncthreads();
            }
            const int x = 16 * a + t / 16, y = 16 * (b & 1) + t % 16;
            const int db = b < 2 ? J.db1 : H;
            if (x < J.da && y < db) out[(b < 2 ? J.o1 : J.o2) + (int64_t)x * db + y] = red[t];
            __syncthreads();
        }
    // bias: nodes of the four lane rows, then the wavefronts
#pragma unroll
    for (int a = 0; a < 2; a++) {
        double q = sum[a];
        q += __shfl_xor(q, 16, 64);
        q += __shfl_xor(q, 32, 64);
        if (lane < 16) red[wave * 32 + 16 * a + lane] = q;
    }
    __syncthreads();
    if (t < J.da) out[J.ob + t] = ((red[t] + red[32 + t]) + red[64 + t]) + red[96 + t];
}

// grad[e] = sum over the nwg shares (fixed order): 32 parameters per
// workgroup, 8 threads each adding every eighth share.
__global__ __launch_bounds__(256) void k_nn_reduce(int np, int nwg, const double* __restrict__ partials,
                                                    float* __restrict__ grad) {
    __shared__ double sh[8][33];
    const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
    const int e = blockIdx.x * 32 + x;
    double s = 0;
    if (e < np) {
#pragma unroll 8
        for (int k = y; k < nwg; k += 8) s += partials[(int64_t)k * np + e];
    }
    sh[y][x] = s;
    __syncthreads();
    if (y == 0 && e < np) {
        double q = sh[0][x];
        for (int k = 1; k < 8; k++) q += sh[k][x];
        grad[e] = (float)q;
    }
}

// Adam (Kingma & Ba 2015) with bias correction, and the BF16 copy of the
// updated weights (round to nearest even).
__global__ void k_nn_adam(int np, float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m1,
                          float* __restrict__ m2, float lr, float b1, float b2, float eps, float c1, float c2,
                          bf16w* __restrict__ wb) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= np) return;
    const float gt = g[t];
    const float a = b1 * m1[t] + (1.f - b1) * gt;
    const float b = b2 * m2[t] + (1.f - b2) * gt * gt;
    m1[t] = a;
    m2[t] = b;
    const float v = w[t] - lr * (a / c1) / (sqrtf(b / c2) + eps);
    w[t] = v;
    uint32_t u = __float_as_uint(v);
    u += 0x7FFFu + ((u >> 16) & 1u);
    wb[t].u = (uint16_t)(u >> 16);
}

__global__ void k_nn_to_bf16(int np, const float* __restrict__ w, bf16w* __restrict__ wb) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= np) return;
    uint32_t u = __float_as_uint(w[t]);
    u += 0x7FFFu + ((u >> 16) & 1u);
    wb[t].u = (uint16_t)(u >> 16);
}

// Edge weights w_p = |tr A_p| / sum_{q in row, q != diag} |tr A_q| (w = 0 on
// the diagonal block), thread per block row.
__global__ void k_nn_edge_weights(int n, int nf, const int* __restrict__ rp, const int* __restrict__ ci,
                                  const double* __restrict__ vals, float* __restrict__ w) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double sum = 0;
    for (int p = rp[i]; p < rp[i + 1]; p++) {
        if (ci[p] == i) continue;
        double tr = 0;
        for (int a = 0; a < nf; a++) tr += vals[((int64_t)p * nf + a) * nf + a];
        sum += fabs(tr);
    }
    for (int p = rp[i]; p < rp[i + 1]; p++) {
        double tr = 0;
        for (int a = 0; a < nf; a++) tr += vals[((int64_t)p * nf + a) * nf + a];
        w[p] = (ci[p] == i || sum == 0) ? 0.f : (float)(fabs(tr) / sum);
    }
}

__global__ void k_nn_gather_index(int64_t nnzb, const int* __restrict__ idx, const float* __restrict__ src,
                                  float* __restrict__ dst) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < nnzb) dst[t] = src[idx[t]];
}

// Post-smoother selection (device-side, no host decision):
// s1 = delta.r1, s2 = delta.A delta.  If s1 > 0 and s2 > 0 the correction
// alpha delta with alpha = s1 / s2 lowers the energy norm of the error by
// s1^2 / s2; z += alpha delta.  Otherwise z += w D^-1 r1 (block Jacobi).
// With unit_step the correction is delta itself, accepted when it lowers the
// energy norm: delta.A delta - 2 delta.r1 < 0.
__global__ void k_nn_select(int64_t count, int nf, const double* s, int slot_s1, int slot_s2,
                            const double* __restrict__ delta, const double* __restrict__ r1,
                            const double* __restrict__ invD, double omega, int unit_step, double* __restrict__ z,
                            int* __restrict__ counters, const double* __restrict__ r,
                            const double* __restrict__ Adelta, double* __restrict__ Az) {
    const double s1 = s[slot_s1], s2 = s[slot_s2];
    const bool use = unit_step ? (s2 - 2.0 * s1 < 0) : (s1 > 0 && s2 > 0);
    const double alpha = unit_step ? 1.0 : s1 / s2;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t == 0) counters[use ? 0 : 1] += 1;
    if (t >= count) return;
    if (use) {
        z[t] += alpha * delta[t];
        // A z = A z0 + alpha A delta with A z0 = r - r1 (no product)
        if (Az) Az[t] = (r[t] - r1[t]) + alpha * Adelta[t];
    } else {
        const int64_t i = t / nf;
        const int a = (int)(t - i * nf);
        const double* D = invD + (i * nf + a) * nf;
        const double* r = r1 + i * nf;
        double v = 0;
        for (int b = 0; b < nf; b++) v += D[b] * r[b];
        z[t] += omega * v;
    }
}

inline int g1(int64_t n, int bs = 256) { return (int)((n + bs - 1) / bs); }

}  // namespace

// ------------------------------------------------------------ launchers
static int prep_wgs(int n, int nf) {
    const int R = 256 / nf;
    return std::min((n + R - 1) / R, kPrepWGs);
}
void nn_prep(Ctx& c, int n, int nf, const double* r1, const float* invD, float* v, double* partials) {
    FH_CHECK(nf >= 1 && nf <= kMaxNf, -3, "face block size out of range for the network");
    if (n <= 0) return;
    hipLaunchKernelGGL(k_nn_prep, dim3(prep_wgs(n, nf)), dim3(256), 0, c.stream, n, nf, r1, invD, v, partials);
    FH_HIP(hipGetLastError());
}
void nn_encode(Ctx& c, int n, int nf, const double* partials, const float* v, const float* feat, int slot_sigma,
               const void* We, const void* be, bool bf16, float* u, float* x0, float* h) {
    FH_CHECK(nf >= 1 && nf <= kMaxNf, -3, "face block size out of range for the network");
    if (n <= 0) return;
    const int g = std::min((n + kEncodeNodes - 1) / kEncodeNodes, kEncodeMaxWGs), np = prep_wgs(n, nf);
    if (bf16)
        hipLaunchKernelGGL(k_nn_encode<bf16w>, dim3(g), dim3(256), 0, c.stream, n, nf, np, partials, v, feat,
                           c.d_scalars, slot_sigma, (const bf16w*)We, (const bf16w*)be, u, x0, h);
    else
        hipLaunchKernelGGL(k_nn_encode<float>, dim3(g), dim3(256), 0, c.stream, n, nf, np, partials, v, feat,
                           c.d_scalars, slot_sigma, (const float*)We, (const float*)be, u, x0, h);
    FH_HIP(hipGetLastError());
}
static dim3 layer_grid(int n) { return dim3((unsigned)(((int64_t)n + kLTile * kLWaves - 1) / (kLTile * kLWaves))); }
void nn_layer(Ctx& c, int n, const int* rp, const int* ci, const float* w, const float* hin, const void* S,
              const void* N, const void* cb, bool bf16, float* hout, float* m_out) {
    if (n <= 0) return;
    FH_CHECK(bf16 == (m_out == nullptr), -3, "the BF16 layer is inference only, the FP32 layer stores the aggregate");
    if (bf16)
        hipLaunchKernelGGL(k_nn_layer<LAYER_INFER>, layer_grid(n), dim3(kLWaves * 64), 0, c.stream, n, rp, ci, w, hin,
                           S, N, cb, (const float*)nullptr, hout, m_out);
    else
        hipLaunchKernelGGL(k_nn_layer<LAYER_TRAIN>, layer_grid(n), dim3(kLWaves * 64), 0, c.stream, n, rp, ci, w, hin,
                           S, N, cb, (const float*)nullptr, hout, m_out);
    FH_HIP(hipGetLastError());
}
void nn_layer_back(Ctx& c, int n, const int* rp, const int* ci, const float* wT, const float* dpre, const float* S,
                   const float* N, const float* h, float* dprev) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_nn_layer<LAYER_BACK>, layer_grid(n), dim3(kLWaves * 64), 0, c.stream, n, rp, ci, wT, dpre, S,
                       N, (const void*)nullptr, h, dprev, (float*)nullptr);
    FH_HIP(hipGetLastError());
}
void nn_out(Ctx& c, int n, int nf, const float* h, const float* u, const void* Wo, const void* bo, bool bf16,
            int slot_sigma, const double* e1, double* delta) {
    FH_CHECK(nf >= 1 && nf <= kMaxNf, -3, "face block size out of range for the output layer");
    const int g = g1((int64_t)n * nf);
    if (bf16)
        hipLaunchKernelGGL(k_nn_out<bf16w>, dim3(g), dim3(256), 0, c.stream, n, nf, h, u, (const bf16w*)Wo,
                           (const bf16w*)bo, c.d_scalars, slot_sigma, e1, delta);
    else
        hipLaunchKernelGGL(k_nn_out<float>, dim3(g), dim3(256), 0, c.stream, n, nf, h, u, (const float*)Wo,
                           (const float*)bo, c.d_scalars, slot_sigma, e1, delta);
    FH_HIP(hipGetLastError());
}
void nn_out_back(Ctx& c, int n, int nf, const double* Adiff, int slot_e0, int slot_sigma, const float* Wo,
                 const float* h, float* gy, float* dh) {
    hipLaunchKernelGGL(k_nn_out_back, dim3((n + kNodesPerWG - 1) / kNodesPerWG), dim3(256), 0, c.stream, n, nf, Adiff,
                       c.d_scalars, slot_e0, slot_sigma, Wo, h, gy, dh);
    FH_HIP(hipGetLastError());
}
void nn_weight_grads(Ctx& c, int n, const NnShape& sh, const float* gy, const float* dh, const float* h,
                     const float* m, const float* x0, double* partials, float* grad) {
    const int64_t nH = (int64_t)n * H;
    NnOuterArgs a{};
    for (int l = 0; l < sh.layers; l++)
        a.job[l] = {dh + (l + 1) * nH, h + l * nH, m + l * nH, H, H, sh.S(l), sh.N(l), sh.c(l)};
    a.job[sh.layers] = {gy, h + sh.layers * nH, nullptr, sh.nf, H, sh.Wo(), 0, sh.bo()};
    a.job[sh.layers + 1] = {dh, x0, nullptr, H, sh.din(), sh.We(), 0, sh.be()};
    const int64_t np = sh.total();
    // 4 wavefronts of 4 nodes: at least one step each, at most kOuterWGs shares
    const int g = (int)std::min<int64_t>(std::max<int64_t>(1, ((int64_t)n + 63) / 64), kOuterWGs);
    hipLaunchKernelGGL(k_nn_outer, dim3(g, sh.layers + 2), dim3(256), 0, c.stream, n, np, a, partials);
    FH_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_nn_reduce, dim3((unsigned)((np + 31) / 32)), dim3(256), 0, c.stream, (int)np, g, partials,
                       grad);
    FH_HIP(hipGetLastError());
}
size_t nn_partials_bytes(const NnShape& sh) {
    return sizeof(double) * std::max<size_t>(kPrepWGs, (size_t)kOuterWGs * sh.total());
}
void nn_adam(Ctx& c, int np, float* w, const float* g, float* m1, float* m2, float lr, float b1, float b2, float eps,
             int step, void* wb) {
    const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    hipLaunchKernelGGL(k_nn_adam, dim3(g1(np)), dim3(256), 0, c.stream, np, w, g, m1, m2, lr, b1, b2, eps, c1, c2,
                       (bf16w*)wb);
    FH_HIP(hipGetLastError());
}
void nn_to_bf16(Ctx& c, int np, const float* w, void* wb) {
    hipLaunchKernelGGL(k_nn_to_bf16, dim3(g1(np)), dim3(256), 0, c.stream, np, w, (bf16w*)wb);
    FH_HIP(hipGetLastError());
}
void nn_edge_weights(Ctx& c, const Bcsr& A, float* w) {
    FH_CHECK(A.prec == Prec::F64, -3, "edge weights need the FP64 operator");
    hipLaunchKernelGGL(k_nn_edge_weights, dim3(g1(A.nbr)), dim3(256), 0, c.stream, A.nbr, A.bs_r, A.rowptr.as<int>(),
                       A.colidx.as<int>(), A.vals.as<double>(), w);
    FH_HIP(hipGetLastError());
}
void nn_gather_index(Ctx& c, int64_t nnzb, const int* idx, const float* src, float* dst) {
    hipLaunchKernelGGL(k_nn_gather_index, dim3(g1(nnzb)), dim3(256), 0, c.stream, nnzb, idx, src, dst);
    FH_HIP(hipGetLastError());
}
void nn_select(Ctx& c, int64_t count, int nf, int slot_s1, int slot_s2, const double* delta, const double* r1,
               const double* invD, double omega, bool unit_step, double* z, int* counters, const double* r,
               const double* Adelta, double* Az) {
    hipLaunchKernelGGL(k_nn_select, dim3(g1(count)), dim3(256), 0, c.stream, count, nf, c.d_scalars, slot_s1, slot_s2,
                       delta, r1, invD, omega, (int)unit_step, z, counters, r, Adelta, Az);
    FH_HIP(hipGetLastError());
}

}  // namespace fh
