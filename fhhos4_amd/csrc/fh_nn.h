// Learned post-smoother of the flexible outer iteration: a small
// message-passing network over the face graph predicts, from the residual
// left by the multigrid cycle and the diffusion coefficients of the two
// cells of every face, a correction of the preconditioned vector.
//
// Network (hidden width H = 32, L message-passing layers):
//   v_i   = D_i^-1 r1_i                 (block-Jacobi image of the residual)
//   sigma = RMS(v),  u_i = v_i / sigma  (the network is applied to u: the
//                                        correction scales exactly with r1
//                                        for positive factors)
//   x0_i  = [u_i, f_i]                  (f_i: mean and half-difference of
//                                        log kappa of the face's two cells)
//   h0_i  = relu(We x0_i + be)
//   m_i   = sum_j w_ij h_j              (w_ij = |tr A_ij| / sum_k |tr A_ik|)
//   h_i  <- relu(S_l h_i + N_l m_i + c_l),  l = 1..L
//   delta_i = sigma (u_i + Wo h_i + bo)
// With Wo = 0 the correction is the undamped block-Jacobi step D^-1 r1.
//
// Training minimises the relative energy norm of the error left after the
// correction, (e1 - delta)^T A (e1 - delta) / e1^T A e1, over pairs
// (r1 = A e1, e1) generated by the plain solver.
#pragma once
#include <vector>

#include "fh_common.h"

namespace fh {

constexpr int kNnHidden = 32;
constexpr int kNnMaxLayers = 6;
// device scalar slots used by the network
constexpr int kNnSlotSigma = 481, kNnSlotS1 = 482, kNnSlotS2 = 483, kNnSlotE = 484,
              kNnSlotE0 = 485;

struct NnShape {
    int nf = 3, layers = 3;
    int din() const { return nf + 2; }
    // parameter offsets (floats)
    int64_t We() const { return 0; }
    int64_t be() const { return We() + (int64_t)kNnHidden * din(); }
    int64_t S(int l) const { return be() + kNnHidden + (int64_t)l * (2 * kNnHidden * kNnHidden + kNnHidden); }
    int64_t N(int l) const { return S(l) + kNnHidden * kNnHidden; }
    int64_t c(int l) const { return N(l) + kNnHidden * kNnHidden; }
    int64_t Wo() const { return S(layers); }
    int64_t bo() const { return Wo() + (int64_t)nf * kNnHidden; }
    int64_t total() const { return bo() + nf; }
};

// Graph data of one operator: edge weights of every stored block (and of
// the reverse edge, for the backward pass), face features, FP32 block
// inverses.  The block structure is the operator's (device arrays of A).
struct NnGraph {
    const Bcsr* A = nullptr;
    int n = 0, nf = 0;
    DevBuf w, wT, feat, invD32, invD64;
};
std::unique_ptr<NnGraph> nn_graph_create(Ctx& c, const Bcsr& A, const double* face_features);

class Mpnn {
public:
    Mpnn(Ctx& c, int nf, int layers, uint64_t seed);
    const NnShape& shape() const { return sh_; }
    void set_params(const float* p);
    void get_params(float* p) const;
    // Workspace for graphs of up to n nodes (no allocation afterwards).
    void reserve(int n);
    // delta = network correction of r1 (FP64 device vectors of n*nf); bf16
    // selects the BF16 copy of the weights (inference), else FP32 weights and
    // the activations are kept for a backward pass.
    void forward(const NnGraph& g, const double* r1, double* delta, bool bf16);
    // Relative energy error of the corrected vector and the gradient of it
    // (FP32, host, length total()) for one pair; no update.
    double loss_grad(const NnGraph& g, const double* r1, const double* e1, float* grad_host);
    // One Adam step on one pair; returns the loss before the step.
    double train_step(const NnGraph& g, const double* r1, const double* e1, float lr);

private:
    Ctx& c_;
    NnShape sh_;
    DevBuf p32_, p16_, grad_, m1_, m2_, partials_;
    int step_ = 0;
    int cap_ = 0;
    DevBuf v_, u_, x0_, gy_, h_, m_, dh_, diff_, Adiff_;
    struct Event {
        hipEvent_t e = nullptr;
        Event() { FH_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming)); }
        ~Event() { (void)hipEventDestroy(e); }
        Event(const Event&) = delete;
        Event& operator=(const Event&) = delete;
    } scalars_;  // loss_grad: the loss has reached the host
    // delta into out, or e1 - delta when e1 is not null
    void forward(const NnGraph& g, const double* r1, const double* e1, double* out, bool bf16);
    void backward(const NnGraph& g);
};

// ------------------------------------------------------------ launchers
// v = D^-1 r1 and partial sums of |v|^2, which nn_encode adds.
void nn_prep(Ctx& c, int n, int nf, const double* r1, const float* invD, float* v, double* partials);
void nn_encode(Ctx& c, int n, int nf, const double* partials, const float* v, const float* feat, int slot_sigma,
               const void* We, const void* be, bool bf16, float* u, float* x0, float* h);
void nn_layer(Ctx& c, int n, const int* rp, const int* ci, const float* w, const float* hin, const void* S,
              const void* N, const void* cb, bool bf16, float* hout, float* m_out);
// Gradient at a layer's input h from that at its output (after the relu).
void nn_layer_back(Ctx& c, int n, const int* rp, const int* ci, const float* wT, const float* dpre, const float* S,
                   const float* N, const float* h, float* dprev);
// delta, or e1 - delta when e1 is not null.
void nn_out(Ctx& c, int n, int nf, const float* h, const float* u, const void* Wo, const void* bo, bool bf16,
            int slot_sigma, const double* e1, double* delta);
void nn_out_back(Ctx& c, int n, int nf, const double* Adiff, int slot_e0, int slot_sigma, const float* Wo,
                 const float* h, float* gy, float* dh);
// Gradients of all parameters; dh: the gradients at the outputs of the encoder
// and the layers (n x 32 each), h their outputs, m the layers' aggregates.
void nn_weight_grads(Ctx& c, int n, const NnShape& sh, const float* gy, const float* dh, const float* h,
                     const float* m, const float* x0, double* partials, float* grad);
size_t nn_partials_bytes(const NnShape& sh);
void nn_adam(Ctx& c, int np, float* w, const float* g, float* m1, float* m2, float lr, float b1, float b2, float eps,
             int step, void* wb);
void nn_to_bf16(Ctx& c, int np, const float* w, void* wb);
void nn_edge_weights(Ctx& c, const Bcsr& A, float* w);
void nn_gather_index(Ctx& c, int64_t nnzb, const int* idx, const float* src, float* dst);
// z += alpha delta (accepted) or omega D^-1 r1 (block-Jacobi fallback); with
// Az, an accepted correction also writes A z = (r - r1) + alpha A delta.
void nn_select(Ctx& c, int64_t count, int nf, int slot_s1, int slot_s2, const double* delta, const double* r1,
               const double* invD, double omega, bool unit_step, double* z, int* counters,
               const double* r = nullptr, const double* Adelta = nullptr, double* Az = nullptr);

}  // namespace fh
