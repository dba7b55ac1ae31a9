"""Message-passing network at the edges of its tiles: fewer nodes than one
wavefront's 16, node counts that are no multiple of 16, 64 or 128, faces with 1
to 10 unknowns and rows of up to 11 edges (more than one batch of gathered
neighbours).

Tolerances: FP32 sums of at most 64 + 11 terms over the layers, relative to the
largest entry: 2 * 75 * 6e-8 per layer and a condition of the output of a few
units stay below 1e-4; the gradient passes through the layers twice."""
import numpy as np
import pytest

from oracle import oracle as O

torch = pytest.importorskip("torch")
F = pytest.importorskip("fhhos4_amd")
G = F.fhgpu
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh,n,k,layers", [("quad", 2, 0, 1), ("quad", 2, 3, 2), ("hex", 2, 1, 2), ("hex", 2, 3, 3),
                                             ("hex", 3, 2, 1), ("quad", 9, 1, 3), ("hex", 4, 0, 2)])
def test_network_matches_oracle(mesh, n, k, layers):
    print("case %s n=%d k=%d layers=%d" % (mesh, n, k, layers), flush=True)
    ctx = G.Context(0)
    P = G.HhoProblem(dim=3 if mesh == "hex" else 2, mesh=mesh, n=n, k=k, perturb=0.15, seed=3, kappa="lognormal",
                     sigma=1.0)
    A = P.matrix(ctx, keep_host=True)
    feat = G.face_features(P)
    g = G.NnGraph(ctx, A, feat)
    nn = G.Mpnn(ctx, P.nf, layers=layers, seed=11)
    rng = np.random.default_rng(6)
    p = nn.get_params()
    params = (p + 0.2 * rng.standard_normal(p.size)).astype(np.float32)
    nn.set_params(params)
    e1 = rng.standard_normal(P.n_unknowns)
    S = P.scipy()
    r1 = S @ e1
    ref = O.mpnn_forward(S, P.nf, feat, params.astype(np.float64), r1, layers=layers)
    d = torch.zeros(P.n_unknowns, dtype=torch.float64, device="cuda")
    nn.forward(g, torch.from_numpy(r1).cuda(), d, bf16=False)
    assert np.abs(d.cpu().numpy() - ref).max() <= 1e-4 * np.abs(ref).max()
    nn.forward(g, torch.from_numpy(r1).cuda(), d, bf16=True)
    assert np.linalg.norm(d.cpu().numpy() - ref) <= 3e-2 * np.linalg.norm(ref)
    loss_ref, grad_ref = O.mpnn_loss_grad(S, P.nf, feat, params.astype(np.float64), r1, e1, layers=layers)
    loss, grad = nn.loss_grad(g, torch.from_numpy(r1).cuda(), torch.from_numpy(e1).cuda())
    assert abs(loss - loss_ref) <= 1e-4 * abs(loss_ref)
    assert np.abs(grad - grad_ref).max() <= 2e-4 * np.abs(grad_ref).max()


def test_refused_pair_leaves_the_gradient_buffer():
    """A pair without energy is refused before anything is written to the
    caller's gradient, and the network works on as before."""
    import ctypes as C

    ctx = G.Context(0)
    P = G.HhoProblem(dim=2, mesh="quad", n=6, k=1, perturb=0.15, seed=3)
    g = G.NnGraph(ctx, P.matrix(ctx, keep_host=True), G.face_features(P))
    nn = G.Mpnn(ctx, P.nf, layers=2, seed=11)
    rng = np.random.default_rng(6)
    e1 = rng.standard_normal(P.n_unknowns)
    pair = [torch.from_numpy(v).cuda() for v in (P.scipy() @ e1, e1)]
    loss, grad = nn.loss_grad(g, *pair)
    zero = torch.zeros_like(pair[0])
    torch.cuda.synchronize()
    buf = np.full(nn.num_params(), 7.0, dtype=np.float32)
    value = C.c_double(7.0)
    for r, e in [(zero, zero), (zero, pair[1]), (-pair[0], pair[1])]:
        torch.cuda.synchronize()
        rc = G.lib().fh_nn_loss_grad(ctx.h, nn.h, g.h, r.data_ptr(), e.data_ptr(), C.byref(value), buf.ctypes.data)
        assert rc == -2 and value.value == 7.0
        assert np.all(buf == 7.0)
    loss2, grad2 = nn.loss_grad(g, *pair)
    assert loss2 == loss and np.array_equal(grad, grad2)


@pytest.mark.parametrize("solver", ["fcg", "cg"])
def test_network_set_after_setup_is_refused(solver):
    """Setup allocates what the learned post-smoother works on."""
    ctx = G.Context(0)
    P = G.HhoProblem(dim=2, mesh="quad", n=6, k=1, perturb=0.15, seed=3)
    A = P.matrix(ctx, keep_host=True)
    s = G.Solver(ctx, solver=solver, prec="bj")
    s.setup(A)
    s.set_learned_smoother(G.Mpnn(ctx, P.nf, layers=2, seed=11), G.NnGraph(ctx, A, G.face_features(P)))
    b = torch.from_numpy(P.rhs()).cuda()
    with pytest.raises(G.FhError, match="before Setup"):
        s.solve(b, torch.zeros_like(b))
