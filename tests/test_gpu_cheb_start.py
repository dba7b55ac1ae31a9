"""Chebyshev steps on scalar rows that form the vector they start from (a first
step from zero, the correction of a coarse level) against the two passes they
replace, bit for bit: while launches on a matrix are timed, its steps run as two
passes.  Rows in CSR below and above 4096 and in SELL-64, one to four steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
F = pytest.importorskip("fhhos4_amd")
G = F.fhgpu


@pytest.mark.parametrize("dim,mesh,n,csr", [(2, "quad", 8, False), (3, "hex", 6, False), (3, "stetra", 5, False),
                                            (3, "hex", 12, False), (3, "hex", 12, True), (2, "stri", 50, True)])
@pytest.mark.parametrize("degree", [1, 2, 4])
def test_cycle_is_that_of_two_passes(dim, mesh, n, csr, degree):
    print("case %s n=%d csr=%d cheb%d" % (mesh, n, csr, degree), flush=True)
    ctx = G.Context(0)
    P = G.HhoProblem(dim=dim, mesh=mesh, n=n, k=0, perturb=0.1, seed=3, kappa="lognormal", sigma=1.0)
    A = P.matrix(ctx, keep_host=True)
    assert A.info()["bs"] == 1
    r = torch.from_numpy(np.random.default_rng(n).standard_normal(P.n_unknowns)).cuda()
    if csr:
        A.set_sliced(False)
    kw = dict(solver="fcg", prec="aggregamg", nu=(1, 1), smoothers=("cheb%d" % degree,) * 2, max_coarse=40)
    s = G.Solver(ctx, **kw)
    s.setup(A)
    z, z2 = torch.empty_like(r), torch.empty_like(r)
    s.apply_prec(r, z)
    assert A.layout() == (4 if not csr and P.n_unknowns >= 4096 else 0)
    G.profile_begin(ctx, A, 1)
    s.apply_prec(r, z2)
    launches, _ = G.profile_end(ctx)
    assert launches > 0  # the finest level's residual: A is the level's matrix
    assert torch.equal(z, z2)
    s32 = G.Solver(ctx, mg_prec="f32", **kw)
    s32.setup(A)
    s32.apply_prec(r, z2)
    # FP32 rounding through the steps of two or three levels
    assert float(torch.linalg.norm(z - z2)) <= 1e-5 * float(torch.linalg.norm(z))
