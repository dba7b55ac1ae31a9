"""GPU assembly of general cells (bilinear quadrilaterals, trilinear
hexahedra), every dimension and degree, on the smallest meshes and on one
whose cells do not fill the last wavefront of any loop: block values and
right-hand side against the host assembly of the same problem, the element
layout against the block rows, and the GPU post-processing against the host's.

Tolerance: both sides form the operator from the same integrals by different
orders of sums and factorisations; with neighbouring coefficients e^6 apart
their difference stays below 1e-12 of the largest block entry (the entries
themselves agree to 1e-14 with a 64-bit reference of the same formulas)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
F = pytest.importorskip("fhhos4_amd")
G = F.fhgpu


@pytest.fixture(scope="module")
def ctx():
    assert torch.cuda.is_available(), "no ROCm device visible"
    return G.Context(0)


@pytest.mark.parametrize("mesh,n", [("quad", 2), ("quad", 7), ("hex", 2), ("hex", 3)])
@pytest.mark.parametrize("k", [0, 1, 2, 3])
def test_assembly_matches_host(ctx, mesh, n, k):
    print("case %s n=%d k=%d" % (mesh, n, k), flush=True)
    kw = dict(dim=3 if mesh == "hex" else 2, mesh=mesh, n=n, k=k, perturb=0.15, seed=5 + k, kappa="lognormal",
              sigma=3.0, source="modes", source_seed=3, source_modes=4)
    H = G.HhoProblem(**kw)
    P = G.HhoProblem(defer_assembly=True, **kw)
    A, b = P.assemble_gpu(ctx, keep_host=True)
    rp, ci, v = H.blocks()
    rp2, ci2, v2 = A.blocks()
    assert np.array_equal(rp, rp2) and np.array_equal(ci, ci2)
    assert np.abs(v - v2).max() <= 1e-12 * np.abs(v).max()
    bh = H.rhs()
    assert np.abs(bh - b.cpu().numpy()).max() <= 1e-12 * np.abs(bh).max()
    # symmetric up to the same rounding
    D = A.scipy()
    assert abs(D - D.T).max() <= 1e-12 * np.abs(v).max()
    x = torch.from_numpy(np.random.default_rng(k).standard_normal(P.n_unknowns)).cuda()
    if A.layout() == 5:
        y, y2 = torch.empty_like(x), torch.empty_like(x)
        G.spmv(ctx, A, x, y)
        A.set_elem(False)
        G.spmv(ctx, A, x, y2)
        assert float((y - y2).abs().max()) <= 1e-13 * float(np.abs(v).max()) * 60
    e, eh = P.l2_error_gpu(ctx, x), H.l2_error(x.cpu().numpy())
    assert abs(e - eh) <= 1e-10 * eh
