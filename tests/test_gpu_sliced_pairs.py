"""Sliced block rows just below and above the number of slices from which a
wavefront takes two (32 768): quadrilaterals at k = 1, nine rows of two unknowns
a slice, so 294 144 rows make 32 683 slices and 295 680 rows 32 854, the last
one not full.

Tolerance: a row sums at most 14 products, 16 roundings of |A| |x| (FP64 2.2e-16,
FP32 6e-8 with the rounded values)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
F = pytest.importorskip("fhhos4_amd")
G = F.fhgpu


@pytest.mark.parametrize("n", [384, 385])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_products(n, prec):
    print("case quad n=%d k=1 %s" % (n, prec), flush=True)
    ctx = G.Context(0)
    P = G.HhoProblem(dim=2, mesh="quad", n=n, k=1, perturb=0.15, seed=2, defer_assembly=True)
    A, b = P.assemble_gpu(ctx, keep_host=True)
    S = A.scipy()
    M = A if prec == "f64" else A.convert("f32")
    dt, eps = (torch.float64, 2.3e-16) if prec == "f64" else (torch.float32, 6e-8)
    rng = np.random.default_rng(n)
    x = torch.from_numpy(rng.standard_normal(P.n_unknowns)).to(dt).cuda()
    r = torch.from_numpy(rng.standard_normal(P.n_unknowns)).to(dt).cuda()
    y, z = torch.empty_like(x), torch.empty_like(x)
    G.spmv(ctx, M, x, y)
    assert M.layout() == 1
    G.residual(ctx, M, r, x, z)
    xh, rh = x.cpu().numpy().astype(np.float64), r.cpu().numpy().astype(np.float64)
    ref, bound = S @ xh, 18 * eps * (abs(S) @ np.abs(xh) + np.abs(rh))
    assert np.all(np.abs(y.cpu().numpy() - ref) <= bound)
    assert np.all(np.abs(z.cpu().numpy() - (rh - ref)) <= bound)
