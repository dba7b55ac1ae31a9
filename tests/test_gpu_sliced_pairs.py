"""Sliced block rows just below and above the number of slices from which a
wavefront takes two (32 768).

Products and residuals on quadrilaterals at k = 1: nine rows of two unknowns a
slice, so 294 144 rows make 32 683 slices and 295 680 rows 32 854, the last one
not full.  Tolerance: a row sums at most 14 products, 16 roundings of |A| |x|
(FP64 2.2e-16, FP32 6e-8 with the rounded values).

Every operation on block rows of the other block sizes, odd ones, with the
inverse blocks distributed over the lanes and not, and in two parts of short and
long rows; values in FP64, FP32 and BF16.  Tolerance: a row sums at most 70
products with diagonally dominant blocks, so 128 roundings of the largest entry
bound an operation amply; a cycle with two Chebyshev steps before and after its
correction stays within sixteen operations' roundings."""
import numpy as np
import pytest
import scipy.sparse as sp

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


def _rows(nf, widths, nbr, seed):
    """Blocks of nbr rows: row i has widths[i % len(widths)] of them, the
    diagonal one included (symmetric values are not needed here)."""
    rng = np.random.default_rng(seed)
    i = np.arange(nbr)[:, None]
    off = np.array([0, 1, -1, 37, -37, 4099, -4099][:max(widths)])
    cols = (i + off) % nbr
    w = np.asarray(widths)[np.arange(nbr) % len(widths)]
    cols[np.arange(len(off))[None, :] >= w[:, None]] = nbr  # past the row
    cols.sort(axis=1)
    keep = cols < nbr
    rp = np.concatenate([[0], np.cumsum(w)])
    ci = cols[keep]
    v = rng.uniform(-1, 1, (len(ci), nf, nf)).astype(np.float32).astype(np.float64)
    v[ci == np.repeat(np.arange(nbr), w)] += 2 * nf * max(widths) * np.eye(nf)
    return rp, ci, v


# n_f, blocks per row, block rows; a slice has min(64 / lanes of a row, 64 / n_f) rows
FORMS = [(3, [5], 4 * 32768 + 5),       # odd n_f, inverse blocks distributed (4 rows x 9 lanes)
         (3, [2], 10 * 32768 + 3),      # odd n_f, not distributed (10 x 9 > 64)
         (6, [7], 3 * 32768 + 2),       # three rows of 21 lanes, distributed
         (6, [3], 7 * 32768 + 1),       # seven rows of 9 lanes, not distributed
         (10, [6], 2 * 32768 + 1),      # 30 lanes a row
         (4, [1], 16 * 32768 + 1),      # one block a row
         (2, [2, 7], 2 * 32 * 32768 + 2)]  # two parts: short and long rows by a map


@pytest.mark.parametrize("nf,widths,nbr", FORMS)
def test_operations_on_two_slices(nf, widths, nbr):
    print("case nf=%d widths=%s rows=%d" % (nf, widths, nbr), flush=True)
    ctx = G.Context(0)
    rp, ci, v = _rows(nf, widths, nbr, nf)
    A = G.Matrix.from_blocks(ctx, nbr, nf, rp, ci, v)
    S = sp.bsr_matrix((v, ci, rp), shape=(nbr * nf, nbr * nf))
    D = v[ci == np.repeat(np.arange(nbr), np.diff(rp))]
    rng = np.random.default_rng(nf)
    x, b = (rng.uniform(-1, 1, nbr * nf).astype(np.float32).astype(np.float64) for _ in range(2))
    for store in ["f64", "f32"] + (["bf16"] if nf % 2 == 0 else []):
        M = A if store == "f64" else A.convert(store)
        dt, eps = (torch.float64, 2.3e-16) if store == "f64" else (torch.float32, 6e-8)
        T = S
        if store == "bf16":
            T = sp.bsr_matrix((torch.from_numpy(v).to(torch.bfloat16).double().numpy(), ci, rp), shape=S.shape)
        Ax = T @ x
        tol = 128 * eps
        xd, bd = torch.from_numpy(x).to(dt).cuda(), torch.from_numpy(b).to(dt).cuda()
        y = torch.empty_like(xd)
        G.spmv(ctx, M, xd, y)
        assert M.layout() == (2 if len(widths) > 1 else 1)
        assert np.abs(y.cpu().numpy() - Ax).max() <= tol * np.abs(Ax).max()
        y = xd.clone()
        G.spmv(ctx, M, xd, y, alpha=0.5, beta=-2.0)
        assert np.abs(y.cpu().numpy() - (0.5 * Ax - 2 * x)).max() <= tol * np.abs(Ax).max()
        G.residual(ctx, M, bd, xd, y)
        assert np.abs(y.cpu().numpy() - (b - Ax)).max() <= tol * np.abs(Ax).max()
        bj = G.BlockJacobi(ctx, A, omega=0.7, dprec="f64" if store == "f64" else "f32")
        z = np.linalg.solve(D, (b - Ax).reshape(nbr, nf, 1)).reshape(-1)
        y = xd.clone()
        bj.sweep(bd, y, torch.empty_like(y), nsweeps=1, A=M)
        ref = x + 0.7 * z
        # the residual's rounding passes through D^-1 (entries of about 1 / 2 n_f w)
        assert np.abs(y.cpu().numpy() - ref).max() <= tol * np.abs(ref).max()


@pytest.mark.parametrize("nf,widths,nbr", [f for f in FORMS if f[0] != 4])
@pytest.mark.parametrize("store", ["f64", "f32"])
def test_chebyshev_steps_on_two_slices(nf, widths, nbr, store):
    """A two-level cycle with Chebyshev steps on the finest level, on the sliced
    rows against the block rows."""
    print("case nf=%d widths=%s rows=%d %s" % (nf, widths, nbr, store), flush=True)
    ctx = G.Context(0)
    A = G.Matrix.from_blocks(ctx, nbr, nf, *_rows(nf, widths, nbr, nf))
    nc = 64  # coarse level: the first unknowns of the first rows
    i = np.arange(nc)
    P = G.Matrix.from_blocks(ctx, nc, nf, np.minimum(np.arange(nbr + 1), nc), i, np.tile(np.eye(nf), (nc, 1, 1)))
    Ac = G.Matrix.from_blocks(ctx, nc, nf, np.arange(nc + 1), i, np.tile(4.0 * np.eye(nf), (nc, 1, 1)))
    r = torch.randn(nbr * nf, dtype=torch.float64, device="cuda")

    def cycle(prec):
        s = G.Solver(ctx, solver="fcg", prec="mg", nu=(1, 1), smoothers=("cheb2", "cheb2"), max_coarse=nc * nf,
                     mg_prec=prec)
        s.set_level(0, None, P)
        s.set_level(1, Ac)
        s.setup(A)
        z = torch.empty_like(r)
        s.apply_prec(r, z)
        return z

    z = cycle(store)
    if store == "f64":
        assert A.layout() == (2 if len(widths) > 1 else 1)
    A.set_sliced(False)
    ref = cycle("f64")
    assert float((z - ref).abs().max()) <= 16 * 128 * (2.3e-16 if store == "f64" else 6e-8) * float(ref.abs().max())
