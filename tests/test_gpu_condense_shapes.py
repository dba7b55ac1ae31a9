"""Batched condensation and cell recovery over cell shapes and face graphs,
against dense numpy solves: the shapes of one wavefront per cell (smallest,
odd tile edges, 63 face unknowns), the shapes of the general kernels (another
number of cell unknowns, more face unknowns or faces), numbers of cells that do
not fill the last workgroup, and every kind of face: interior, eliminated, in
one cell, twice in one cell (sums of several contributions), in three cells.  A
face of three cells and cells of more than eight faces take the pattern built
on the host, all others the one built on the device.

Tolerance: a block entry is a sum of nc products per contribution after a
backward-stable solve with condition number below 2: 64 nc units in the last
place of the largest entry bound it amply."""
from fractions import Fraction

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


def _faces(rng, ncells, nfc, kind):
    """A ring-like graph: face f of cell c is shared with cell c + 1 for half
    of the faces; some faces eliminated; the special kinds change a few."""
    nfaces = 0
    faces = -np.ones((ncells, nfc), dtype=np.int32)
    for c in range(ncells):
        for j in range(nfc):
            if faces[c, j] != -1:
                continue
            if rng.random() < 0.15:
                continue  # eliminated
            faces[c, j] = nfaces
            if c + 1 < ncells and rng.random() < 0.6:
                free = np.nonzero(faces[c + 1] == -1)[0]
                if len(free):
                    faces[c + 1, rng.choice(free)] = nfaces
            nfaces += 1
    if nfaces == 0:
        faces[0, 0], nfaces = 0, 1
    if kind == "three" and ncells >= 3:
        faces[0, 0] = faces[1, 0] = faces[2, 0] = nfaces
        nfaces += 1
    if kind == "threes":  # every face in three cells or four
        for c in range(ncells):
            faces[c] = (c // 3 * nfc + np.arange(nfc)) % (nfc * max(1, ncells // 3))
        nfaces = int(faces.max()) + 1
    if kind == "twice" and nfc >= 2:
        faces[ncells // 2, :2] = nfaces
        nfaces += 1
    return faces, nfaces


CASES = [(nc, nf, nfc, n, "plain") for nc, nf, nfc, n in
         [(1, 1, 1, 1), (1, 1, 6, 5), (3, 2, 3, 9), (4, 3, 6, 6), (6, 3, 4, 7), (10, 6, 4, 3), (10, 4, 4, 10),
          (20, 10, 6, 4), (20, 10, 4, 5), (20, 9, 7, 3), (3, 2, 8, 11), (1, 16, 1, 3),
          (2, 2, 4, 3), (5, 3, 5, 3), (20, 10, 7, 2), (4, 3, 9, 3), (35, 15, 6, 3), (8, 4, 8, 5), (9, 3, 11, 3)]] + \
        [(4, 3, 6, 7, "threes"), (20, 10, 6, 9, "threes"), (4, 3, 6, 6, "three"), (10, 6, 4, 5, "twice"), (2, 3, 4, 5, "three"), (20, 10, 6, 3, "twice")]


@pytest.mark.parametrize("nc,nf,nfc,ncells,kind", CASES)
def test_condense_and_recover(ctx, nc, nf, nfc, ncells, kind):
    print("case nc=%d nf=%d nfc=%d cells=%d %s" % (nc, nf, nfc, ncells, kind), flush=True)
    rng = np.random.default_rng(nc * 1000 + nf * 10 + nfc)
    faces, nfaces = _faces(rng, ncells, nfc, kind)
    m = nfc * nf
    nl = nc + m
    R = rng.standard_normal((ncells, nl, nl))
    local = 0.5 * (R + R.transpose(0, 2, 1)) + nl * np.eye(nl)
    local[:, nc:, nc:] += 0.1 * rng.standard_normal((ncells, m, m))  # A_FF need not be symmetric
    local[:, nc:, :nc] = np.nan  # not read
    BT, BF = rng.standard_normal((ncells, nc)), rng.standard_normal((nfaces, nf))
    xF = rng.standard_normal(nfaces * nf)
    A = np.zeros((nfaces, nf, nfaces, nf))
    b = BF.copy()
    xT = np.zeros((ncells, nc))
    pairs = set()
    for c in range(ncells):
        TT, TF, FF = local[c, :nc, :nc], local[c, :nc, nc:], local[c, nc:, nc:]
        X = np.linalg.solve(TT, np.concatenate([TF, BT[c][:, None]], 1))
        S, y = FF - TF.T @ X[:, :m], TF.T @ X[:, m]
        xe = np.zeros(m)
        for i, f in enumerate(faces[c]):
            if f < 0:
                continue
            b[f] -= y[i * nf:(i + 1) * nf]
            xe[i * nf:(i + 1) * nf] = xF[f * nf:(f + 1) * nf]
            for j, g in enumerate(faces[c]):
                if g >= 0:
                    A[f, :, g, :] += S[i * nf:(i + 1) * nf, j * nf:(j + 1) * nf]
                    pairs.add((int(f), int(g)))
        xT[c] = np.linalg.solve(TT, BT[c] - TF @ xe)
    loc = torch.from_numpy(local).cuda()
    bt, bf = torch.from_numpy(BT.reshape(-1)).cuda(), torch.from_numpy(BF.reshape(-1)).cuda()
    M, bd = G.condense_batched(ctx, faces, loc, nc, nf, nfaces, B_T=bt, B_F=bf)
    rp, ci, v = M.blocks()
    got = [(r, int(c)) for r in range(nfaces) for c in ci[rp[r]:rp[r + 1]]]
    assert got == sorted(pairs)
    tol = 64 * nc * 2.3e-16
    ref = np.array([A[r, :, c, :] for r, c in got])
    assert np.abs(v - ref).max() <= tol * np.abs(ref).max()
    assert np.abs(bd.cpu().numpy().reshape(nfaces, nf) - b).max() <= tol * np.abs(b).max()
    got_xT = G.cell_recover_batched(ctx, faces, loc, nc, nf, nfaces, torch.from_numpy(xF).cuda(), B_T=bt).cpu().numpy()
    assert np.abs(got_xT - xT).max() <= tol * np.abs(xT).max()
    # no right-hand sides: the same operator (blocks of three contributions and
    # more in any order of the sum)
    M2, b2 = G.condense_batched(ctx, faces, loc, nc, nf, nfaces, rhs=False)
    assert b2 is None
    v2 = M2.blocks()[2]
    if kind == "plain":
        assert np.array_equal(v2, v)
    assert np.abs(v2 - ref).max() <= tol * np.abs(ref).max()
    z = G.cell_recover_batched(ctx, faces, loc, nc, nf, nfaces, torch.zeros(nfaces * nf, dtype=torch.float64,
                                                                              device="cuda"))
    assert float(z.abs().max()) == 0.0
    # a matrix that is not positive definite is refused
    loc[ncells - 1, nc - 1, nc - 1] = -1.0
    with pytest.raises(G.FhError, match="positive definite"):
        G.condense_batched(ctx, faces, loc, nc, nf, nfaces)
    with pytest.raises(G.FhError, match="positive definite"):
        G.cell_recover_batched(ctx, faces, loc, nc, nf, nfaces, torch.from_numpy(xF).cuda())


def _one_face_per_slot(rng, ncells, nfc, nc, nf):
    """Cells without common faces: every block has one contribution."""
    m = nfc * nf
    R = rng.standard_normal((ncells, nc + m, nc + m))
    local = 0.5 * (R + R.transpose(0, 2, 1)) + (nc + m) * np.eye(nc + m)
    return np.arange(ncells * nfc, dtype=np.int32).reshape(ncells, nfc), local


@pytest.mark.parametrize("nc,nf,nfc", [(1, 1, 2), (3, 2, 3), (4, 3, 6), (6, 3, 4), (10, 6, 4), (20, 10, 6), (5, 3, 5)])
def test_infinite_diagonal_drops_the_unknown(ctx, nc, nf, nfc):
    """A cell unknown whose diagonal entry is +Inf is eliminated with the value
    zero: every quotient by its pivot is zero."""
    print("case nc=%d nf=%d nfc=%d" % (nc, nf, nfc), flush=True)
    rng = np.random.default_rng(nc)
    ncells, m = nc, nfc * nf  # unknown c of cell c
    faces, local = _one_face_per_slot(rng, ncells, nfc, nc, nf)
    BT, BF, xF = rng.standard_normal((ncells, nc)), rng.standard_normal(ncells * m), rng.standard_normal(ncells * m)
    xT, b, S = np.zeros((ncells, nc)), BF.reshape(ncells, m).copy(), []
    for c in range(ncells):
        local[c, c, c] = np.inf
        keep = np.arange(nc) != c
        TT, TF = local[c, :nc, :nc][keep][:, keep], local[c, :nc, nc:][keep]
        S.append(local[c, nc:, nc:] - TF.T @ np.linalg.solve(TT, TF))
        b[c] -= TF.T @ np.linalg.solve(TT, BT[c, keep])
        xT[c, keep] = np.linalg.solve(TT, BT[c, keep] - TF @ xF[c * m:(c + 1) * m])
    loc, bt = torch.from_numpy(local).cuda(), torch.from_numpy(BT.reshape(-1)).cuda()
    M, bd = G.condense_batched(ctx, faces, loc, nc, nf, ncells * nfc, B_T=bt, B_F=torch.from_numpy(BF).cuda())
    v = M.blocks()[2].reshape(ncells, nfc, nfc, nf, nf).transpose(0, 1, 3, 2, 4).reshape(ncells, m, m)
    z = G.cell_recover_batched(ctx, faces, loc, nc, nf, ncells * nfc, torch.from_numpy(xF).cuda(), B_T=bt).cpu().numpy()
    tol = 64 * nc * 2.3e-16
    assert np.abs(v - np.array(S)).max() <= tol * np.abs(np.array(S)).max()
    assert np.abs(bd.cpu().numpy().reshape(ncells, m) - b).max() <= tol * np.abs(b).max()
    assert np.abs(z.reshape(ncells, nc) - xT).max() <= tol * max(np.abs(xT).max(), 1e-300)


@pytest.mark.parametrize("scale", [2.0 ** -1000, 2.0 ** 1000])
@pytest.mark.parametrize("nc,nf,nfc", [(4, 3, 6), (20, 10, 6)])
def test_power_of_four_scales_through(ctx, nc, nf, nfc, scale):
    """Scaled by a power of four, every square root, quotient and product of
    the algorithm is the unscaled one times a power of two, to the last bit."""
    print("case nc=%d nf=%d nfc=%d scale=%g" % (nc, nf, nfc, scale), flush=True)
    rng = np.random.default_rng(7)
    ncells, m = 32, nfc * nf
    faces, local = _one_face_per_slot(rng, ncells, nfc, nc, nf)
    # no entry so small that a scaled product would be subnormal
    local = np.where(local < 0, local - 0.5, local + 0.5)
    BT, BF, xF = rng.standard_normal((ncells, nc)), rng.standard_normal(ncells * m), rng.standard_normal(ncells * m)
    out = []
    for s in (1.0, scale):
        loc, bt, bf = (torch.from_numpy(s * a.reshape(-1)).cuda() for a in (local, BT, BF))
        M, bd = G.condense_batched(ctx, faces, loc, nc, nf, ncells * nfc, B_T=bt, B_F=bf)
        z = G.cell_recover_batched(ctx, faces, loc, nc, nf, ncells * nfc, torch.from_numpy(xF).cuda(), B_T=bt)
        out.append((M.blocks()[2] / s, bd.cpu().numpy() / s, z.cpu().numpy()))
    for a, w in zip(*out):
        assert np.array_equal(a, w)


@pytest.mark.parametrize("nc,nf,nfc", [(8, 4, 8), (9, 4, 8), (20, 8, 8), (35, 15, 6)])
def test_large_shapes_run_on_the_matrix_cores(ctx, nc, nf, nfc):
    """Shapes beyond one wavefront's with 32 face unknowns or more: with A_TT = I
    the solves are exact and a block entry is A_FF minus the product A_TF^T A_TF
    that the matrix instruction forms, a chain of fused multiply-adds over
    ascending cell unknowns.  Entry by entry the products are subtracted from
    A_FF one after the other, which rounds differently."""
    rng = np.random.default_rng(nc)
    m = nf * nfc
    local = rng.standard_normal((1, nc + m, nc + m))
    local[0, :nc, :nc] = np.eye(nc)
    T, FF = local[0, :nc, nc:], local[0, nc:, nc:]
    faces = np.arange(nfc, dtype=np.int32).reshape(1, nfc)
    M, _ = G.condense_batched(ctx, faces, torch.from_numpy(local).cuda(), nc, nf, nfc)
    v = M.blocks()[2].reshape(nfc, nfc, nf, nf).transpose(0, 2, 1, 3).reshape(m, m)
    same = 0
    for p, q in rng.integers(0, m, (200, 2)):
        acc, one = 0.0, float(FF[p, q])
        for k in range(nc):
            t = Fraction(T[k, p]) * Fraction(T[k, q])
            acc = float(t + Fraction(acc))
            one = float(Fraction(one) - t)
        assert v[p, q] == FF[p, q] - acc
        same += one == FF[p, q] - acc
    assert same < 200  # the two orders can be told apart
