"""Timed workloads of the library, from the smallest call to the largest.

Every case is one use of the public Python API (fhhos4_amd.fhgpu and .gmg) on
systems of this repository's own families: hexahedra, quadrilaterals,
tetrahedra and Cartesian boxes, HHO degrees 0 to 3, per-cell lognormal kappa.

    listed()             the standing cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what a program holds before the call, on the GPU
    run(state)           one pass, with its outputs
    work(case)           bytes and operations one pass cannot do without
    tolerance(case)      largest difference between two correct results
    exact(case, seed)    the outputs in 64 bits by plain torch, or None

kind        a pass
product     y = A x or r = b - A x: every Krylov iteration and residual test
smooth      block-Jacobi or multicolour Gauss-Seidel sweeps from zero
precond     z = M r with one geometric multigrid cycle
solve       b -> x with CG / FCG and a multigrid, to 1e-8
condense    element matrices -> face system, then the cells' unknowns
assemble    mesh -> face operator and right-hand side
network     the learned post-smoother: a correction, or a loss gradient
"""
import ctypes
import math

import numpy as np
import torch

from fhhos4_amd import fhgpu as G
from fhhos4_amd import gmg

DEV = "cuda"


# ----------------------------------------------------------------- the cases
def listed():
    return [
        # a small 2-D Poisson solve, as a time step or a parameter study calls
        # it thousands of times: latency and launches count
        dict(name="solve_cart2d_n32_k1", kind="solve", mesh="cart", dim=2, n=32, k=1, prec="gmg", mode="f64"),
        # the benchmark's solver (FCG(4), p-first aggregation AMG) on a member
        # of its family that a workstation-sized study uses
        dict(name="solve_hex_n32_k3_f64", kind="solve", mesh="hex", dim=3, n=32, k=3, prec="amg", mode="f64"),
        # the same with the FP32 multigrid and FCG's FP32-stored product, the
        # fastest setting of the benchmark, on the largest mesh listed here
        dict(name="solve_hex_n64_k3_mixed", kind="solve", mesh="hex", dim=3, n=64, k=3, prec="amg", mode="mixed"),
        # one FP32 geometric multigrid cycle: a preconditioner inside the
        # caller's own Krylov loop
        dict(name="precond_cart_n32_k2_f32", kind="precond", mesh="cart", dim=3, n=32, k=2, store="f32"),
        # the fine-level product of the headline family, bandwidth-bound
        dict(name="spmv_hex_n64_k3_f64", kind="product", mesh="hex", dim=3, n=64, k=3, store="f64", op="spmv"),
        # a residual on tetrahedra with BF16-stored values and FP32 vectors
        dict(name="residual_tet_n23_k2_bf16", kind="product", mesh="stetra", dim=3, n=23, k=2, store="bf16",
             op="residual"),
        # block-Jacobi sweeps on an odd number of quadrilaterals (n_f = 3)
        dict(name="jacobi_quad_n181_k2_f64", kind="smooth", mesh="quad", dim=2, n=181, k=2, store="f64",
             method="jacobi"),
        # one symmetric multicolour Gauss-Seidel sweep on tetrahedra
        dict(name="gs_tet_n16_k1_f64", kind="smooth", mesh="stetra", dim=3, n=16, k=1, store="f64", method="gs"),
        # a program with element matrices of its own: condensation, then the
        # recovery of the cell unknowns
        dict(name="condense_hex_n24_k3", kind="condense", mesh="hex", dim=3, n=24, k=3),
        # the headline family's operator from the mesh: paid once per system
        dict(name="assemble_hex_n24_k3", kind="assemble", mesh="hex", dim=3, n=24, k=3),
        # the learned post-smoother: inference inside FCG (BF16 weights)
        dict(name="network_forward_hex_n32_k3", kind="network", mesh="hex", dim=3, n=32, k=3, pas="forward"),
        # and one training pair's loss and gradient (FP32 weights)
        dict(name="network_grad_hex_n16_k3", kind="network", mesh="hex", dim=3, n=16, k=3, pas="grad"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "precond", "product", "product", "smooth", "condense", "condense", "assemble",
                       "assemble", "network"])
    c = dict(kind=kind)
    if kind == "solve":
        if rng.random() < 0.4:
            # meshes that coarsen to at most a thousand unknowns
            c.update(mesh="cart", dim=2, n=rng.choice([24, 28, 32, 40, 48, 56, 64, 80, 96, 128]),
                     k=rng.randint(1, 2), prec="gmg", mode="f64")
        else:
            c.update(mesh="hex", dim=3, n=_log_int(rng, 9, 56), k=rng.randint(1, 3), prec="amg",
                     mode=rng.choice(["f64", "f32", "mixed"]))
    elif kind == "precond":
        c.update(mesh="cart", dim=3, n=rng.choice([8, 12, 16, 20, 24, 28, 32]), k=rng.randint(1, 2),
                 store=rng.choice(["f64", "f32", "bf16"]))
    elif kind == "product":
        mesh, dim, hi = rng.choice([("hex", 3, 60), ("stetra", 3, 32), ("quad", 2, 400), ("stri", 2, 300)])
        c.update(mesh=mesh, dim=dim, n=_log_int(rng, 5, hi), k=rng.randint(0 if mesh == "hex" else 1, 3),
                 store=rng.choice(["f64", "f32"] if mesh == "hex" else ["f64", "f32", "bf16"]),
                 op=rng.choice(["spmv", "residual"]))
        if mesh == "stetra":
            c["k"] = min(c["k"], 2)
    elif kind == "smooth":
        mesh, dim, hi = rng.choice([("hex", 3, 24), ("stetra", 3, 20), ("quad", 2, 300), ("stri", 2, 200)])
        c.update(mesh=mesh, dim=dim, n=_log_int(rng, 5, hi), k=rng.randint(1, 2), store=rng.choice(["f64", "f32"]),
                 method=rng.choice(["jacobi", "gs"]))
    elif kind == "condense":
        mesh, dim, hi = rng.choice([("hex", 3, 23), ("stetra", 3, 14), ("quad", 2, 150), ("stri", 2, 120)])
        c.update(mesh=mesh, dim=dim, n=_log_int(rng, 4, hi), k=rng.randint(0, 3))
        if mesh == "stetra":
            c["k"] = min(c["k"], 2)
    elif kind == "assemble":
        mesh, dim, hi = rng.choice([("hex", 3, 23), ("quad", 2, 150)])
        c.update(mesh=mesh, dim=dim, n=_log_int(rng, 4, hi), k=rng.randint(0, 3))
    else:
        pas = rng.choice(["forward", "grad"])
        mesh, dim, hi = rng.choice([("hex", 3, 30 if pas == "forward" else 15),
                                    ("quad", 2, 250 if pas == "forward" else 70)])
        c.update(mesh=mesh, dim=dim, n=_log_int(rng, 5, hi), k=rng.randint(1, 3), pas=pas)
    return c


# ------------------------------------------------------------------- helpers
def _problem(case, seed):
    """The case's mesh and coefficients (the system is assembled on the GPU)."""
    kw = dict(dim=case["dim"], mesh=case["mesh"], n=case["n"], k=case["k"], seed=seed + 1, source="pisine",
              defer_assembly=True)
    if case["kind"] == "precond":
        # piecewise-constant kappa on subdomains of four cells
        kw.update(kappa="subdomain", sigma=2.0, subdomain=4)
    elif case["kind"] == "solve" and case["prec"] == "gmg":
        kw.update(kappa="one", source="modes", source_seed=seed + 1, source_modes=8)
    elif case["mesh"] == "stetra" or case["mesh"] == "stri":
        kw.update(perturb=0.1, kappa="lognormal", sigma=1.0)
    else:
        kw.update(perturb=0.15, kappa="lognormal", sigma=3.0)
    return G.HhoProblem(**kw)


def _rand(seed, *shape, dtype=torch.float64):
    g = torch.Generator(device=DEV).manual_seed(1000003 * (seed + 1))
    return torch.randn(*shape, generator=g, dtype=dtype, device=DEV)


class _View:
    """Device memory of a matrix as a tensor, without a copy; the matrix
    lives as long as the tensor."""

    def __init__(self, owner, ptr, n, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=(n,), typestr=typestr, data=(ptr, False), version=2)


def _device_arrays(A):
    """(row pointers, block columns, FP64 values) of A in device memory."""
    i = A.info()
    p = [ctypes.c_void_p() for _ in range(3)]
    if G.lib().fh_mat_device_arrays(A.h, *[ctypes.byref(t) for t in p]) < 0:
        raise RuntimeError("no device arrays")
    size = (i["nbr"] + 1, i["nnzb"], i["nnzb"] * i["bs"] ** 2)
    return [torch.as_tensor(_View(A, q.value, n, t), device=DEV) for q, n, t in zip(p, size, ("<i4", "<i4", "<f8"))]


def _tuned_args(mode):
    """The benchmark's solver: FCG(4) with the p-first aggregation AMG."""
    kw = dict(solver="fcg", prec="aggregamg", cycle="K", kcycle_levels=2, nu=(1, 0), coarse_nu=(1, 1),
              smoothers=("cheb1", "cheb1"), coarse_smoother="cheb4", theta=0.1, max_coarse=2500, tol=1e-8,
              max_iter=1000, fcg_truncation=4)
    if mode != "f64":
        kw.update(mg_prec="f32", mg_store="f32")
    if mode == "mixed":
        kw.update(outer_prec="f32", replace_every=12)
    return kw


def _cell_faces(P):
    """Block row of every face of every cell (-1: an eliminated face), faces
    of a cell in the order of their numbers."""
    fc = P.face_cells()
    nfc = {"hex": 6, "cart": 6 if P.args["dim"] == 3 else 4, "quad": 4, "stetra": 4, "stri": 3}[P.args["mesh"]]
    cells = fc.reshape(-1)
    faces = np.repeat(np.arange(P.nb, dtype=np.int32), 2)
    ok = cells >= 0
    cells, faces = cells[ok], faces[ok]
    order = np.argsort(cells, kind="stable")
    cells, faces = cells[order], faces[order]
    first = np.searchsorted(cells, np.arange(P.info["ncells"]))
    out = np.full((P.info["ncells"], nfc), -1, dtype=np.int32)
    out[cells, np.arange(len(cells)) - first[cells]] = faces
    return out


def _sizes(dim, k):
    """Cell, reconstruction and face unknowns of degree k."""
    c = lambda d, p: math.comb(p + d, d)
    return c(dim, k), c(dim, k + 1), c(dim - 1, k)


def _counts(case):
    """Cells, faces per cell, unknown faces, stored blocks of the mesh."""
    n, dim, mesh = case["n"], case["dim"], case["mesh"]
    if mesh in ("hex", "cart", "quad"):
        nb = dim * n ** (dim - 1) * (n - 1)
        # faces of a cell inside the domain, per axis: 2, or 1 at either end
        ways = {2: n - 2, 1: 2} if n > 1 else {0: 1}
        tot, acc = {0: 1}, None
        for _ in range(dim):
            acc = {}
            for s, w in tot.items():
                for f, v in ways.items():
                    acc[s + f] = acc.get(s + f, 0) + w * v
            tot = acc
        return n ** dim, 2 * dim, nb, sum(w * s * s for s, w in tot.items()) - nb
    if mesh == "stetra":
        nb = 12 * n ** 3 - 6 * n ** 2
        return 6 * n ** 3, 4, nb, 7 * nb - 36 * n ** 2
    nb = 3 * n ** 2 - 2 * n
    return 2 * n ** 2, 3, nb, 5 * nb - 8 * n


# ------------------------------------------------------------------- prepare
def prepare(case, seed):
    ctx = G.Context(0)
    s = dict(case=case, ctx=ctx)
    kind = case["kind"]
    P = _problem(case, seed)
    s["P"] = P
    if kind == "solve" and case["prec"] == "gmg":
        H = gmg.build_hierarchy(ctx, P)
        s["H"], s["A"], s["b"] = H, H[0][1], P.b_device
        s["solver"] = G.Solver(ctx, solver="cg", prec="mg", cycle="V", nu=(1, 1), smoothers=("bj23", "bj23"),
                               tol=1e-8, max_iter=500)
        gmg.attach(s["solver"], H)
        s["solver"].setup(s["A"])
        s["x"] = torch.zeros_like(s["b"])
    elif kind == "solve":
        s["A"], s["b"] = P.assemble_gpu(ctx)
        s["solver"] = G.Solver(ctx, **_tuned_args(case["mode"]))
        s["solver"].setup(s["A"])
        s["x"] = torch.zeros_like(s["b"])
    elif kind == "precond":
        s["H"] = H = gmg.build_hierarchy(ctx, P)
        s["A"] = H[0][1]
        mg = {} if case["store"] == "f64" else dict(mg_prec="f32", mg_store=case["store"])
        s["solver"] = G.Solver(ctx, solver="fcg", prec="mg", cycle="V", nu=(2, 2), smoothers=("bj", "bj"), relax=0.5,
                               **mg)
        gmg.attach(s["solver"], H)
        s["solver"].setup(s["A"])
        s["r"] = _rand(seed, P.n_unknowns)
        s["z"] = torch.zeros_like(s["r"])
    elif kind == "product":
        A, b = P.assemble_gpu(ctx)
        s["A"] = A if case["store"] == "f64" else A.convert(case["store"])
        dt = torch.float64 if case["store"] == "f64" else torch.float32
        s["x"], s["b"] = _rand(seed, P.n_unknowns, dtype=dt), b.to(dt)
        s["y"] = torch.empty_like(s["x"])
    elif kind == "smooth":
        A, b = P.assemble_gpu(ctx)
        dt = torch.float64 if case["store"] == "f64" else torch.float32
        s["A64"] = A
        s["A"] = A if case["store"] == "f64" else A.convert("f32")
        s["bj"] = G.BlockJacobi(ctx, A, omega=0.5 if case["method"] == "jacobi" else 1.0, dprec=case["store"])
        s["b"] = _rand(seed, P.n_unknowns, dtype=dt)
        s["x"], s["work"] = torch.zeros_like(s["b"]), torch.zeros_like(s["b"])
        if case["method"] == "gs":
            s["col"] = G.Colouring(ctx, A)
    elif kind == "condense":
        nc, _, nf = _sizes(case["dim"], case["k"])
        s["faces"] = _cell_faces(P)
        ncell, nfc = s["faces"].shape
        nl = nc + nfc * nf
        R = _rand(seed, ncell, nl, nl)
        s["local"] = (0.5 * (R + R.transpose(1, 2)) + nl * torch.eye(nl, dtype=R.dtype, device=DEV)).contiguous()
        s["nc"], s["nf"] = nc, nf
        s["BT"], s["BF"] = _rand(seed + 1, ncell * nc), _rand(seed + 2, P.nb * nf)
        s["xF"] = _rand(seed + 3, P.nb * nf)
    elif kind == "network":
        A, _ = P.assemble_gpu(ctx)
        s["A"], s["graph"] = A, G.NnGraph(ctx, A, G.face_features(P))
        s["nn"] = G.Mpnn(ctx, P.nf, layers=3, seed=seed + 1)
        s["nn"].set_params(_weights(s["nn"], seed))
        s["e1"] = _rand(seed, P.n_unknowns)
        s["r1"] = torch.empty_like(s["e1"])
        G.spmv(ctx, A, s["e1"], s["r1"])
        s["delta"] = torch.empty_like(s["r1"])
    torch.cuda.synchronize()
    return s


def _weights(nn, seed):
    """Weights of a network in training: the initial ones, moved a little (the
    initial output layer is zero)."""
    g = np.random.default_rng(seed)
    return (nn.get_params() + 0.05 * g.standard_normal(nn.num_params())).astype(np.float32)


# ----------------------------------------------------------------------- run
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "solve":
        s["solver"].solve(s["b"], s["x"])
        return s["x"]
    if kind == "precond":
        s["solver"].apply_prec(s["r"], s["z"])
        return s["z"]
    if kind == "product":
        if case["op"] == "spmv":
            G.spmv(s["ctx"], s["A"], s["x"], s["y"])
        else:
            G.residual(s["ctx"], s["A"], s["b"], s["x"], s["y"])
        return s["y"]
    if kind == "smooth":
        if case["method"] == "jacobi":
            s["bj"].sweep(s["b"], s["x"], s["work"], nsweeps=3, x_is_zero=True, A=s["A"])
        else:
            s["x"].zero_()
            G.mcgs_sweep(s["ctx"], s["A"], s["bj"], s["col"], 2, s["b"], s["x"])
        return s["x"]
    if kind == "condense":
        nb = s["P"].nb
        M, b = G.condense_batched(s["ctx"], s["faces"], s["local"], s["nc"], s["nf"], nb, B_T=s["BT"], B_F=s["BF"])
        xT = G.cell_recover_batched(s["ctx"], s["faces"], s["local"], s["nc"], s["nf"], nb, s["xF"], B_T=s["BT"])
        rp, ci, vals = _device_arrays(M)
        return dict(rowptr=rp, colidx=ci, vals=vals, b=b, xT=xT)
    if kind == "assemble":
        A, b = s["P"].assemble_gpu(s["ctx"])
        rp, ci, vals = _device_arrays(A)
        return dict(rowptr=rp, colidx=ci, vals=vals, b=b)
    if case["pas"] == "forward":
        s["nn"].forward(s["graph"], s["r1"], s["delta"], bf16=True)
        return s["delta"]
    loss, grad = s["nn"].loss_grad(s["graph"], s["r1"], s["e1"])
    return dict(loss=loss, grad=grad)


# ---------------------------------------------------------------------- work
def work(case):
    ncell, nfc, nb, nnzb = _counts(case)
    nc, nr, nf = _sizes(case["dim"], case["k"])
    kind, m, N = case["kind"], nfc * nf, nb * nf
    sv = {"f64": 8, "f32": 4, "bf16": 2}[case.get("store", "f64")]
    sx = 8 if sv == 8 else 4
    # the operator once: the blocks and their columns, or, where fewer, the
    # symmetric cell matrices and their faces
    op = lambda v: min(nnzb * (nf * nf * v + 4), ncell * (m * (m + 1) // 2 * v + 4 * nfc))
    flops = 2.0 * nnzb * nf * nf
    if kind == "product":
        return dict(bytes=op(sv) + N * sx * (2 if case["op"] == "spmv" else 3), flops=flops)
    if kind == "smooth":
        sweeps = 2
        extra = nb * nf * nf * sx + 2 * N * sx
        return dict(bytes=sweeps * op(sv) + 3 * extra, flops=sweeps * flops + 6.0 * nb * nf * nf)
    if kind == "precond":
        # three residuals, three block-Jacobi passes and the transfers on the
        # finest level, an eighth of that on each level below
        one = 4 * op(sv) + 4 * nb * nf * nf * sx + 12 * N * sx + 2 * N * 8
        return dict(bytes=one * 8 // 7, flops=5.0 * flops)
    if kind == "solve":
        if case["prec"] == "gmg":
            its, vis = 14, 4.0 / 3.0
            one = 3 * op(8) + 2 * nb * nf * nf * 8 + 20 * N * 8
            return dict(bytes=its * one * vis, flops=its * 4.0 * flops)
        its = 55
        so, sm = (8, 8) if case["mode"] == "f64" else ((8, 4) if case["mode"] == "f32" else (4, 4))
        # an iteration: FCG's product, the first-mode residual and the
        # block-Jacobi step of the finest level, about 40 passes over the
        # scalar face level and those below it, the vectors
        one = op(so) + nnzb * (nf * sm + 4) + nb * nf * nf * sm + 24 * N * 8 + 25 * nnzb * (sm + 4)
        return dict(bytes=its * one, flops=its * (flops * 1.2 + 60.0 * nnzb))
    nl = nc + m
    if kind == "condense":
        by = ncell * (nl * nl - nc * m + nc * nc + nc * m + 3 * nc) * 8 + nnzb * (nf * nf * 8 + 4) + 3 * N * 8
        fl = ncell * (2.0 * m * m * nc + 2 * nc ** 3 / 3.0 + 2.0 * nc * nc * (m + 2) + 4.0 * nc * m)
        return dict(bytes=by, flops=fl)
    if kind == "assemble":
        q, qf, nh = (case["k"] + 2) ** case["dim"], (case["k"] + 2) ** (case["dim"] - 1), nl
        fl = 2.0 * ncell * (q * (nr * nr / 2 * case["dim"] + nc * nr) + nfc * qf * (nr * (nf + nc) + nf * (nf + nr)) +
                            nr ** 3 / 6 + nr * nr * nh + nr * nh * nh / 2 + nc * (nr + nc) * nh +
                            nfc * nf * nh * (nr + nc + nf + nh / 2) + nc * nc * m + nc * m * m / 2)
        return dict(bytes=ncell * (8 * 24 + 100 + 8 * (m * (m + 1) // 2)) + nnzb * (nf * nf * 8 + 4) + N * 8, flops=fl)
    # network: activations of 32 channels, the edges, three layers
    H = 32
    fwd = nb * (nf * nf * 4 + nf * 20) + 3 * (2 * nb * H * 4 + nnzb * 8) + nb * H * 4
    ffl = 2.0 * nb * (nf * nf + H * (nf + 2) + 3 * 2 * H * H + nf * H) + 3 * 2.0 * nnzb * H
    if case["pas"] == "forward":
        return dict(bytes=fwd, flops=ffl)
    return dict(bytes=3 * fwd + op(8) + 5 * N * 8, flops=3 * ffl + flops)


# ----------------------------------------------------------------- tolerance
def tolerance(case):
    """About four times the largest difference seen between this library and
    exact() over the ranges above (MI355X), in the 2-norm."""
    kind, f64 = case["kind"], case.get("store", "f64") == "f64"
    if kind == "product":
        return {"rel": 4e-15 if f64 else 1e-6}  # seen 7e-16; FP32 sums 3e-7 (BF16 values are inputs)
    if kind == "smooth":
        return {"rel": 2e-15 if f64 else 4e-7}  # seen 3e-16; 8e-8
    if kind == "precond":
        return {"rel": 1e-15 if f64 else 4e-7}  # seen 2e-16; 7e-8
    if kind == "solve":
        # two solves that stop at ||r|| < 1e-8 ||b||: rounding alone moves x
        # by up to 6e-11, a stop one iteration apart by up to 2e-9
        return {"rel": 4e-9}
    if kind == "condense":
        return {"rel": 2e-15}  # seen 4e-16
    if kind == "assemble":
        return {"rel": 4e-14}  # seen 9e-15 (coefficients of neighbouring cells differ by e^6)
    if case["pas"] == "forward":
        return {"rel": 5e-3}  # seen 1.2e-3: activations rounded to BF16
    return {"rel": 2e-6}  # seen 4e-7: FP32 activations and sums


# --------------------------------------------------------------------- exact
class _Blocks:
    """Block rows in 64 bits on the device, and their plain products."""

    def __init__(self, A):
        i = A.info()
        self.bs, self.nbr = i["bs"], i["nbr"]
        rp, ci, v = _device_arrays(A)
        self.ci = ci.long()
        self.row = torch.repeat_interleave(torch.arange(self.nbr, device=DEV), (rp[1:] - rp[:-1]).long())
        self.v = v.view(-1, self.bs, self.bs)

    def __matmul__(self, x):
        y = torch.zeros(self.nbr, self.bs, dtype=torch.float64, device=DEV)
        X = x.view(-1, self.bs)
        for a in range(0, len(self.ci), 1 << 20):
            e = slice(a, a + (1 << 20))
            y.index_add_(0, self.row[e], (self.v[e] * X[self.ci[e]][:, None, :]).sum(-1))
        return y.view(-1)

    def inverse_diagonal(self):
        d = torch.nonzero(self.row == self.ci)[:, 0]
        out = torch.empty(self.nbr, self.bs, self.bs, dtype=torch.float64, device=DEV)
        out[self.row[d]] = torch.linalg.inv(self.v[d])
        return out

    def dense(self):
        nbc = int(self.ci.max()) + 1
        D = torch.zeros(self.nbr, nbc, self.bs, self.bs, dtype=torch.float64, device=DEV)
        D[self.row, self.ci] = self.v
        return D.permute(0, 2, 1, 3).reshape(self.nbr * self.bs, nbc * self.bs)


def _apply_blocks(D, r):
    return (D * r.view(-1, 1, D.shape[2])).sum(-1).view(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "solve" and _counts(case)[2] * _sizes(case["dim"], case["k"])[2] > 16000:
        return None  # a direct solution takes too long
    s = prepare(case, seed) if kind in ("condense", "network", "smooth") else None
    P = s["P"] if s else _problem(case, seed)
    ctx = s["ctx"] if s else G.Context(0)
    if kind == "solve":
        A, b = P.assemble_gpu(ctx)
        return torch.linalg.solve(_Blocks(A).dense(), b)
    if kind == "product":
        A, b = P.assemble_gpu(ctx)
        B = _Blocks(A)
        x = _rand(seed, P.n_unknowns, dtype=torch.float64 if case["store"] == "f64" else torch.float32).double()
        if case["store"] != "f64":
            b = b.float().double()
            if case["store"] == "bf16":
                B.v = B.v.float().bfloat16().double()
            elif case["mesh"] != "hex":
                B.v = B.v.float().double()
        return B @ x if case["op"] == "spmv" else b - B @ x
    if kind == "smooth":
        B, b = _Blocks(s["A64"]), s["b"].double()
        D = B.inverse_diagonal()
        if case["store"] != "f64":
            B.v = B.v.float().double()
        x = torch.zeros_like(b)
        if case["method"] == "jacobi":
            for _ in range(3):
                x = x + 0.5 * _apply_blocks(D, b - B @ x)
            return x
        nco, colour = s["col"].get()
        colour = torch.from_numpy(colour).to(DEV)
        X = x.view(-1, B.bs)
        for c in list(range(nco)) + list(range(nco - 1, -1, -1)):
            z = _apply_blocks(D, b - B @ x).view(-1, B.bs)
            X[colour == c] += z[colour == c]
        return x
    if kind == "precond":
        return _vcycle(gmg.build_hierarchy(ctx, P), _rand(seed, P.n_unknowns), case["store"])
    if kind == "condense":
        return _condense_exact(s)
    if kind == "assemble":
        if P.info["redraws"]:
            return None  # the mesh kept its vertices off the plain draw
        return _assemble_exact(case, P)
    return _network_exact(s, case["pas"])


def _vcycle(H, r, store):
    """One V(2,2) cycle from zero with block Jacobi (omega = 1/2), R = P^T;
    the products use the values as the multigrid stores them."""
    ops = []
    for _, A, P in H:
        p = None
        if P is not None:
            rp, ci, v = P.blocks()
            bs = v.shape[1]
            row = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
            p = [torch.from_numpy(t).to(DEV) for t in (row, ci.astype(np.int64), v)] + [bs]
        ops.append((_Blocks(A), p))

    def cycle(l, b):
        B, p = ops[l]
        if p is None:
            return torch.linalg.solve(B.dense(), b)
        D = B.inverse_diagonal()
        if store == "bf16":
            B.v = B.v.float().bfloat16().double()
        x = 0.5 * _apply_blocks(D, b)
        x = x + 0.5 * _apply_blocks(D, b - B @ x)
        row, col, v, bs = p
        res = (b - B @ x).view(-1, bs)
        rc = torch.zeros(ops[l + 1][0].nbr, bs, dtype=torch.float64, device=DEV)
        rc.index_add_(0, col, (v * res[row][:, :, None]).sum(1))
        e = cycle(l + 1, rc.view(-1)).view(-1, bs)
        dx = torch.zeros(B.nbr, bs, dtype=torch.float64, device=DEV)
        dx.index_add_(0, row, (v * e[col][:, None, :]).sum(2))
        x = x + dx.view(-1)
        for _ in range(2):
            x = x + 0.5 * _apply_blocks(D, b - B @ x)
        return x

    return cycle(0, r)


def _scatter(faces, nb, nf, S, F, bF):
    """Face system of cell matrices S (cells x m x m) and vectors F."""
    ncell, nfc = faces.shape
    f = torch.as_tensor(faces, device=DEV).long()
    key = f[:, :, None] * nb + f[:, None, :]
    ok = (f[:, :, None] >= 0) & (f[:, None, :] >= 0)
    uniq, inv = torch.unique(key[ok], return_inverse=True)
    B = S.view(ncell, nfc, nf, nfc, nf).permute(0, 1, 3, 2, 4)[ok]
    vals = torch.zeros(len(uniq), nf, nf, dtype=torch.float64, device=DEV).index_add_(0, inv, B)
    rowptr = torch.zeros(nb + 1, dtype=torch.int64, device=DEV)
    rowptr[1:] = torch.cumsum(torch.bincount(uniq // nb, minlength=nb), 0)
    b = bF.clone().view(nb, nf).index_add_(0, f[f >= 0], F.view(ncell, nfc, nf)[f >= 0])
    return dict(rowptr=rowptr.int(), colidx=(uniq % nb).int(), vals=vals.view(-1), b=b.view(-1))


def _condense_exact(s):
    nc, nf, nb, faces = s["nc"], s["nf"], s["P"].nb, s["faces"]
    L, BT = s["local"], s["BT"].view(-1, nc, 1)
    TT, TF, FF = L[:, :nc, :nc].contiguous(), L[:, :nc, nc:].contiguous(), L[:, nc:, nc:].contiguous()
    X = torch.linalg.solve(TT, torch.cat([TF, BT], 2))
    FT = TF.transpose(1, 2).contiguous()
    out = _scatter(faces, nb, nf, FF - FT @ X[:, :, :-1].contiguous(), -(FT @ X[:, :, -1:].contiguous())[:, :, 0],
                   s["BF"])
    f = torch.as_tensor(faces, device=DEV).long()
    xf = torch.where((f >= 0)[:, :, None], s["xF"].view(nb, nf)[f.clamp(min=0)], 0.0).reshape(len(f), -1, 1)
    out["xT"] = torch.linalg.solve(TT, BT - TF @ xf)[:, :, 0]
    return out


def _legendre(p, x):
    """Legendre polynomials 0..p at x and their derivatives (last axis)."""
    L, D = [torch.ones_like(x)], [torch.zeros_like(x)]
    for q in range(1, p + 1):
        L.append(x if q == 1 else ((2 * q - 1) * x * L[-1] - (q - 1) * L[-2]) / q)
        D.append((2 * q - 1) * L[q - 1] + (D[q - 2] if q > 1 else 0.0))
    return torch.stack(L, -1), torch.stack(D, -1)


def _vertices(P):
    """Grid vertices moved by the seeded uniform draw of the mesh."""
    a = P.args
    n, dim = a["n"], a["dim"]
    ax = [np.arange(n + 1)] * dim
    idx = np.stack([g.reshape(-1) for g in np.meshgrid(*ax, indexing="ij")][::-1], 1)  # x fastest
    X = np.zeros((len(idx), 3))
    X[:, :dim] = idx * (1.0 / n)
    inner = np.all((idx > 0) & (idx < n), 1)
    gid = np.arange(len(idx), dtype=np.uint64)
    with np.errstate(over="ignore"):
        for d in range(dim):
            key = np.uint64(a["seed"]) * np.uint64(0x100000001B3) ^ (gid * np.uint64(4) + np.uint64(d))
            r = key + np.uint64(0x9E3779B97F4A7C15)
            r = (r ^ (r >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
            r = (r ^ (r >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
            r = r ^ (r >> np.uint64(31))
            u = (r >> np.uint64(11)).astype(np.float64) * (2.0 / 9007199254740992.0) - 1.0
            X[inner, d] += a["perturb"] / n * u[inner]
    return torch.from_numpy(X).to(DEV)


def _assemble_exact(case, P):
    """HHO on bilinear / trilinear cells in plain batched torch: tensor
    Legendre bases, Gauss rules of k + 2 points, the saddle-point
    reconstruction, the two-sided stabilisation and the condensation."""
    n, dim, k, nb = case["n"], case["dim"], case["k"], P.nb
    nc, nr, nf = _sizes(dim, k)
    V = _vertices(P)
    kappa = torch.from_numpy(P.cell_kappa()).to(DEV)
    ncell = n ** dim
    ijk = torch.stack([(torch.arange(ncell, device=DEV) // n ** d) % n for d in range(dim)], 1)
    vid = lambda off: sum((ijk[:, d] + off[d]) * (n + 1) ** d for d in range(dim))
    corner = torch.stack([vid([(c >> d) & 1 for d in range(dim)]) for c in range(2 ** dim)], 1)
    # unknown faces: cell by cell its +x, +y (, +z) interface inside the domain
    up = torch.stack([ijk[:, d] < n - 1 for d in range(dim)], 1)
    num = torch.where(up, torch.cumsum(up.reshape(-1).long(), 0).view(-1, dim) - 1, -1)
    faces = torch.full((ncell, 2 * dim), -1, dtype=torch.long, device=DEV)
    for d in range(dim):
        faces[:, 2 * d + 1] = num[:, d]
        low = ijk[:, d] > 0
        faces[low, 2 * d] = num[torch.nonzero(low)[:, 0] - n ** d, d]
    gx, gw = (torch.from_numpy(t).to(DEV) for t in np.polynomial.legendre.leggauss(k + 2))
    grid = lambda t, d: torch.stack([g.reshape(-1) for g in torch.meshgrid(*[t] * d, indexing="ij")][::-1], 1)
    if dim == 2:
        rexp = [(a, d - a) for d in range(k + 2) for a in range(d, -1, -1)]
        fexp = [(d,) for d in range(k + 1)]
    else:
        rexp = [(a, b, d - a - b) for d in range(k + 2) for a in range(d, -1, -1) for b in range(d - a, -1, -1)]
        fexp = [(d - j, j) for d in range(k + 1) for j in range(d + 1)]

    def shape(xi):
        """Corner shape functions at xi (points x dim) and their gradients."""
        N, dN = [], []
        for c in range(2 ** dim):
            f = [0.5 * (1 + (1 if (c >> d) & 1 else -1) * xi[:, d]) for d in range(dim)]
            g = [0.5 * (1 if (c >> d) & 1 else -1) for d in range(dim)]
            N.append(math.prod(f))
            dN.append(torch.stack([g[d] * math.prod([f[e] for e in range(dim) if e != d], start=torch.ones_like(f[0]))
                                   for d in range(dim)], -1))
        return torch.stack(N, 0), torch.stack(dN, 0)

    def basis(x, ctr, hw):
        """psi (cells x points x nr) and its gradient (.. x dim)."""
        LD = [_legendre(k + 1, (x[..., d] - ctr[:, None, d]) / hw[:, None, d]) for d in range(dim)]
        psi = torch.stack([math.prod([LD[d][0][..., e[d]] for d in range(dim)]) for e in rexp], -1)
        g = [torch.stack([math.prod([LD[a][1][..., e[a]] / hw[:, None, a] if a == d else LD[a][0][..., e[a]]
                                     for a in range(dim)]) for e in rexp], -1) for d in range(dim)]
        return psi, torch.stack(g, -1)

    S_all = torch.empty(ncell, 2 * dim * nf, 2 * dim * nf, dtype=torch.float64, device=DEV)
    F_all = torch.empty(ncell, 2 * dim * nf, dtype=torch.float64, device=DEV)
    qc, wc = grid(gx, dim), math.prod(grid(gw, dim).unbind(1))
    Nc, dNc = shape(qc)
    qf, wf = grid(gx, dim - 1), math.prod(grid(gw, dim - 1).unbind(1))
    Lf = [_legendre(k, qf[:, d])[0] for d in range(dim - 1)]
    phi = torch.stack([math.prod([Lf[d][:, e[d]] for d in range(dim - 1)]) for e in fexp], -1)
    for c0 in range(0, ncell, 2048):
        e = slice(c0, min(ncell, c0 + 2048))
        C = V[corner[e]][..., :dim]
        kap = kappa[e]
        ctr, hw = C.mean(1), 0.5 * (C.amax(1) - C.amin(1))
        bmm = lambda a, b: torch.matmul(a.contiguous(), b.contiguous())
        x = torch.einsum("cp,ncd->npd", Nc, C)
        J = torch.einsum("cpq,ncr->nprq", dNc, C)
        wd = wc * torch.linalg.det(J)
        psi, g = basis(x, ctr, hw)
        f = dim * math.pi ** 2 * torch.sin(math.pi * x).prod(-1)
        S = sum(bmm((g[..., d] * (wd * kap[:, None])[..., None]).transpose(1, 2), g[..., d]) for d in range(dim))
        M = bmm((psi[..., :nc] * wd[..., None]).transpose(1, 2), psi)
        Lm = (psi * wd[..., None]).sum(1)
        BT = (psi[..., :nc] * (wd * f)[..., None]).sum(1)
        nh = nc + 2 * dim * nf
        B = torch.zeros(len(C), nr, nh, dtype=torch.float64, device=DEV)
        B[:, :, :nc] = S[:, :, :nc]
        traces = []
        for fc in range(2 * dim):
            axis, side = fc // 2, fc % 2
            tang = [d for d in range(dim) if d != axis]
            def at(q):
                full = torch.empty(len(q), dim, dtype=torch.float64, device=DEV)
                full[:, axis] = 2.0 * side - 1.0
                for j, d in enumerate(tang):
                    full[:, d] = q[:, j]
                N, dN = shape(full)
                xs = torch.einsum("cp,ncd->npd", N, C)
                t = torch.einsum("cpq,ncr->nprq", dN[:, :, tang], C)
                if dim == 2:
                    nv = torch.stack([t[..., 1, 0], -t[..., 0, 0]], -1)
                else:
                    nv = torch.linalg.cross(t[..., 0], t[..., 1], dim=-1)
                return xs, nv
            x0, nv0 = at(torch.zeros(1, dim - 1, dtype=torch.float64, device=DEV))
            sg = torch.where((nv0[:, 0] * (x0[:, 0] - ctr)).sum(-1) < 0, -1.0, 1.0)
            ring = [[-1.0], [1.0]] if dim == 2 else [[-1.0, -1.0], [1.0, -1.0], [1.0, 1.0], [-1.0, 1.0]]
            xr, _ = at(torch.tensor(ring, dtype=torch.float64, device=DEV))
            hF = (torch.roll(xr, -1, 1) - xr).norm(dim=-1).amax(1)
            xs, nv = at(qf)
            nv = nv * sg[:, None, None]
            ps, gs = basis(xs, ctr, hw)
            kgn = kap[:, None, None] * (gs * nv[:, :, None, :]).sum(-1)
            wk = (kgn * wf[:, None]).transpose(1, 2)
            B[:, :, nc + fc * nf:nc + (fc + 1) * nf] = bmm(wk, phi.expand(len(C), -1, -1))
            B[:, :, :nc] -= bmm(wk, ps[..., :nc])
            wa = (phi * (wf * nv.norm(dim=-1))[..., None]).transpose(1, 2)
            traces.append((bmm(wa, phi.expand(len(C), -1, -1)), bmm(wa, ps), kap / hF))
        R = torch.zeros_like(B)
        R[:, 1:] = torch.linalg.solve(S[:, 1:, 1:].contiguous(), B[:, 1:].contiguous())
        R[:, 0] = -(Lm[:, 1:, None] * R[:, 1:]).sum(1)
        R[:, 0, :nc] += Lm[:, :nc]
        R[:, 0] /= Lm[:, :1]
        A = bmm(R.transpose(1, 2), bmm(S, R))
        Dt = torch.linalg.solve(M[:, :, :nc].contiguous(), bmm(M, R))
        Dt[:, torch.arange(nc), torch.arange(nc)] -= 1.0
        for fc, (Mf, Tf, coef) in enumerate(traces):
            Pf = torch.linalg.solve(Mf, Tf)
            D = bmm(Pf, R) - bmm(Pf[:, :, :nc], Dt)
            j = torch.arange(nf)
            D[:, j, nc + fc * nf + j] -= 1.0
            A = A + coef[:, None, None] * bmm(D.transpose(1, 2), bmm(Mf, D))
        X = torch.linalg.solve(A[:, :nc, :nc].contiguous(), torch.cat([A[:, :nc, nc:], BT[:, :, None]], 2))
        FT = A[:, :nc, nc:].transpose(1, 2)
        S_all[e] = A[:, nc:, nc:] - bmm(FT, X[:, :, :-1])
        F_all[e] = -bmm(FT, X[:, :, -1:])[:, :, 0]
    zero = torch.zeros(nb * nf, dtype=torch.float64, device=DEV)
    return _scatter(faces.cpu().numpy(), nb, nf, S_all, F_all, zero)


def _network_exact(s, pas):
    """The network in 64 bits (its weights rounded as inference stores them),
    the gradient of the relative energy error by autograd."""
    B, nf, H = _Blocks(s["A"]), s["P"].nf, 32
    nb = B.nbr
    p = torch.from_numpy(s["nn"].get_params()).to(DEV)
    if pas == "forward":
        p = p.bfloat16()
    p = p.double().requires_grad_(pas == "grad")
    pos = [0]

    def take(*shape):
        a = pos[0]
        pos[0] += math.prod(shape)
        return p[a:pos[0]].view(*shape)

    tr = B.v.diagonal(dim1=1, dim2=2).sum(-1).abs() * (B.row != B.ci)
    tot = torch.zeros(nb, dtype=torch.float64, device=DEV).index_add_(0, B.row, tr)
    w = torch.where(tot[B.row] > 0, tr / tot[B.row].clamp(min=1e-300), 0.0)
    v = _apply_blocks(B.inverse_diagonal(), s["r1"]).view(nb, nf)
    sigma = (v * v).mean().sqrt()
    u = v / sigma
    x = torch.cat([u, torch.from_numpy(G.face_features(s["P"])).to(DEV)], 1)
    We, be = take(H, nf + 2), take(H)
    h = torch.relu(x @ We.t() + be)
    for _ in range(3):
        Sl, Nl, cl = take(H, H), take(H, H), take(H)
        m = torch.zeros_like(h).index_add(0, B.row, w[:, None] * h[B.ci])
        h = torch.relu(h @ Sl.t() + m @ Nl.t() + cl)
    Wo, bo = take(nf, H), take(nf)
    delta = (sigma * (u + h @ Wo.t() + bo)).reshape(-1)
    if pas == "forward":
        return delta
    e1, r1 = s["e1"], s["r1"]
    e = e1 - delta.detach()
    Ae = B @ e
    E0 = (e1 * r1).sum()
    delta.backward(-2.0 * Ae / E0)
    return dict(loss=float((e * Ae).sum() / E0), grad=p.grad.cpu().numpy())
