"""Buffers that the assembly and the condensation take from released ones:
results do not depend on what such a buffer held before, results that are
alive keep their values."""
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
F = pytest.importorskip("fhhos4_amd")
G = F.fhgpu

KW = dict(dim=3, mesh="hex", k=2, perturb=0.15, source="modes", source_seed=3, source_modes=4, defer_assembly=True)


def _assemble(ctx, n, seed):
    A, b = G.HhoProblem(n=n, seed=seed, **KW).assemble_gpu(ctx)
    return A, A.blocks()[2].copy(), b.cpu().numpy()


@pytest.mark.parametrize("order", [(8, 8, 9, 8), (9, 8, 8, 9)])
def test_assembly_again(order):
    ctx = G.Context(0)
    first = {}
    held = None
    for n in order + order:
        A, v, b = _assemble(ctx, n, 7)
        if n in first:
            assert np.array_equal(first[n][0], v) and np.array_equal(first[n][1], b)
        first[n] = (v, b)
        if held is not None:  # the matrix before this one is still alive
            assert np.array_equal(held[0].blocks()[2], held[1])
        held = (A, v)


def test_condensation_again():
    ctx = G.Context(0)
    nc, nf, nfc, n = 4, 3, 6, 12
    ncell, m = n ** 3, nc + nf * nfc
    c = np.arange(ncell)[:, None]
    faces = np.hstack([3 * c + np.arange(3), 3 * ((c + 1) % ncell) + np.arange(3)]).astype(np.int32)
    nb = int(faces.max()) + 1
    want = {}
    for k in (0, 1, 0, 1):
        g = np.random.default_rng(k).standard_normal((ncell, m, m))
        loc = torch.from_numpy(g @ g.transpose(0, 2, 1) + m * np.eye(m)).cuda()
        M, b = G.condense_batched(ctx, faces, loc, nc, nf, nb, B_T=torch.ones(ncell, nc, dtype=torch.float64).cuda())
        v = M.blocks()[2].copy()
        if k in want:
            # a block of two cells is the sum of two terms in either order
            assert np.array_equal(want[k], v)
        want[k] = v


def _used():
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free, total


def test_kept_memory_is_bounded_and_released():
    ctx = G.Context(0)
    P = G.HhoProblem(dim=3, mesh="hex", n=20, k=3, perturb=0.15, seed=1, defer_assembly=True)
    gc.collect()  # nothing of other tests is released meanwhile
    P.assemble_gpu(ctx)  # what the first call sets up for good
    G.release_memory()
    used, total = _used()
    held = [P.assemble_gpu(ctx)[0] for _ in range(20)]  # 0.3 GB each
    assert _used()[0] - used > total // 72 + (1 << 29)
    del held
    torch.cuda.empty_cache()
    kept = _used()[0] - used
    slack = 64 << 20
    assert kept <= total // 72 + slack
    G.release_memory()
    assert _used()[0] - used <= slack
    G.release_memory()  # nothing left to free
