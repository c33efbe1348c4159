"""Bricks of more than one pencil along x or more than one step along y (Q1..Q3 applies): what a pencil or
a step carries to the next, in every kernel that has such bricks, against the oracle. The brick of a mesh is
the library's choice; the meshes here are ones that it gives the shape named."""
import ctypes as C
import os

import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import make_pair, rel_err

# degree, cells, {pencils, steps} of the kernel whose lanes are z planes of cells (Q3; mapped, residual, tangent)
PLANES = [(1, (33, 90, 34), (1, 2)), (1, (17, 60, 260), (2, 2)), (2, (17, 30, 50), (2, 1)), (2, (33, 90, 9), (1, 2)),
          (2, (17, 17, 260), (2, 2)), (3, (17, 60, 34), (2, 1)), (3, (9, 23, 180), (1, 2)), (3, (17, 17, 260), (2, 2))]
# degree, cells, {pencils, steps, cells of a pencil} of the kernel whose lanes are cells (Q1, Q2 Cartesian applies)
CELLS = [(1, (50, 23, 260), (2, 1, 16)), (1, (50, 90, 260), (2, 4, 16)), (1, (17, 90, 90), (1, 2, 8)),
         (2, (33, 23, 180), (1, 2, 16)), (2, (50, 23, 260), (2, 1, 16)), (2, (17, 90, 90), (1, 2, 8))]


def chosen(degree, nc):
    """choose_brick of the library's kernels.hpp"""
    import meltpooldg_amd as M
    brick, cells = (C.c_int * 2)(1, 1), (C.c_int * 3)(1, 1, 16)
    C.CDLL(M.LIB_PATH)._ZN4mpdg12choose_brickEiPKiPiS2_(degree, (C.c_int * 3)(*nc), brick, cells)
    return tuple(brick), tuple(cells)


def test_the_meshes_have_the_bricks_named():
    assert [chosen(k, nc)[0] for k, nc, _ in PLANES] == [b for _, _, b in PLANES]
    assert [chosen(k, nc)[1] for k, nc, _ in CELLS] == [b for _, _, b in CELLS]


def check_vmult(torch, degree, nc, seed, precision, **kw):
    orc, gop, _ = make_pair(torch, degree, nc, L=(1.0, 0.8, 1.3), precision=precision, seed=seed, **kw)
    x = torch.tensor(np.random.default_rng(seed + 1).uniform(-1.0, 1.0, orc.n_dofs),
                     dtype=torch.float64 if precision == 0 else torch.float32, device="cuda")
    y = torch.full_like(x, float("nan"))
    gop.vmult(y, x)
    torch.cuda.synchronize()
    assert rel_err(y.cpu().numpy(), orc.vmult(x.cpu().numpy().astype(np.float64))) < (1e-12 if precision == 0 else 1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("degree,nc,mode,dmask", [(k, nc, ("qp", "cell", "law")[i % 3], (0, 0b100100)[i % 2])
                                                  for i, (k, nc, _) in enumerate(PLANES[5:] + CELLS)])
def test_vmult(cuda, degree, nc, mode, dmask, precision):
    check_vmult(cuda, degree, nc, 71, precision, mode=mode, dirichlet=dmask)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("degree,nc", [(k, nc) for k, nc, _ in PLANES])
def test_mapped_vmult(cuda, degree, nc, precision):
    check_vmult(cuda, degree, nc, 73, precision, mode="cell" if nc[2] < 100 else "const", mapped=0.05)


@pytest.mark.gpu
@pytest.mark.parametrize("degree,nc,mode", [(k, nc, ("law", "qp", "cell")[i % 3]) for i, (k, nc, _) in enumerate(PLANES)])
def test_residual(cuda, degree, nc, mode):
    torch = cuda
    orc, gop, data = make_pair(torch, degree, nc, mode=mode, seed=75)
    rng = np.random.default_rng(76)
    T = data["T"].cpu().numpy() if mode == "law" else rng.uniform(0.0, 2.0, orc.n_dofs)
    T_old, q = T - 0.1 * rng.uniform(0.0, 1.0, orc.n_dofs), rng.uniform(0.0, 100.0, orc.n_dofs)
    r = torch.full((orc.n_dofs,), 0.5, dtype=torch.float64, device="cuda")  # create_rhs accumulates
    gop.create_rhs(r, *(torch.tensor(a, device="cuda") for a in (T, T_old, q)))
    torch.cuda.synchronize()
    assert rel_err(r.cpu().numpy(), orc.create_rhs(np.full(orc.n_dofs, 0.5), T, T_old, q)) < 1e-11


@pytest.mark.gpu
@pytest.mark.parametrize("degree,nc", [(k, nc) for k, nc, _ in PLANES])
def test_tangent(cuda, degree, nc):
    torch = cuda
    import meltpooldg_amd as M
    from tests.test_gpu_tangent import pair
    orc, op, *_ = pair(torch, M, degree, nc, tuple(0.1 * n for n in nc), 0b001000, True, (0.2, -0.4, 0.1))
    src = np.random.default_rng(77).uniform(-1.0, 1.0, orc.n_dofs)
    dst = torch.full((orc.n_dofs,), float("nan"), dtype=torch.float64, device="cuda")
    op.vmult(dst, torch.tensor(src, device="cuda"))
    assert rel_err(dst.cpu().numpy(), orc.vmult(src)) < 1e-12
    d = torch.empty_like(dst)
    op.compute_diagonal(d)
    assert rel_err(d.cpu().numpy(), orc.diagonal()) < 1e-12


# the smoothing steps that sum the planes shared by bricks; tolerances as for the oracle's V-cycle on small meshes
@pytest.mark.gpu
@pytest.mark.parametrize("precision,tol", [("FP64", 1e-9), ("FP32", 1e-4)])
@pytest.mark.parametrize("degree,nc", [(1, (40, 24, 20)), (2, (36, 20, 12)), (3, (36, 12, 20))])
def test_vcycle(cuda, degree, nc, precision, tol):
    torch = cuda
    import meltpooldg_amd as M
    assert min(nc) > 8  # several bricks in every direction
    orc, gop, _ = make_pair(torch, degree, nc, mode="qp", seed=78, dirichlet=0b010000)
    og = O.GMG(orc, nc_coarse=10, coarse_degree=1, cheb_degree=3, smoothing_range=20.0, eig_iters=20)
    pc = M.GMGPreconditioner(gop, precision=getattr(M, precision), n_cells_coarse=10, coarse_degree=1, smoother_degree=3,
                             smoothing_range=20.0, eig_cg_n_iterations=20)
    pc.update()
    assert [level[:2] for level in pc.levels()] == [level[:2] for level in og.levels()]
    b = np.random.default_rng(79).uniform(-1.0, 1.0, orc.n_dofs)
    out = torch.empty(orc.n_dofs, dtype=torch.float64, device="cuda")
    pc.vmult(out, torch.tensor(b, device="cuda"))
    torch.cuda.synchronize()
    assert rel_err(out.cpu().numpy(), og.vcycle(b)) < tol
