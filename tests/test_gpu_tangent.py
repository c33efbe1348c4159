"""GPU parity of the full Newton tangent (temperature-dependent liquid/solid material and a
prescribed velocity, heat_diffuse_operator.cpp:1028-1056): apply, diagonal and residual against
the oracle, GMRES against the oracle's solution, and the reference's golden norm sequences of the
velocity and velocity + solidification cases run through HeatDiffuseOperation with GMRES."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_oracle import MUSHY, TANGENT_GOLDEN

pytestmark = pytest.mark.gpu

GPU_MUSHY = dict(conductivity=MUSHY["k"], specific_heat=MUSHY["cp"], density=MUSHY["rho"],
                 solidus=MUSHY["T_solidus"], liquidus=MUSHY["T_liquidus"])
DT = 0.01


def pair(torch, M, degree, nc, L, dmask, solid, vel, seed=0):
    """Oracle and GPU operators with the tangent at a temperature field that crosses the mushy interval."""
    rng = np.random.default_rng(seed)
    orc = O.Operator(degree, nc, L, dirichlet_mask=dmask)
    X = orc.node_coords()
    T = 1970.0 + 6.0 * np.sin(7 * X[0] + 1.0) * np.cos(5 * X[1]) + 2.0 * X[2] + 0.1 * rng.standard_normal(orc.n_dofs)
    T_old = T - 0.4 * np.cos(4 * X[0]) - 0.05 * rng.standard_normal(orc.n_dofs)
    orc.set_tangent(DT, material=MUSHY, velocity=vel, do_solidification=solid, T_old=T_old)
    orc.set_T(T)
    op = M.HeatDiffuseMultiPhaseOperator(degree, nc, L, dirichlet_faces=dmask)
    op.reset_time_increment(DT)
    op.set_tangent(GPU_MUSHY, velocity=vel, do_solidification=solid)
    Td, Tod = (torch.tensor(a, device="cuda") for a in (T, T_old))
    op.bind_temperature(Td, Tod)
    return orc, op, T, T_old, Td, Tod


CASES = [(1, (5, 4, 3), (0.5, 0.4, 0.3), 0, True, (-0.3, 0.1, 0.05)),
         (2, (3, 4, 2), (0.3, 0.4, 0.2), 0b000011, True, (0.2, -0.4, 0.1)),
         (3, (3, 2, 2), (0.3, 0.2, 0.2), 0, False, (-0.5, 0.0, 0.0)),
         (4, (2, 2, 3), (0.2, 0.2, 0.3), 0b110000, True, (0.0, 0.3, -0.2)),
         (2, (7, 5, 6), (0.7, 0.5, 0.6), 0b001100, True, (0.1, 0.1, 0.1)),
         # rows of cells longer than one block (several segments, the last one partial);
         # without velocity and/or without solidification
         (3, (20, 2, 2), (2.0, 0.2, 0.2), 0b000001, True, (0.0, 0.0, 0.0)),
         (1, (70, 2, 1), (0.7, 0.2, 0.1), 0, False, (0.0, 0.0, 0.0)),
         (4, (13, 2, 2), (0.65, 0.1, 0.1), 0b000010, True, (0.2, 0.0, -0.1)),
         (2, (30, 2, 1), (0.6, 0.04, 0.02), 0, False, (0.0, 0.1, 0.0))]


@pytest.mark.parametrize("degree,nc,L,dmask,solid,vel", CASES)
def test_tangent_vmult_matches_oracle(cuda, degree, nc, L, dmask, solid, vel):
    torch = cuda
    import meltpooldg_amd as M
    orc, op, *_ = pair(torch, M, degree, nc, L, dmask, solid, vel)
    src = np.random.default_rng(1).uniform(-1, 1, orc.n_dofs)
    dst = torch.empty(orc.n_dofs, dtype=torch.float64, device="cuda")
    op.vmult(dst, torch.tensor(src, device="cuda"))
    ref = orc.vmult(src, threads=1)
    assert np.linalg.norm(dst.cpu().numpy() - ref) <= 1e-12 * np.linalg.norm(ref)


@pytest.mark.parametrize("degree,nc,L,dmask,solid,vel", CASES[:4] + CASES[5:])
def test_tangent_diagonal_and_residual_match_oracle(cuda, degree, nc, L, dmask, solid, vel):
    torch = cuda
    import meltpooldg_amd as M
    orc, op, T, T_old, Td, Tod = pair(torch, M, degree, nc, L, dmask, solid, vel, seed=3)
    d = torch.empty(orc.n_dofs, dtype=torch.float64, device="cuda")
    op.compute_diagonal(d)
    ref = orc.diagonal()
    assert np.linalg.norm(d.cpu().numpy() - ref) <= 1e-12 * np.linalg.norm(ref)
    q = np.random.default_rng(4).uniform(0, 100, orc.n_dofs)
    r = torch.full((orc.n_dofs,), 0.5, dtype=torch.float64, device="cuda")  # create_rhs accumulates
    op.create_rhs(r, Td, Tod, torch.tensor(q, device="cuda"))
    ref = orc.create_rhs(np.full(orc.n_dofs, 0.5), T, T_old, q)
    assert np.linalg.norm(r.cpu().numpy() - ref) <= 1e-11 * np.linalg.norm(ref)


FIELD_CASES = [(1, (5, 4, 3), (0.5, 0.4, 0.3), 0, True),
               (2, (3, 4, 2), (0.3, 0.4, 0.2), 0b000011, True),
               (3, (20, 2, 2), (2.0, 0.2, 0.2), 0b000001, False),
               (4, (13, 2, 2), (0.65, 0.1, 0.1), 0b110000, True)]


@pytest.mark.parametrize("degree,nc,L,dmask,solid", FIELD_CASES)
def test_tangent_velocity_field_matches_oracle(cuda, degree, nc, L, dmask, solid):
    """Velocity DoF field (heat_diffuse_operator.cpp:975-978, :449-452): apply, diagonal and residual
    against the oracle; None restores the constant vector given to set_tangent."""
    torch = cuda
    import meltpooldg_amd as M
    vel = (0.1, -0.2, 0.05)
    orc, op, T, T_old, Td, Tod = pair(torch, M, degree, nc, L, dmask, solid, vel, seed=7)
    X = orc.node_coords()
    vf = np.concatenate([-0.3 + 0.8 * X[1] * X[2], 0.2 * np.sin(9 * X[0]), 0.1 + 0.5 * X[0] - 0.3 * X[2] ** 2])
    orc.set_tangent(DT, material=MUSHY, do_solidification=solid, T_old=T_old, velocity_field=vf)
    vfd = torch.tensor(vf, device="cuda")
    op.set_velocity_field(vfd)
    op.bind_temperature(Td, Tod)
    src = np.random.default_rng(8).uniform(-1, 1, orc.n_dofs)
    dst = torch.empty(orc.n_dofs, dtype=torch.float64, device="cuda")
    op.vmult(dst, torch.tensor(src, device="cuda"))
    ref = orc.vmult(src, threads=1)
    assert np.linalg.norm(dst.cpu().numpy() - ref) <= 1e-12 * np.linalg.norm(ref)
    d = torch.empty(orc.n_dofs, dtype=torch.float64, device="cuda")
    op.compute_diagonal(d)
    ref = orc.diagonal()
    assert np.linalg.norm(d.cpu().numpy() - ref) <= 1e-12 * np.linalg.norm(ref)
    q = np.random.default_rng(9).uniform(0, 100, orc.n_dofs)
    r = torch.full((orc.n_dofs,), 0.5, dtype=torch.float64, device="cuda")
    op.create_rhs(r, Td, Tod, torch.tensor(q, device="cuda"))
    ref = orc.create_rhs(np.full(orc.n_dofs, 0.5), T, T_old, q)
    assert np.linalg.norm(r.cpu().numpy() - ref) <= 1e-11 * np.linalg.norm(ref)
    # back to the constant vector: the tangent must be bound again first
    op.set_velocity_field(None)
    with pytest.raises(M.MpdgError):
        op.vmult(dst, torch.tensor(src, device="cuda"))
    op.bind_temperature(Td, Tod)
    op.vmult(dst, torch.tensor(src, device="cuda"))
    orc.set_tangent(DT, material=MUSHY, velocity=vel, do_solidification=solid, T_old=T_old)
    ref = orc.vmult(src, threads=1)
    assert np.linalg.norm(dst.cpu().numpy() - ref) <= 1e-12 * np.linalg.norm(ref)


# edges of the wavefronts' pencils (16 cells along x) and of the bricks (4 cells along z, Q1: 8)
@pytest.mark.parametrize("field", [False, True])
@pytest.mark.parametrize("degree,nc,solid", [(1, (17, 3, 9), True), (1, (16, 1, 8), False), (2, (33, 2, 5), True), (2, (1, 3, 4), False),
                                             (3, (18, 2, 5), True)])
def test_tangent_at_brick_edges(cuda, degree, nc, solid, field):
    torch = cuda
    import meltpooldg_amd as M
    L = tuple(0.1 * n for n in nc)
    orc, op, T, T_old, Td, Tod = pair(torch, M, degree, nc, L, 0b000001, solid, (0.2, -0.4, 0.1))
    if field:
        # the constant velocity as a field: the coefficients are then stored per direction
        v = torch.tensor([0.2, -0.4, 0.1], dtype=torch.float64, device="cuda").repeat_interleave(op.n_dofs)
        op.set_velocity_field(v)
        op.bind_temperature(Td, Tod)
    src = np.random.default_rng(6).uniform(-1, 1, orc.n_dofs)
    dst = torch.full((orc.n_dofs,), float("nan"), dtype=torch.float64, device="cuda")
    op.vmult(dst, torch.tensor(src, device="cuda"))
    ref = orc.vmult(src, threads=1)
    assert np.linalg.norm(dst.cpu().numpy() - ref) <= 1e-12 * np.linalg.norm(ref)
    d = torch.empty_like(dst)
    op.compute_diagonal(d)
    ref = orc.diagonal()
    assert np.linalg.norm(d.cpu().numpy() - ref) <= 1e-12 * np.linalg.norm(ref)


def test_velocity_field_needs_the_tangent(cuda):
    torch = cuda
    import meltpooldg_amd as M
    op = M.HeatDiffuseMultiPhaseOperator(2, (2, 2, 2))
    with pytest.raises(M.MpdgError):
        op.set_velocity_field(torch.zeros(3 * op.n_dofs, dtype=torch.float64, device="cuda"))
    op.reset_time_increment(DT)
    op.set_tangent(GPU_MUSHY)
    with pytest.raises(ValueError):
        op.set_velocity_field(torch.zeros(op.n_dofs, dtype=torch.float64, device="cuda"))


def test_tangent_is_bitwise_repeatable(cuda):
    """Tangent apply, diagonal and residual applied repeatedly give identical bits (the blocks add
    their shared rows in eight colour classes, one after the other, without atomics)."""
    torch = cuda
    import meltpooldg_amd as M
    orc, op, T, T_old, Td, Tod = pair(torch, M, 2, (40, 12, 10), (0.8, 0.24, 0.2), 0b000011, True,
                                      (0.2, -0.4, 0.1), seed=11)
    src = torch.tensor(np.random.default_rng(12).uniform(-1, 1, orc.n_dofs), device="cuda")
    q = torch.tensor(np.random.default_rng(13).uniform(0, 100, orc.n_dofs), device="cuda")
    outs = []
    for _ in range(3):
        dst = torch.empty(orc.n_dofs, dtype=torch.float64, device="cuda")
        op.vmult(dst, src)
        d = torch.empty_like(dst)
        op.compute_diagonal(d)
        r = torch.full_like(dst, 0.5)
        op.create_rhs(r, Td, Tod, q)
        torch.cuda.synchronize()
        outs.append([v.cpu().numpy().copy() for v in (dst, d, r)])
    for o in outs[1:]:
        for a, b in zip(outs[0], o):
            assert np.array_equal(a, b)
    ref = orc.vmult(src.cpu().numpy(), threads=1)
    assert np.linalg.norm(outs[0][0] - ref) <= 1e-12 * np.linalg.norm(ref)


@pytest.mark.parametrize("restart", [0, 5])
def test_gmres_matches_oracle(cuda, restart):
    """J x = b with the non-symmetric tangent: GMRES + inverse diagonal on the GPU and in the oracle reach
    the same solution; the iteration counts agree within 2 (same Krylov spaces, different rounding)."""
    torch = cuda
    import meltpooldg_amd as M
    orc, op, *_ = pair(torch, M, 2, (6, 5, 4), (0.6, 0.5, 0.4), 0, True, (-0.8, 0.3, 0.1), seed=5)
    b = np.random.default_rng(6).uniform(-1, 1, orc.n_dofs)
    xr, itr, _ = orc.gmres(b, rel_tol=1e-12, precond=1, restart=restart or 28, criterion=1, threads=1)
    pc = M.JacobiPreconditioner(op)
    pc.update()
    x = torch.zeros(orc.n_dofs, dtype=torch.float64, device="cuda")
    it = M.LinearSolver.solve(op, x, torch.tensor(b, device="cuda"),
                              M.LinearSolverData(solver_type=M.SOLVER_GMRES, rel_tolerance=1e-12,
                                                 criterion=M.CRIT_RHS, gmres_restart=restart), pc)
    assert itr > 0 and abs(it - itr) <= 2
    assert np.linalg.norm(x.cpu().numpy() - xr) <= 1e-9 * np.linalg.norm(xr)


@pytest.mark.parametrize("case", sorted(TANGENT_GOLDEN))
def test_tangent_golden_norm_sequences(cuda, case):
    """2D Q1 32x32 on [0,0.1]^2 as a one-cell-thick 3D mesh; Newton with GMRES + Jacobi."""
    torch = cuda
    import meltpooldg_amd as M
    nc, L = (32, 32, 1), (0.1, 0.1, 1.0)
    op = M.HeatDiffuseMultiPhaseOperator(1, nc, L)
    orc = O.Operator(1, nc, L)
    if case == "velocity":
        dt, tol = 1e-3, 1e-6
        op.set_tangent(dict(conductivity=55.563, specific_heat=460.0, density=7850.0), velocity=(-0.01, 0.0, 0.0))
        T0 = np.full(orc.n_dofs, 1000.0)
        placeholder = torch.tensor(T0, device="cuda")
        op.set_robin(2, alpha=25.0, T_inf_conv=300.0, emissivity=0.98, T_inf_rad=300.0, T=placeholder)
    else:
        dt, tol = 0.01, 1e-7
        op.set_tangent(GPU_MUSHY, velocity=(-0.005, 0.0, 0.0), do_solidification=True)
        T0 = 1960.0 + 20.0 * orc.node_coords()[0] / 0.1
    pc = M.JacobiPreconditioner(op)
    heat = M.HeatDiffuseOperation(op, pc, predictor=M.PREDICTOR_LINEAR,
                                  linear=M.LinearSolverData(solver_type=M.SOLVER_GMRES, rel_tolerance=1e-12),
                                  nlsolve=M.NonlinearSolverData(residual_tolerance=tol))
    heat.set_initial_condition(torch.tensor(T0, device="cuda"))
    norms = []
    for _ in range(5):
        heat.solve(dt)
        norms.append(op.l2_norm(heat.solution()))
    assert ["%.5e" % v for v in norms] == ["%.5e" % v for v in TANGENT_GOLDEN[case]]


# cells beyond a row's full pencils of 16 share blocks of the coefficients with the next rows'
@pytest.mark.parametrize("degree,nc", [(1, (5, 6, 7)), (2, (21, 2, 5)), (2, (47, 3, 3)), (3, (11, 5, 2))])
def test_tangent_at_row_remainders(cuda, degree, nc):
    torch = cuda
    import meltpooldg_amd as M
    orc, op, T, T_old, Td, Tod = pair(torch, M, degree, nc, tuple(0.1 * n for n in nc), 0b000010, True, (0.2, -0.4, 0.1))
    src = np.random.default_rng(7).uniform(-1, 1, orc.n_dofs)
    dst = torch.full((orc.n_dofs,), float("nan"), dtype=torch.float64, device="cuda")
    op.vmult(dst, torch.tensor(src, device="cuda"))
    ref = orc.vmult(src, threads=1)
    assert np.linalg.norm(dst.cpu().numpy() - ref) <= 1e-12 * np.linalg.norm(ref)
    d = torch.empty_like(dst)
    op.compute_diagonal(d)
    ref = orc.diagonal()
    assert np.linalg.norm(d.cpu().numpy() - ref) <= 1e-12 * np.linalg.norm(ref)


@pytest.mark.parametrize("field", [False, True])
@pytest.mark.parametrize("degree", [1, 2, 3])
def test_a_nan_stays_in_its_cells(cuda, degree, field):
    """Of the source: in the apply; of the bound temperature: in the apply and the diagonal."""
    torch = cuda
    import meltpooldg_amd as M
    from tests.test_gpu_operator import nan_reach
    nc = (18, 5, 9)
    want, at = nan_reach(degree, nc)
    orc, op, T, T_old, Td, Tod = pair(torch, M, degree, nc, tuple(0.1 * n for n in nc), 0, True, (0.2, -0.4, 0.1))
    if field:
        v = torch.tensor([0.2, -0.4, 0.1], dtype=torch.float64, device="cuda").repeat_interleave(op.n_dofs)
        op.set_velocity_field(v)
        op.bind_temperature(Td, Tod)
    x, y = torch.zeros(want.shape, dtype=torch.float64, device="cuda"), torch.empty(want.size, dtype=torch.float64, device="cuda")
    x[at] = float("nan")
    op.vmult(y, x.view(-1))
    assert np.array_equal(torch.isnan(y).view(want.shape).cpu().numpy(), want)
    x[at] = 0.0
    Tn = Td.clone()
    Tn.view(want.shape)[at] = float("nan")
    op.bind_temperature(Tn, Tod)
    op.vmult(y, x.view(-1))
    assert np.array_equal(torch.isnan(y).view(want.shape).cpu().numpy(), want)
    op.compute_diagonal(y)
    assert np.array_equal(torch.isnan(y).view(want.shape).cpu().numpy(), want)
