"""The work that a user of this package has it do, as measurable cases.

A case is one call (or the few calls) that a time loop repeats: the operator apply in its
discretisations, conductivities, geometries and precisions; the right-hand side; the Newton
tangent; a linear solve with multigrid; implicit time steps; the training direction of the
learned guess. ``listed`` has one case for each, from the smallest mesh (launch latency) to the
benchmark's 57 M unknowns; ``draw`` takes others from the same ranges, odd sizes among them.

``exact`` restates what the calls compute with plain torch in float64 (cell-wise tensor
contractions on gathered DoFs, Jacobi CG for the solves, shifted matrix products for the
network), without this package's kernels.
"""
import math

import numpy as np
import torch

import meltpooldg_amd as M

TANH_LAW = (1.0, 0.5, 1.0, 0.1)  # k0 (1 + a tanh((T - T0) / w))
MUSHY = dict(conductivity=(55.563, 17.0), specific_heat=(460.0, 700.0), density=(7850.0, 7850.0),
             solidus=1966.0, liquidus=1974.0)
VELOCITY = (-0.3, 0.1, 0.05)
FLUX = dict(peak=1e3, sigma=0.05, x0=0.3, y0=0.5, vx=1.0)  # the laser scan's surface flux
DT = 1e-3
DT_TANGENT = 0.01
CONVECTION = 50.0
N_STEPS = 3


def listed():
    return [
        # an apply on a small mesh, as on a multigrid's lower levels and in quick studies: latency
        _case("vmult_q2_16", kind="vmult", degree=2, nc=(16, 16, 16), k="const"),
        # linear elements with convection on the top and side faces, ragged box
        _case("vmult_q1_robin", kind="vmult", degree=1, nc=(101, 60, 37), k="const", robin=0b100011),
        # the headline apply: 57 M unknowns, conductivity per quadrature point
        _case("vmult_q3_128", kind="vmult", degree=3, nc=(128, 128, 128), k="qp"),
        # fourth order with the conductivity law evaluated inside the apply
        _case("vmult_q4_96_law", kind="vmult", degree=4, nc=(96, 96, 96), k="law"),
        # curved cells: metric per quadrature point
        _case("vmult_q3_96_mapped", kind="vmult", degree=3, nc=(96, 96, 96), k="const", mapped=0.05),
        # the single precision applies that multigrid smoothing is made of
        _case("vmult_f32_q2_64", kind="vmult", degree=2, nc=(64, 64, 64), k="const", f32=True),
        _case("vmult_f32_q3_ragged", kind="vmult", degree=3, nc=(75, 62, 49), k="cell", f32=True, dirichlet=0b010000),
        # the residual of a step with a moving laser and k(T)
        _case("rhs_q2_64_law", kind="rhs", degree=2, nc=(64, 64, 64), k="law"),
        # Newton iteration of the melting problem: coefficients at T, one tangent apply
        _case("tangent_q2_solid", kind="tangent", degree=2, nc=(70, 50, 33), k="const"),
        # one linear system with the mixed precision multigrid
        _case("solve_q3_64", kind="solve", degree=3, nc=(64, 64, 64), k="qp", levels="f32"),
        # implicit steps of the laser scan, conductivity and multigrid following T
        _case("steps_q2_64", kind="steps", degree=2, nc=(64, 64, 64), k="law", levels="f32"),
        # one training sample of the learned guess, forward and backward
        _case("train_q2_32", kind="train", degree=2, nc=(32, 32, 32), k="const"),
    ]


def _case(name, kind, degree, nc, k, f32=False, mapped=0.0, dirichlet=0, robin=0, levels=""):
    c = dict(kind=kind, degree=degree, nx=nc[0], ny=nc[1], nz=nc[2], k=k, f32=f32, mapped=mapped,
             dirichlet=dirichlet, robin=robin, levels=levels)
    if name:
        c["name"] = name
    return c


def draw(rng):
    kind = rng.choice(["vmult"] * 6 + ["rhs", "tangent", "solve", "steps", "train"])
    degree = rng.choice([1, 2, 2, 3, 3, 4])
    if kind in ("solve", "steps"):
        # boxes that coarsen by two down to at most four cells per direction
        halvings = rng.randint(2, 4)
        most = 3 if degree == 4 and halvings == 4 else 4
        nc = [rng.randint(low, most) * 2 ** halvings for low in (3, 2, 2)]
        return _case(None, kind, degree, nc, "law" if kind == "steps" else rng.choice(["const", "qp", "cell"]),
                     levels=rng.choice(["f32", "f32", "f64"]))
    if kind == "train":
        n = rng.choice([12, 16, 20, 24, 32])
        return _case(None, kind, rng.choice([1, 2]), (n, n, n), "const")
    most = {"vmult": 57e6, "rhs": 6e6, "tangent": 4e6}[kind]
    dofs = math.exp(rng.uniform(math.log(3e4), math.log(most)))
    side = dofs ** (1.0 / 3.0) / degree
    nc = [max(2, int(round(side * math.exp(rng.uniform(-0.4, 0.4))))) for _ in range(3)]
    while (nc[0] * degree + 1) * (nc[1] * degree + 1) * (nc[2] * degree + 1) > most:
        nc = [max(2, n - 1) for n in nc]
    if kind == "rhs":
        return _case(None, kind, degree, nc, rng.choice(["const", "qp", "law"]))
    if kind == "tangent":
        return _case(None, kind, degree, nc, "const")
    mapped = rng.random() < 0.2
    f32 = rng.random() < 0.4
    robin = 0b100000 if rng.random() < 0.15 and not f32 and not mapped else 0
    return _case(None, kind, degree, nc, "const" if mapped else rng.choice(["const", "qp", "qp", "cell", "law"]), f32=f32,
                 mapped=0.05 if mapped else 0.0, dirichlet=rng.choice([0, 0, 0b010000, 0b000011]) if not robin else 0,
                 robin=robin)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _cells(c):
    return c["nx"], c["ny"], c["nz"]


def _n_dofs(c):
    k = c["degree"]
    return (k * c["nx"] + 1) * (k * c["ny"] + 1) * (k * c["nz"] + 1)


def _n_qp(c):
    return c["nx"] * c["ny"] * c["nz"] * (c["degree"] + 1) ** 3


def _dtype(c):
    return torch.float32 if c["f32"] else torch.float64


def _uniform(gen, n, lo, hi, dtype=torch.float64):
    return torch.empty(n, dtype=torch.float64, device="cuda").uniform_(lo, hi, generator=gen).to(dtype)


def _temperature(gen, c, mean, wave, noise):
    """A smooth field on the DoF grid with a little noise, as a scan in progress has it."""
    k = c["degree"]
    x, y, z = (torch.linspace(0.0, 1.0, k * n + 1, dtype=torch.float64, device="cuda") for n in _cells(c))
    a = torch.empty(3, dtype=torch.float64, device="cuda").uniform_(0.5, 1.5, generator=gen)
    f = mean + wave * torch.sin(7.0 * a[0] * x)[None, None, :] * torch.cos(5.0 * a[1] * y)[None, :, None] \
        + 0.3 * wave * a[2] * z[:, None, None]
    f = f.reshape(-1)
    return f + noise * torch.randn(f.numel(), dtype=torch.float64, device="cuda", generator=gen)


def _inputs(c, seed):
    """The tensors of a case, made from the seed alone."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    n, d = _n_dofs(c), {}
    if c["k"] == "qp":
        d["k"] = (1.0 + 0.5 * torch.tanh((_uniform(gen, _n_qp(c), 0.0, 2.0) - 1.0) / 0.1)).to(_dtype(c))
    elif c["k"] == "cell":
        d["k"] = _uniform(gen, c["nx"] * c["ny"] * c["nz"], 0.5, 1.5, _dtype(c))
    elif c["k"] == "law":
        d["T"] = _temperature(gen, c, 0.95, 0.15, 0.002 if c["kind"] != "steps" else 0.0).to(_dtype(c))
    if c["kind"] == "vmult":
        d["src"] = _uniform(gen, n, -1.0, 1.0, _dtype(c))
    elif c["kind"] == "rhs":
        if "T" not in d:
            d["T"] = _temperature(gen, c, 0.95, 0.15, 0.002)
        d["T_old"] = d["T"] - 0.01 * _uniform(gen, n, 0.0, 1.0)
        d["q"] = _uniform(gen, n, 0.0, 100.0)
    elif c["kind"] == "tangent":
        d["T"] = _temperature(gen, c, 1970.0, 6.0, 0.1)
        d["T_old"] = d["T"] - 0.4 * _uniform(gen, n, 0.0, 1.0)
        d["src"] = _uniform(gen, n, -1.0, 1.0)
    elif c["kind"] == "solve":
        d["b"] = _uniform(gen, n, -1.0, 1.0)
    elif c["kind"] == "train":
        d["T1"] = _temperature(gen, c, 0.95, 0.15, 0.0)
        rate = _temperature(gen, c, 0.02, 0.02, 0.0)
        d["T0"] = d["T1"] - rate
        d["T2"] = d["T1"] + rate + 0.001 * _temperature(gen, c, 0.0, 1.0, 0.0)
        d["q"] = _uniform(gen, n, 0.0, 100.0)
        d["z"] = 0.01 * _temperature(gen, c, 0.0, 1.0, 0.1)
        w = []
        for ci, co in zip((4, 16, 16, 16), (16, 16, 16, 1)):
            w.append(torch.randn(co * ci * 27, dtype=torch.float64, device="cuda", generator=gen)
                     * math.sqrt(2.0 / (27 * ci)))
            w.append(0.05 * torch.randn(co, dtype=torch.float64, device="cuda", generator=gen))
        d["weights"] = torch.cat(w).float().cpu().numpy()
    return d


def prepare(case, seed):
    c, d = case, _inputs(case, seed)
    s = dict(case=c, d=d)
    if c["kind"] == "train":
        net = M.LearnedPredictor(_cells(c), degree=c["degree"], coarsening=1, qscale=1e-3, seed=1)
        net.set_weights(d["weights"])
        net.output_scale = 0.5
        s["net"] = net
        return s
    op = M.HeatDiffuseMultiPhaseOperator(c["degree"], _cells(c), rho_cp=1.0, precision=M.FP32 if c["f32"] else M.FP64,
                                         dirichlet_faces=c["dirichlet"])
    op.reset_time_increment(DT_TANGENT if c["kind"] == "tangent" else DT)
    if c["k"] == "const":
        op.set_conductivity_constant(1.0)
    elif c["k"] == "qp":
        op.set_conductivity_qp(d["k"])
    elif c["k"] == "cell":
        op.set_conductivity_cell(d["k"])
    else:
        op.set_conductivity_law(M.LAW_TANH, TANH_LAW, d["T"])
    if c["mapped"]:
        op.set_mapping(M.node_coordinates(c["degree"], _cells(c), mapping_amplitude=c["mapped"]))
    if c["robin"]:
        op.set_robin(c["robin"], alpha=CONVECTION)
    if c["kind"] == "rhs":
        op.set_surface_flux(t=DT, **FLUX)
    if c["kind"] == "tangent":
        op.set_tangent(MUSHY, velocity=VELOCITY, do_solidification=True)
    s["op"] = op
    if c["kind"] != "steps":
        s["dst"] = op.new_vector()
    if c["kind"] in ("solve", "steps"):
        f32 = c["levels"] == "f32"
        s["pc"] = M.GMGPreconditioner(op, precision=M.FP32 if f32 else M.FP64, n_cells_coarse=4, coarse_degree=2,
                                      pre_smoother_degree=1 if f32 else 0)
        s["solver"] = M.LinearSolverData(solver_type=M.SOLVER_FCG if f32 else M.SOLVER_CG, rel_tolerance=1e-10,
                                         criterion=M.CRIT_RHS, max_iterations=2000)
        if c["kind"] == "solve":
            s["pc"].update()
        else:
            s["heat"] = M.HeatDiffuseOperation(op, s["pc"], predictor=M.PREDICTOR_EXTRAPOLATION, linear=s["solver"],
                                               step_mode=M.STEP_LINEAR, extrapolation_order=6)
    return s


def run(state):
    c, d = state["case"], state["d"]
    if c["kind"] == "train":
        loss, gradients = state["net"].gradients(d["T0"], d["T1"], d["q"], d["z"], d["T2"])
        return {"loss": loss, "gradients": gradients}
    op = state["op"]
    if c["kind"] == "vmult":
        op.vmult(state["dst"], d["src"])
        return state["dst"]
    if c["kind"] == "rhs":
        state["dst"].zero_()
        op.create_rhs(state["dst"], d["T"], d["T_old"], d["q"])
        return state["dst"]
    if c["kind"] == "tangent":
        op.bind_temperature(d["T"], d["T_old"])
        op.vmult(state["dst"], d["src"])
        return state["dst"]
    if c["kind"] == "solve":
        state["dst"].zero_()
        M.LinearSolver.solve(op, state["dst"], d["b"], state["solver"], state["pc"])
        return state["dst"]
    heat = state["heat"]
    heat.set_initial_condition(d["T"])
    for i in range(N_STEPS):
        op.set_surface_flux(t=(i + 1) * DT, **FLUX)
        heat.solve(DT)
    return heat.solution(), heat.old_solution()


def work(case):
    """Bytes of the inputs and outputs, operations of the cell-wise contractions (twelve
    one-dimensional sweeps of n1^4 multiply-adds per cell and apply, and the point work)."""
    c = case
    n, nq, n1 = _n_dofs(c), _n_qp(c), c["degree"] + 1
    item = 4 if c["f32"] else 8
    apply_flops = 2.0 * 12 * n1 * nq + 12.0 * nq
    k_bytes = {"const": 0, "qp": item * nq, "cell": item * c["nx"] * c["ny"] * c["nz"], "law": item * n}[c["k"]]
    if c["mapped"]:
        k_bytes += 3 * 8 * n
    if c["kind"] == "vmult":
        law = 2.0 * 3 * n1 * nq if c["k"] == "law" else 0.0
        return {"bytes": 2 * item * n + k_bytes, "flops": apply_flops + law}
    if c["kind"] == "rhs":
        return {"bytes": 8 * 5 * n + (k_bytes if c["k"] == "qp" else 0), "flops": apply_flops}
    if c["kind"] == "tangent":
        return {"bytes": 8 * 4 * n, "flops": 2.0 * apply_flops}
    if c["kind"] == "solve":
        # at the least one outer apply and one fine-level smoothing step
        return {"bytes": 2 * 8 * n + k_bytes, "flops": 2 * apply_flops}
    if c["kind"] == "steps":
        return {"bytes": N_STEPS * (2 * 8 * n + k_bytes), "flops": N_STEPS * 2 * apply_flops}
    taps = 27 * (4 * 16 + 16 * 16 + 16 * 16 + 16)
    return {"bytes": 5 * 8 * n + 8 * taps, "flops": 3 * 2.0 * taps * n}


# ---------------------------------------------------------------------------
# the same in float64 with plain torch
# ---------------------------------------------------------------------------
def _tables(k):
    """Gauss-Lobatto nodes, Gauss points and weights on [0, 1]; S[q][i] basis values, G[q][i]
    basis derivatives at the Gauss points."""
    inner = np.sort(np.polynomial.legendre.Legendre.basis(k).deriv().roots().real) if k > 1 else np.zeros(0)
    nodes = np.concatenate([[0.0], 0.5 * (1.0 + inner), [1.0]])
    p, w = np.polynomial.legendre.leggauss(k + 1)
    pts, w = 0.5 * (1.0 + p), 0.5 * w
    n1 = k + 1
    S, G = np.ones((n1, n1)), np.zeros((n1, n1))
    for i in range(n1):
        for q in range(n1):
            for j in range(n1):
                if j != i:
                    S[q, i] *= (pts[q] - nodes[j]) / (nodes[i] - nodes[j])
            for m in range(n1):
                if m != i:
                    t = 1.0 / (nodes[i] - nodes[m])
                    for j in range(n1):
                        if j != i and j != m:
                            t *= (pts[q] - nodes[j]) / (nodes[i] - nodes[j])
                    G[q, i] += t
    return nodes, pts, w, S, G


class _Exact:
    """The operator on arrays of cells (cz, cy, cx, z, y, x)."""

    def __init__(self, c, d, device="cuda"):
        self.c, self.d, self.dev = c, d, device
        k = self.k = c["degree"]
        self.n1 = k + 1
        self.nodes, self.pts, w, S, G = _tables(k)
        t = lambda a: torch.tensor(a, dtype=torch.float64, device=device)  # noqa: E731
        self.w, self.S, self.G = t(w), t(S), t(G)
        self.nc = _cells(c)
        self.nd = [k * n + 1 for n in self.nc]
        self.W = self.w[:, None, None] * self.w[:, None] * self.w
        self.h = [1.0 / n for n in self.nc]
        self.vol = self.h[0] * self.h[1] * self.h[2]
        self.cm = 1.0 / (DT_TANGENT if c["kind"] == "tangent" else DT)
        self.kappa = None
        if c["k"] in ("qp", "cell"):
            self.kappa = d["k"].double()
            self.kappa = self.kappa.reshape(self.nc[2], self.nc[1], self.nc[0], self.n1, self.n1, self.n1) \
                if c["k"] == "qp" else self.kappa.reshape(self.nc[2], self.nc[1], self.nc[0], 1, 1, 1)
        self.free = self._free()
        self.metric = self._mapped() if c["mapped"] else None

    def _free(self):
        m = self.c["dirichlet"]
        if not m:
            return None
        f = torch.ones(self.nd[2], self.nd[1], self.nd[0], dtype=torch.float64, device=self.dev)
        for bit, (dim, at) in enumerate(((2, 0), (2, -1), (1, 0), (1, -1), (0, 0), (0, -1))):
            if m >> bit & 1:
                f.select(dim, at).zero_()
        return f

    def grid(self, v):
        return v.double().reshape(self.nd[2], self.nd[1], self.nd[0])

    def gather(self, v):
        n1, k = self.n1, self.k
        return v.unfold(0, n1, k).unfold(1, n1, k).unfold(2, n1, k)

    def along(self, u, A, axis):
        """A applied to the cell index `axis` (0: x, 1: y, 2: z)."""
        dim = 5 - axis
        return torch.movedim(torch.matmul(torch.movedim(u, dim, -1).contiguous(), A.t().contiguous()), -1, dim)

    def values(self, u, x=None, y=None, z=None):
        S = self.S
        u = self.along(u, S if x is None else x, 0)
        u = self.along(u, S if y is None else y, 1)
        return self.along(u, S if z is None else z, 2)

    def gradient(self, u):
        return [self.values(u, x=self.G), self.values(u, y=self.G), self.values(u, z=self.G)]

    def integrate(self, val, flux):
        """sum_q val N + flux . grad_xi N, as cell DoFs."""
        St, Gt = self.S.t(), self.G.t()
        e = self.values(val, St, St, St) if val is not None else 0.0
        if flux is not None:
            e = e + self.values(flux[0], Gt, St, St)
            e = e + self.values(flux[1], St, Gt, St)
            e = e + self.values(flux[2], St, St, Gt)
        return e

    def scatter(self, e):
        k, (cz, cy, cx) = self.k, e.shape[:3]
        out = torch.zeros(self.nd[2], self.nd[1], self.nd[0], dtype=torch.float64, device=self.dev)
        for a in range(self.n1):
            for b in range(self.n1):
                for i in range(self.n1):
                    out[a:a + k * (cz - 1) + 1:k, b:b + k * (cy - 1) + 1:k, i:i + k * (cx - 1) + 1:k] += e[..., a, b, i]
        return out

    def _mapped(self):
        axes = []
        for n in self.nc:
            h = 1.0 / n
            axes.append(np.concatenate([i * h + self.nodes[:-1] * h for i in range(n)] + [np.array([1.0])]))
        x, y, z = (torch.tensor(a, dtype=torch.float64, device=self.dev) for a in axes)
        zero = torch.zeros(self.nd[2], self.nd[1], self.nd[0], dtype=torch.float64, device=self.dev)
        X = zero + x + self.c["mapped"] * torch.sin(2 * np.pi * y)[:, None] * torch.sin(2 * np.pi * z)[:, None, None]
        J = [self.gradient(self.gather(f)) for f in (X, zero + y[:, None], zero + z[:, None, None])]
        # the adjugate's rows: det * d xi_a / d x
        C = [[J[(b + 1) % 3][(a + 1) % 3] * J[(b + 2) % 3][(a + 2) % 3] - J[(b + 1) % 3][(a + 2) % 3] * J[(b + 2) % 3][(a + 1) % 3]
              for b in range(3)] for a in range(3)]
        det = J[0][0] * C[0][0] + J[0][1] * C[1][0] + J[0][2] * C[2][0]
        G = [[sum(C[a][i] * C[b][i] for i in range(3)) / det * self.W for b in range(3)] for a in range(3)]
        return det * self.W, G

    def law(self, T):
        k0, a, T0, w = TANH_LAW
        return k0 * (1.0 + a * torch.tanh((self.values(self.gather(self.grid(T))) - T0) / w))

    def apply(self, v, mass=None, kappa=None):
        """J v on the DoF grid (constrained rows and columns zero)."""
        kappa = self.kappa if kappa is None else kappa
        mass = self.cm if mass is None else mass
        v = self.grid(v)
        if self.free is not None:
            v = v * self.free
        u = self.gather(v)
        val, g = self.values(u), self.gradient(u)
        if self.metric is None:
            s = self.W * self.vol * (1.0 if kappa is None else kappa)
            e = self.integrate(mass * self.vol * self.W * val, [s / self.h[a] ** 2 * g[a] for a in range(3)])
        else:
            jxw, G = self.metric
            e = self.integrate(mass * jxw * val, [sum(G[a][b] * g[b] for b in range(3)) for a in range(3)])
        out = self.scatter(e)
        if self.c["robin"]:
            out = out + self.robin(v)
        return out if self.free is None else out * self.free

    def mass_1d(self, axis):
        n, k = self.nc[axis], self.k
        m = torch.zeros(k * n + 1, k * n + 1, dtype=torch.float64, device=self.dev)
        loc = self.S.t() @ (self.w[:, None] * self.S) * self.h[axis]
        for i in range(n):
            m[k * i:k * i + k + 1, k * i:k * i + k + 1] += loc
        return m

    def robin(self, v):
        out = torch.zeros_like(v)
        for face in range(6):
            if not self.c["robin"] >> face & 1:
                continue
            d, at = face // 2, 0 if face % 2 == 0 else -1
            other = [a for a in range(3) if a != d]
            f = v.select(2 - d, at)  # the higher of the other axes first
            out.select(2 - d, at).add_(CONVECTION * (self.mass_1d(other[1]) @ f @ self.mass_1d(other[0])))
        return out

    def flux_rhs(self, t):
        """The surface flux on z+ against the face's basis functions."""
        k, one = self.k, []
        for axis, centre in ((0, FLUX["x0"] + FLUX["vx"] * t), (1, FLUX["y0"])):
            n, h = self.nc[axis], self.h[axis]
            x = (torch.arange(n, dtype=torch.float64, device=self.dev)[:, None]
                 + torch.tensor(self.pts, dtype=torch.float64, device=self.dev)) * h
            loc = (torch.exp(-(x - centre) ** 2 / (2 * FLUX["sigma"] ** 2)) * self.w * h) @ self.S
            f = torch.zeros(k * n + 1, dtype=torch.float64, device=self.dev)
            for i in range(self.n1):
                f[i:i + k * (n - 1) + 1:k] += loc[:, i]
            one.append(f)
        return FLUX["peak"] * one[1][:, None] * one[0]

    def rhs(self):
        d = self.d
        mass = self.grid(d["T"].double() - d["T_old"].double() - d["q"].double() / self.cm)
        kappa = self.law(d["T"]) if self.c["k"] == "law" else self.kappa
        zero = torch.zeros((), dtype=torch.float64, device=self.dev)
        out = -self.apply(mass, kappa=zero) - self.apply(d["T"], mass=0.0, kappa=kappa)
        out[-1] += self.flux_rhs(DT)
        return out

    def diagonal(self, kappa=None):
        kappa = self.kappa if kappa is None else kappa
        ones = torch.ones(self.nc[2], self.nc[1], self.nc[0], self.n1, self.n1, self.n1, dtype=torch.float64,
                          device=self.dev)
        s = self.W * self.vol * (ones if kappa is None else kappa)
        S2, G2 = (self.S ** 2).t(), (self.G ** 2).t()
        e = self.values(self.cm * self.vol * self.W * ones, S2, S2, S2)
        for a in range(3):
            t = [S2, S2, S2]
            t[a] = G2
            e = e + self.values(s / self.h[a] ** 2 * ones, *t)
        d = self.scatter(e)
        return d if self.free is None else torch.where(self.free > 0, d, torch.ones_like(d))

    def tangent(self):
        d, m = self.d, MUSHY
        cell = lambda v: self.gather(self.grid(v))  # noqa: E731
        phys = lambda u: [g / h for g, h in zip(self.gradient(u), self.h)]  # noqa: E731
        T, gT, T_old = self.values(cell(d["T"])), phys(cell(d["T"])), self.values(cell(d["T_old"]))
        width = m["liquidus"] - m["solidus"]
        fs = ((m["liquidus"] - T) / width).clamp(0.0, 1.0)
        inside = ((fs > 0) & (fs < 1)).double()
        blend = lambda p: p[0] + (p[1] - p[0]) * (3 * fs ** 2 - 2 * fs ** 3)  # noqa: E731
        slope = lambda p: -inside / width * (p[1] - p[0]) * (6 * fs - 6 * fs ** 2)  # noqa: E731
        k, dk = blend(m["conductivity"]), slope(m["conductivity"])
        rho, cp = blend(m["density"]), blend(m["specific_heat"])
        rc, drc = rho * cp, slope(m["specific_heat"]) * rho + slope(m["density"]) * cp
        u = cell(d["src"])
        val, g = self.values(u), phys(u)
        conv = lambda f: sum(v * f[a] for a, v in enumerate(VELOCITY))  # noqa: E731
        v = rc / DT_TANGENT * val + rc * conv(g) + drc * ((T - T_old) / DT_TANGENT + conv(gT)) * val
        jxw = self.W * self.vol
        flux = [jxw / self.h[a] * (k * g[a] + dk * gT[a] * val) for a in range(3)]
        return self.scatter(self.integrate(jxw * v, flux))

    def solve(self, b, x, kappa=None, tol=1e-13):
        """Jacobi CG to ||b - J x|| <= tol ||b||."""
        inv = 1.0 / self.diagonal(kappa)
        r = b - self.apply(x, kappa=kappa)
        stop = tol * float(b.norm())
        z = inv * r
        p, rz = z.clone(), float((r * z).sum())
        for _ in range(3000):
            q = self.apply(p, kappa=kappa)
            alpha = rz / float((p * q).sum())
            x, r = x + alpha * p, r - alpha * q
            if float(r.norm()) <= stop:
                break
            z = inv * r
            new = float((r * z).sum())
            p, rz = z + (new / rz) * p, new
        return x

    def steps(self):
        T = self.grid(self.d["T"])
        old = T
        zero = torch.zeros((), dtype=torch.float64, device=self.dev)
        for i in range(N_STEPS):
            b = self.apply(T, kappa=zero)
            b[-1] += self.flux_rhs((i + 1) * DT)
            old, T = T, self.solve(b, T.clone(), kappa=self.law(T))
        return T, old


def _train_exact(c, d):
    k = c["degree"]
    nx, ny, nz = (k * n + 1 for n in _cells(c))
    T0, T1, T2, q, z = (d[n].double() for n in ("T0", "T1", "T2", "q", "z"))
    n = T1.numel()
    inc = T1 - T0
    s = inc.square().mean().sqrt() + 1e-30
    mean = T1.mean()
    spread = (T1.square().mean() - mean ** 2).clamp(min=0.0).sqrt() + 1e-12 + 1e-6 * mean.abs()
    sz = z.square().mean().sqrt() + 1e-30
    a = torch.stack([inc / s, q * 1e-3 / s, (T1 - mean) / spread, z / sz], dim=1)
    target = (T2 - (2.0 * T1 - T0)) / (0.5 * sz)

    def shifted(f, dx, dy, dz):
        p = torch.nn.functional.pad(f.reshape(nz, ny, nx, -1), (0, 0, 1, 1, 1, 1, 1, 1))
        return p[1 + dz:1 + dz + nz, 1 + dy:1 + dy + ny, 1 + dx:1 + dx + nx].reshape(n, -1)

    taps = [(t % 3 - 1, (t // 3) % 3 - 1, t // 9 - 1) for t in range(27)]
    flat = torch.tensor(d["weights"], dtype=torch.float64, device=a.device)
    layers, o = [], 0
    for ci, co in zip((4, 16, 16, 16), (16, 16, 16, 1)):
        layers.append((flat[o:o + co * ci * 27].reshape(co, ci, 27), flat[o + co * ci * 27:o + co * ci * 27 + co]))
        o += co * ci * 27 + co
    acts = [a]
    for i, (w, b) in enumerate(layers):
        y = b + sum(shifted(acts[-1], *t) @ w[:, :, j].t() for j, t in enumerate(taps))
        acts.append(y.clamp(min=0.0) if i < 3 else y)
    e = acts[-1][:, 0] - target
    g, grads = (2.0 / n * e)[:, None], []
    for i in range(3, -1, -1):
        w = layers[i][0]
        gw = torch.stack([g.t() @ shifted(acts[i], *t) for t in taps], dim=2)
        grads = [gw.reshape(-1), g.sum(0)] + grads
        if i:
            back = sum(shifted(g, -t[0], -t[1], -t[2]) @ w[:, :, j] for j, t in enumerate(taps))
            g = back * (acts[i] > 0)
    return {"loss": float(e.square().mean()), "gradients": torch.cat(grads)}


def exact(case, seed):
    c = case
    if c["kind"] in ("solve", "steps") and _n_dofs(c) > 9e6:
        return None
    d = _inputs(c, seed)
    if c["kind"] == "train":
        return _train_exact(c, d)
    x = _Exact(c, d)
    if c["kind"] == "vmult":
        if c["k"] == "law":
            x.kappa = x.law(d["T"])
        return x.apply(d["src"]).reshape(-1)
    if c["kind"] == "rhs":
        return x.rhs().reshape(-1)
    if c["kind"] == "tangent":
        return x.tangent().reshape(-1)
    if c["kind"] == "solve":
        b = x.grid(d["b"])
        return x.solve(b, torch.zeros_like(b)).reshape(-1)
    T, old = x.steps()
    return T.reshape(-1), old.reshape(-1)
