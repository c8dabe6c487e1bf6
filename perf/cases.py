"""The work that programs have this library do, as cases that can be timed.

A case is a dict of plain values; ``kind`` says which call it is:

* ``laplace``: assembly of the Laplace matrix and right-hand side;
* ``laplace_solve``: a static linear solve with Dirichlet values;
* ``assembly``: Mooney-Rivlin residual and Jacobian, one Newton iteration's assembly;
* ``solver_system``: the same, then the matrix and vector of the free DOFs that a host's own solver takes;
* ``batch``: residual and Jacobian of many meshes of uneven size as one set;
* ``load_step``: a whole load step by Newton's method, from the plain or the learned start;
* ``warm_start``: the learned start alone (the network's forward pass on every node);
* ``gradient``: loss and parameter gradient of the network on one minibatch (its backward pass).

Sizes come from the benchmark, the tests and the training set-up of this
repository, with odd and non-cubic ones beside them.  ``exact`` restates the
results in plain torch in 64 bits from the weak forms, without the library.
"""
import math

import numpy as np
import torch

import cm_amd as cm
from cm_amd import _lib
from cm_amd.train_warm_start import DEFAULT_WEIGHTS, PLAIN_KRYLOV_RTOL, solver_options
from cm_amd.warm_start import N_FEATURES, N_OUTPUTS, WarmStartMLP

JITTER = 0.1  # of the element size, interior nodes


def listed():
    return [
        # the smallest assembly call of the tests: launches and latency
        dict(name="laplace_8", kind="laplace", nx=8, ny=8, nz=8, numbering="grid"),
        # a mesh read from a file, nodes numbered in no order, ragged sizes
        dict(name="laplace_user", kind="laplace", nx=61, ny=47, nz=53, numbering="user"),
        # the benchmark's largest Laplace grid
        dict(name="laplace_128", kind="laplace", nx=128, ny=128, nz=128, numbering="grid"),
        # a linear solve of ordinary size (GMRES(30), point Jacobi: the defaults)
        dict(name="laplace_solve", kind="laplace_solve", nx=33, ny=27, nz=24),
        # a hand-sized elasticity model: what every small test or tutorial problem assembles
        dict(name="mr_4", kind="assembly", nx=4, ny=4, nz=4, precision="fp64"),
        # the benchmark's headline: 32^3, residual and FP64 Jacobian
        dict(name="mr_32", kind="assembly", nx=32, ny=32, nz=32, precision="fp64"),
        # a host with its own solver, FP32 Jacobian, non-cubic mesh
        dict(name="mr_solver_system", kind="solver_system", nx=23, ny=17, nz=11, precision="fp32"),
        # many small meshes at once (the training data's and the batch benchmark's shape)
        dict(name="mr_batch_24", kind="batch", meshes=24, n_min=4, n_max=12, precision="fp32"),
        # a load step by the plain method at the size of the benchmark's smaller solve
        dict(name="step_plain_16", kind="load_step", n=16, start="plain", precision="fp64", stretch=0.10, steps=10,
             c10=2.0, c01=6.0),
        # a load step with the learned start and FP32 Jacobians at the benchmark's size
        dict(name="step_learned_32", kind="load_step", n=32, start="learned", precision="fp32", stretch=0.20, steps=10,
             c10=2.0, c01=6.0),
        # the learned start of that size: 274,625 nodes through the network
        dict(name="warm_start_32", kind="warm_start", n=32, c10=2.0, c01=6.0, load=0.02),
        # one minibatch of the training's default size
        dict(name="gradient_4096", kind="gradient", samples=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["laplace", "laplace", "laplace_solve", "assembly", "assembly", "solver_system", "batch",
                       "load_step", "load_step", "warm_start", "gradient"])
    if kind == "laplace":
        user = rng.random() < 0.5
        hi = 56 if user else 110
        return dict(kind=kind, nx=_log_int(rng, 2, hi), ny=_log_int(rng, 2, hi), nz=_log_int(rng, 2, hi),
                    numbering="user" if user else "grid")
    if kind == "laplace_solve":
        return dict(kind=kind, nx=rng.randint(3, 32), ny=rng.randint(3, 32), nz=rng.randint(3, 24))
    if kind in ("assembly", "solver_system"):
        hi = 28 if kind == "assembly" else 18
        return dict(kind=kind, nx=_log_int(rng, 2, hi), ny=_log_int(rng, 2, hi), nz=_log_int(rng, 2, hi),
                    precision=rng.choice(["fp64", "fp32"]))
    if kind == "batch":
        return dict(kind=kind, meshes=_log_int(rng, 2, 30), n_min=rng.randint(2, 5), n_max=rng.randint(6, 12),
                    precision=rng.choice(["fp64", "fp32"]))
    if kind == "load_step":
        start = rng.choice(["plain", "learned"])
        return dict(kind=kind, n=rng.randint(4, 16), start=start, precision="fp32" if start == "learned" else "fp64",
                    stretch=round(rng.uniform(0.05, 0.15), 3), steps=5, c10=round(rng.uniform(1, 5), 2),
                    c01=round(rng.uniform(0, 10), 2))
    if kind == "warm_start":
        return dict(kind=kind, n=rng.randint(4, 30), c10=round(rng.uniform(1, 5), 2), c01=round(rng.uniform(0, 10), 2),
                    load=round(rng.uniform(0.01, 0.04), 3))
    return dict(kind=kind, samples=_log_int(rng, 64, 8192))


# ---- inputs ------------------------------------------------------------------


def _grid(case, order, seed):
    return cm.RegularMesh.generate(order, (case["nx"], case["ny"], case["nz"]), jitter=JITTER, seed=seed)


def _laplace_mesh(case, seed):
    mesh = _grid(case, 1, seed)
    if case["numbering"] == "user":
        mesh = cm.as_user_mesh(mesh, region_order=np.random.default_rng(seed).permutation(mesh.n_nodes))
    return mesh


def _batch_meshes(case, seed):
    """The meshes of a batch (their sizes are the case's, not the seed's) and their materials."""
    sizes = np.random.default_rng(case["meshes"]).integers(case["n_min"], case["n_max"] + 1, case["meshes"])
    rng = np.random.default_rng(seed)
    meshes = [cm.RegularMesh.generate(2, int(n), jitter=JITTER, seed=seed + 1000 * m) for m, n in enumerate(sizes)]
    return meshes, rng.uniform(1, 5, len(meshes)), rng.uniform(0, 10, len(meshes))


def _deformed(mesh, rng, stretch=1.1):
    """z (3, nodes) and p of a 10% uniaxial stretch with a small perturbation on it."""
    lam = np.array([stretch, stretch ** -0.5, stretch ** -0.5])
    z = mesh.coords * lam[:, None] + 0.002 * rng.uniform(-1, 1, mesh.coords.shape)
    return z, 0.5 * rng.standard_normal(mesh.n_nodes_l)


def _uniaxial_fixed(mesh):
    nq = mesh.n_nodes
    return np.concatenate([mesh.face_nodes(0, 0), nq + mesh.face_nodes(1, 0), 2 * nq + mesh.face_nodes(2, 0),
                           mesh.face_nodes(0, 1)])


def _linear_field(mesh, seed):
    """Every node's value of a seeded linear function, and the boundary nodes."""
    c = np.random.default_rng(seed).uniform(-1, 1, 4)
    u = c[0] + c[1:] @ mesh.coords
    boundary = np.unique(np.concatenate([mesh.face_nodes(a, side) for a in range(3) for side in (0, 1)]))
    return u, boundary


def _minibatch(case, seed):
    """Node features in their units, targets of the training's size and the network's seed."""
    rng = np.random.default_rng(seed)
    n = case["samples"]
    x = np.empty((n, N_FEATURES), np.float32)
    x[:, 0:3] = rng.uniform(0, 1, (n, 3))
    x[:, 3:6] = 0.1 * rng.standard_normal((n, 3))
    x[:, 6] = rng.uniform(0.01, 0.04, n)
    x[:, 7] = rng.uniform(1, 5, n)
    x[:, 8] = rng.uniform(0, 10, n)
    return x, rng.standard_normal((n, N_OUTPUTS)).astype(np.float32), seed


def _precision(case):
    return cm.OC_FP32 if case["precision"] == "fp32" else cm.OC_FP64


class _Borrowed:
    """A device buffer of an equations set as torch sees it (no copy); keeps the set."""

    def __init__(self, eq, buffer, n, typestr):
        self.eq = eq
        self.__cuda_array_interface__ = dict(data=(eq.device_pointer(buffer), False), shape=(int(n),), typestr=typestr,
                                             strides=None, version=2)


def _borrow(eq, buffer, n, typestr="<f8"):
    return torch.as_tensor(_Borrowed(eq, buffer, n, typestr), device="cuda")


def prepare(case, seed):
    cm.initialise(0)
    kind = case["kind"]
    s = dict(kind=kind, out=None)
    if kind == "laplace":
        s["eq"] = cm.LaplaceEquationsSet(_laplace_mesh(case, seed))
    elif kind == "laplace_solve":
        mesh = _grid(case, 1, seed)
        u, boundary = _linear_field(mesh, seed)
        s["eq"] = cm.LaplaceEquationsSet(mesh)
        s["eq"].set_boundary_conditions(boundary, u[boundary])
        s["options"] = cm.newton_options(krylov_relative_tolerance=1e-12, absolute_tolerance=0.0)
    elif kind in ("assembly", "solver_system"):
        mesh = _grid(case, 2, seed)
        z, p = _deformed(mesh, np.random.default_rng(seed))
        s["eq"] = cm.MooneyRivlinEquationsSet(mesh, 2.0, 6.0)
        s["eq"].set_dofs(np.concatenate([z.ravel(), p]))
        if kind == "solver_system":
            s["eq"].uniaxial_boundary_conditions(1.1)
        s["precision"] = _precision(case)
    elif kind == "batch":
        meshes, c10, c01 = _batch_meshes(case, seed)
        s["eq"] = cm.MooneyRivlinBatch(meshes, c10, c01)
        s["eq"].set_dofs(_batch_dofs(meshes, seed))
        s["precision"] = _precision(case)
    elif kind in ("load_step", "warm_start"):
        mesh = cm.RegularMesh.generate(2, case["n"], jitter=JITTER, seed=seed)
        eq = cm.MooneyRivlinEquationsSet(mesh, case["c10"], case["c01"])
        s["eq"] = eq
        s["d0"] = torch.from_numpy(eq.undeformed_dofs()).cuda()
        s["nu"] = 3 * mesh.n_nodes
        if kind == "load_step":
            eq.uniaxial_boundary_conditions(1.0 + case["stretch"])
            eq.set_multigrid()
            s["steps"], s["load"], s["precision"] = case["steps"], case["stretch"] / case["steps"], _precision(case)
            s["net"] = WarmStartMLP.load(DEFAULT_WEIGHTS) if case["start"] == "learned" else None
        else:
            eq.uniaxial_boundary_conditions(1.0 + case["load"])
            s["load"], s["net"] = case["load"], WarmStartMLP.load(DEFAULT_WEIGHTS)
    else:
        s["x"], s["t"], net_seed = _minibatch(case, seed)
        s["net"] = WarmStartMLP(hidden=128, layers=4, seed=net_seed)
    torch.cuda.synchronize()
    return s


def _batch_dofs(meshes, seed):
    """Component-major over the union: z1 of every mesh's nodes, z2, z3, then p."""
    rng = np.random.default_rng(seed)
    parts = [_deformed(m, rng) for m in meshes]
    return np.concatenate([z[c] for c in range(3) for z, _ in parts] + [p for _, p in parts])


# ---- one pass ------------------------------------------------------------------


def _matrix(eq, precision):
    if precision == cm.OC_FP32:
        return _borrow(eq, cm.OC_BUFFER_MATRIX_VALUES_SP, eq.nnz, "<f4")
    return _borrow(eq, cm.OC_BUFFER_MATRIX_VALUES, eq.nnz)


def run(s):
    kind = s["kind"]
    if kind == "gradient":
        loss, g = s["net"].gradient(s["x"], s["t"])
        return dict(loss=np.float32(loss), gradient=g)
    eq = s["eq"]
    if kind == "laplace":
        eq.assemble()
        if s["out"] is None:
            s["out"] = dict(values=_matrix(eq, cm.OC_FP64), rhs=_borrow(eq, cm.OC_BUFFER_RHS, eq.n_rows))
    elif kind == "laplace_solve":
        eq.solve(s["options"])
        if s["out"] is None:
            s["out"] = _borrow(eq, cm.OC_BUFFER_DOFS, eq.n_rows)
    elif kind in ("assembly", "batch", "solver_system"):
        eq.residual_evaluate()
        eq.jacobian_evaluate(s["precision"])
        if kind == "solver_system":
            eq.solver_matrices_assemble(s["precision"])
        if s["out"] is None:
            out = dict(residual=_borrow(eq, cm.OC_BUFFER_RESIDUAL, eq.n_rows), values=_matrix(eq, s["precision"]))
            if kind == "solver_system":
                n, nnz = eq.solver_matrix_info()
                fp32 = s["precision"] == cm.OC_FP32
                out["solver_values"] = _borrow(eq, cm.OC_BUFFER_SOLVER_VALUES_SP if fp32 else cm.OC_BUFFER_SOLVER_VALUES,
                                               nnz, "<f4" if fp32 else "<f8")
                out["solver_vector"] = _borrow(eq, cm.OC_BUFFER_SOLVER_VECTOR, n)
            s["out"] = out
    elif kind == "warm_start":
        _lib.call("oc_dofs_set_device", eq.handle, s["d0"].data_ptr())
        s["net"].warm_start(eq, s["load"])
        cm.synchronise()
        # the increment that the network predicts, per unit load: FP32 as its outputs are
        return ((_borrow(eq, cm.OC_BUFFER_DOFS, eq.n_rows) - s["d0"]) / s["load"]).float()
    else:
        _load_step(s)
        d = _borrow(eq, cm.OC_BUFFER_DOFS, eq.n_rows)
        # the residual tolerance of 1e-10 settles the deformed coordinates to
        # about 5e-11 and the pressure to a few 1e-6
        return dict(z=d[:s["nu"]], p=d[s["nu"]:].float())
    return s["out"]


def _load_step(s):
    """Load step 1 from the undeformed state, as cm_amd.train_warm_start.solve_steps takes it."""
    eq, ref = s["eq"], 0.0
    _lib.call("oc_dofs_set_device", eq.handle, s["d0"].data_ptr())
    if s["net"] is not None:
        eq.load_increment_apply(1, s["steps"])
        ref = eq.residual_norm()  # the plain start's residual: what the tolerance refers to
        _lib.call("oc_dofs_set_device", eq.handle, s["d0"].data_ptr())
        s["net"].warm_start(eq, s["load"])
    eq.load_increment_apply(1, s["steps"])
    eq.newton_solve(solver_options(s["precision"], reference_norm=ref, krylov_rtol=PLAIN_KRYLOV_RTOL))


# ---- what one pass cannot do without ---------------------------------------------


def _mr_sizes(*n):
    """(elements, DOFs, nonzeros) of a triquadratic/trilinear grid."""
    e = math.prod(n)
    q, lin = math.prod(2 * k + 1 for k in n), math.prod(k + 1 for k in n)
    nnz = 9 * math.prod(8 * k + 1 for k in n) + 6 * math.prod(5 * k + 1 for k in n) + math.prod(3 * k + 1 for k in n)
    return e, 3 * q + lin, nnz


MR_RESIDUAL_FLOP, MR_JACOBIAN_FLOP = 86400, 667251  # per element
LAPLACE_FLOP = 4224


def _mr_work(sizes, value_bytes):
    e, n, nnz = sizes
    # connectivity (27 + 8 int32), materials, coordinates and DOFs read; residual and values written
    return dict(bytes=156 * e + 24 * n + value_bytes * nnz, flops=(MR_RESIDUAL_FLOP + MR_JACOBIAN_FLOP) * e)


def work(case):
    kind = case["kind"]
    vb = 4 if case.get("precision") == "fp32" else 8
    if kind in ("laplace", "laplace_solve"):
        n = (case["nx"], case["ny"], case["nz"])
        e, nodes, nnz = math.prod(n), math.prod(k + 1 for k in n), math.prod(3 * k + 1 for k in n)
        return dict(bytes=32 * e + 24 * nodes + 8 * nnz + 8 * nodes, flops=LAPLACE_FLOP * e)
    if kind in ("assembly", "solver_system"):
        sizes = _mr_sizes(case["nx"], case["ny"], case["nz"])
        w = _mr_work(sizes, vb)
        if kind == "solver_system":  # the solver values and vector written too
            w["bytes"] += vb * sizes[2] + 8 * sizes[1]
        return w
    if kind == "batch":
        sizes = np.random.default_rng(case["meshes"]).integers(case["n_min"], case["n_max"] + 1, case["meshes"])
        return _mr_work(tuple(np.sum([_mr_sizes(*[int(n)] * 3) for n in sizes], axis=0).tolist()), vb)
    if kind == "load_step":  # one Jacobian and residual at the least, whatever the iterations
        return _mr_work(_mr_sizes(*[case["n"]] * 3), vb)
    per_sample = 2 * (N_FEATURES * 128 + 3 * 128 * 128 + 128 * N_OUTPUTS)
    if kind == "warm_start":
        e, n, _ = _mr_sizes(*[case["n"]] * 3)
        return dict(bytes=24 * n, flops=per_sample * (2 * case["n"] + 1) ** 3)
    params = N_FEATURES * 128 + 3 * 128 * 128 + 128 * N_OUTPUTS + 4 * 128 + N_OUTPUTS
    return dict(bytes=4 * (case["samples"] * (N_FEATURES + N_OUTPUTS) + 2 * params), flops=3 * per_sample * case["samples"])


# ---- the results in plain torch, 64 bits -------------------------------------------


def _dev(a, dtype=None):
    t = torch.from_numpy(np.ascontiguousarray(a)).cuda()
    return t if dtype is None else t.to(dtype)


def _gauss(points):
    x, w = np.polynomial.legendre.leggauss(points)
    return (x + 1) / 2, w / 2


def _tensor_basis(order, points):
    """Weights (G,), values (G, S) and derivatives (G, S, 3) on the unit cube, first direction fastest."""
    gx, gw = _gauss(points)
    if order == 1:
        val = np.stack([1 - gx, gx])
        der = np.stack([-np.ones_like(gx), np.ones_like(gx)])
    else:
        val = np.stack([(1 - gx) * (1 - 2 * gx), 4 * gx * (1 - gx), gx * (2 * gx - 1)])
        der = np.stack([4 * gx - 3, 4 - 8 * gx, 4 * gx - 1])

    def tensor(a, b, c):  # (nodes, points) of directions 1, 2, 3
        s, g = val.shape[0] ** 3, points ** 3
        return np.einsum("ai,bj,ck->kjicba", a, b, c).reshape(g, s)

    w = np.einsum("i,j,k->kji", gw, gw, gw).ravel()
    d = np.stack([tensor(der, val, val), tensor(val, der, val), tensor(val, val, der)], axis=-1)
    return _dev(w), _dev(tensor(val, val, val)), _dev(d)


def _sum_csr(rows, cols, values, n):
    """(keys row * n + column ascending, sums) of element entries, zeros kept."""
    keys, order = torch.sort((rows.long() * n + cols.long()).reshape(-1))
    new = torch.ones_like(keys, dtype=torch.bool)
    new[1:] = keys[1:] != keys[:-1]
    seg = torch.cumsum(new, 0) - 1
    out = torch.zeros(int(seg[-1]) + 1, dtype=torch.float64, device=keys.device)
    out.index_add_(0, seg, values.reshape(-1)[order])
    return keys[new], out


def _exact_laplace(mesh):
    w, _, d = _tensor_basis(1, 2)
    conn, X = _dev(mesh.elem_nodes).long(), _dev(mesh.coords)
    K = torch.zeros(conn.shape[0], 8, 8, dtype=torch.float64, device="cuda")
    xe = X[:, conn]  # (3, E, 8)
    for g in range(8):
        J = torch.einsum("ces,sk->eck", xe, d[g])
        G = torch.einsum("sk,ekc->esc", d[g], torch.linalg.inv(J))
        K += torch.einsum("esc,etc,e->est", G, G, w[g] * torch.linalg.det(J).abs())
    n = mesh.n_nodes
    _, values = _sum_csr(conn[:, :, None].expand(-1, -1, 8), conn[:, None, :].expand(-1, 8, -1), K, n)
    return dict(values=values, rhs=torch.zeros(n, dtype=torch.float64))


class _Elastic:
    """Mooney-Rivlin residual and Jacobian of a union of meshes, from the energy
    c10 (I1 J^(-2/3) - 3) + c01 (I2 J^(-4/3) - 3) + p (J - 1)."""

    def __init__(self, meshes, c10, c01):
        self.nq, self.nl = sum(m.n_nodes for m in meshes), sum(m.n_nodes_l for m in meshes)
        self.n = 3 * self.nq + self.nl
        q0 = np.cumsum([0] + [m.n_nodes for m in meshes])
        l0 = np.cumsum([0] + [m.n_nodes_l for m in meshes])
        cq = _dev(np.concatenate([m.elem_nodes + q for m, q in zip(meshes, q0)])).long()
        cl = _dev(np.concatenate([m.elem_nodes_l + k for m, k in zip(meshes, l0)])).long()
        self.dof = torch.cat([cq, self.nq + cq, 2 * self.nq + cq, 3 * self.nq + cl], 1)  # (E, 89)
        ne = [m.n_elements for m in meshes]
        self.c10, self.c01 = (_dev(np.repeat(np.asarray(c, np.float64), ne)) for c in (c10, c01))
        X = _dev(np.concatenate([m.coords for m in meshes], axis=1))
        self.w, _, self.d = _tensor_basis(2, 3)
        _, self.psi, _ = _tensor_basis(1, 3)
        self.xe = X[:, cq]  # (3, E, 27)

    def _gradients(self, z, g):
        """F, dN/dX and the weight of Gauss point g in every element."""
        JX = torch.einsum("ces,sk->eck", self.xe, self.d[g])
        dN = torch.einsum("sk,ekc->esc", self.d[g], torch.linalg.inv(JX))
        return torch.einsum("ecs,esj->ecj", z, dN), dN, self.w[g] * torch.linalg.det(JX).abs()

    @staticmethod
    def _energy(F, c10, c01):
        C = F.T @ F
        J = torch.linalg.det(F).abs()
        I1 = torch.trace(C)
        I2 = 0.5 * (I1 * I1 - torch.trace(C @ C))
        return c10 * I1 * J ** (-2 / 3) + c01 * I2 * J ** (-4 / 3)

    def evaluate(self, dofs, jacobian=True):
        ze = dofs[self.dof[:, :81]].reshape(-1, 3, 27)
        pe = dofs[self.dof[:, 81:]]
        E = ze.shape[0]
        R = torch.zeros(E, 89, dtype=torch.float64, device="cuda")
        K = torch.zeros(E, 89, 89, dtype=torch.float64, device="cuda") if jacobian else None
        grad = torch.func.vmap(torch.func.grad(self._energy))
        hess = torch.func.vmap(torch.func.jacfwd(torch.func.grad(self._energy)), chunk_size=65536)
        for g in range(27):
            F, dN, w = self._gradients(ze, g)
            J, Fi = torch.linalg.det(F), torch.linalg.inv(F)
            cof = J[:, None, None] * Fi.transpose(1, 2)  # dJ/dF
            p = pe @ self.psi[g]
            P = grad(F, self.c10, self.c01) + p[:, None, None] * cof
            R[:, :81] += torch.einsum("ecj,esj,e->ecs", P, dN, w).reshape(E, 81)
            R[:, 81:] += (w * (J - 1))[:, None] * self.psi[g]
            if not jacobian:
                continue
            A = hess(F, self.c10, self.c01)
            FiT = Fi.transpose(1, 2)
            A = A + (p * J)[:, None, None, None, None] * (torch.einsum("eij,ekl->eijkl", FiT, FiT)
                                                          - torch.einsum("eil,ekj->eijkl", FiT, FiT))
            A = A * w[:, None, None, None, None]
            T = torch.einsum("eijkl,etl->eijkt", A, dN)
            K[:, :81, :81] += torch.einsum("esj,eijkt->eiskt", dN, T).reshape(E, 81, 81)
            B = torch.einsum("ecj,esj,e->ecs", cof, dN, w).reshape(E, 81)
            K[:, 81:, :81] += self.psi[g][:, None] * B[:, None, :]
        r = torch.zeros(self.n, dtype=torch.float64, device="cuda").index_add_(0, self.dof.reshape(-1), R.reshape(-1))
        if not jacobian:
            return r, None, None
        K[:, :81, 81:] = K[:, 81:, :81].transpose(1, 2)
        keys, values = _sum_csr(self.dof[:, :, None].expand(-1, -1, 89), self.dof[:, None, :].expand(-1, 89, -1), K, self.n)
        return r, keys, values


def _exact_step(case, seed):
    """Load step 1 solved by Newton's method with dense linear solves: small meshes only."""
    mesh = cm.RegularMesh.generate(2, case["n"], jitter=JITTER, seed=seed)
    el = _Elastic([mesh], [case["c10"]], [case["c01"]])
    d = torch.zeros(el.n, dtype=torch.float64, device="cuda")
    d[:3 * mesh.n_nodes] = _dev(mesh.coords.ravel())
    d[_dev(mesh.face_nodes(0, 1)).long()] += case["stretch"] / case["steps"]
    free = torch.ones(el.n, dtype=torch.bool, device="cuda")
    free[_dev(_uniaxial_fixed(mesh)).long()] = False
    for _ in range(12):
        r, keys, values = el.evaluate(d)
        A = torch.zeros(el.n * el.n, dtype=torch.float64, device="cuda")
        A[keys] = values
        A = A.reshape(el.n, el.n)[free][:, free]
        step = torch.linalg.solve(A, -r[free])
        d[free] += step
        if float(step.norm()) < 1e-14 * float(d.norm()):
            break
    # the pressure is settled by the solver's tolerance, not by its precision
    return dict(z=d[:3 * mesh.n_nodes], p=None)


def _exact_network(net, x):
    """The network's outputs in 64 bits, and its parameters as leaves."""
    from cm_amd.warm_start import FEATURE_SCALE, FEATURE_SHIFT
    flat = _dev(net.parameters()).double().requires_grad_()
    h = (x - _dev(FEATURE_SHIFT).double()) * _dev(FEATURE_SCALE).double()
    dims, at = [N_FEATURES] + [net.hidden] * net.layers + [net.outputs], 0
    for k, (a, b) in enumerate(zip(dims[:-1], dims[1:])):
        W, c = flat[at:at + a * b].reshape(b, a), flat[at + a * b:at + a * b + b]
        at += a * b + b
        h = h @ W.T + c
        if k + 2 < len(dims):
            h = torch.nn.functional.gelu(h)
    return h, flat


def _exact_warm_start(case, seed):
    mesh = cm.RegularMesh.generate(2, case["n"], jitter=JITTER, seed=seed)
    cm.initialise(0)
    X = _dev(mesh.coords.T)
    x = torch.zeros(mesh.n_nodes, N_FEATURES, dtype=torch.float64, device="cuda")
    x[:, :3] = X.float().double()
    for k, v in ((6, case["load"]), (7, case["c10"]), (8, case["c01"])):
        x[:, k] = float(np.float32(v))
    with torch.no_grad():
        y, _ = _exact_network(WarmStartMLP.load(DEFAULT_WEIGHTS), x)
    n1 = case["n"] + 1
    i = torch.arange(n1 ** 3, device="cuda")
    T = 2 * case["n"] + 1
    corner = 2 * (i % n1) + 2 * T * ((i // n1) % n1) + 2 * T * T * (i // (n1 * n1))
    out = torch.cat([y[:, 0], y[:, 1], y[:, 2], (case["c10"] + case["c01"]) * y[corner, 3]])
    out[_dev(_uniaxial_fixed(mesh)).long()] = 0.0
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "laplace":
        return _exact_laplace(_laplace_mesh(case, seed))
    if kind == "laplace_solve":  # linear functions are solutions, and in the trilinear space
        return _dev(_linear_field(_grid(case, 1, seed), seed)[0])
    if kind in ("assembly", "solver_system"):
        mesh = _grid(case, 2, seed)
        z, p = _deformed(mesh, np.random.default_rng(seed))
        el = _Elastic([mesh], [2.0], [6.0])
        r, keys, values = el.evaluate(_dev(np.concatenate([z.ravel(), p])))
        out = dict(residual=r, values=values)
        if kind == "solver_system":
            free = torch.ones(el.n, dtype=torch.bool, device="cuda")
            free[_dev(_uniaxial_fixed(mesh)).long()] = False
            out["solver_values"] = values[free[keys // el.n] & free[keys % el.n]]
            out["solver_vector"] = r[free]
        return out
    if kind == "batch":
        meshes, c10, c01 = _batch_meshes(case, seed)
        r, _, values = _Elastic(meshes, c10, c01).evaluate(_dev(_batch_dofs(meshes, seed)))
        return dict(residual=r, values=values)
    if kind == "load_step":
        return _exact_step(case, seed) if case["n"] <= 6 else None
    if kind == "warm_start":
        return _exact_warm_start(case, seed)
    cm.initialise(0)
    x, t, net_seed = _minibatch(case, seed)
    y, flat = _exact_network(WarmStartMLP(hidden=128, layers=4, seed=net_seed), _dev(x).double())
    loss = ((y - _dev(t).double()) ** 2).mean()
    loss.backward()
    return dict(loss=loss.detach(), gradient=flat.grad)
