"""Performance cases: the work a program hands to this framework, through its public entry points.

Each case is a dict of plain values.  `prepare` builds what the program holds before the call (mesh,
operator, solver, vectors, network), `run` makes one pass, `work` states the bytes and operations
the pass cannot do without, and `exact` gives the outputs in 64 bits from plain torch, with its own
numbering, geometry, element matrices, solver and network.

Meshes are boxes of nx x ny x nz hexahedra (each cut into 6 tetrahedra for tet4), graded and sheared
by a smooth map unless `warp` is 0, so that every element has its own geometry.  Vectors are uniform
in [-1, 1]; coefficients, where an operator has one, are log-uniform in [0.1, 10] per element.
"""
import math

import numpy as np
import torch

import sfem_amd as S
from sfem_amd import gmg

DEV = "cuda"
MU, LAM = 1.0 / 2.6, 0.3 / (1.3 * 0.4)  # E = 1, nu = 0.3

# hex8 corner order as (x, y, z) bits, and the six tetrahedra of a cube
CORNERS = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]
TETS = [(0, 1, 3, 7), (0, 1, 7, 5), (0, 4, 5, 7), (1, 2, 3, 6), (1, 3, 7, 6), (1, 5, 6, 7)]


def listed():
    return [
        # The smallest call: the apply inside an unpreconditioned CG on a 32^3-cube tet4 Poisson problem.
        dict(name="tet4_laplacian_32", kind="tet4_laplacian", nx=32, ny=32, nz=32, warp=0, scatter=0),
        # A tet4 mesh as a mesh generator leaves it: elements and nodes in no useful order, ragged extents.
        dict(name="tet4_laplacian_scattered", kind="tet4_laplacian", nx=81, ny=67, nz=74, warp=1, scatter=1),
        # The hex8 diffusion operator with a coefficient, the matrix-free apply of a large plain hex mesh.
        dict(name="hex8_laplacian", kind="hex8_laplacian", nx=125, ny=118, nz=131, warp=1, coeff=1, scatter=0),
        # Elasticity on a plain 128^3 hex8 mesh: the fine-level apply of its multigrid solve.
        dict(name="hex8_elasticity_fp64_128", kind="hex8_elasticity", nx=128, ny=128, nz=128, warp=0, coeff=0,
             scatter=0, fp32=0),
        # The semi-structured Laplacian at its ordinary size, small enough to live in the caches.
        dict(name="sshex8_laplacian_fp64_L8_16", kind="sshex8_laplacian", level=8, nx=16, ny=16, nz=16, warp=0,
             coeff=0, fp32=0),
        # The FP32/bf16 Laplacian of a preconditioner with a coefficient per macro element, beyond the caches.
        dict(name="sshex8_laplacian_fp32_L8_32", kind="sshex8_laplacian", level=8, nx=31, ny=33, nz=32, warp=1,
             coeff=1, fp32=1),
        # The largest call: the FP64 elasticity operator on 171 million unknowns (an outer CG's product).
        dict(name="sshex8_elasticity_fp64_L16_24", kind="sshex8_elasticity", level=16, nx=24, ny=24, nz=24, warp=0,
             coeff=1, fp32=0),
        # The FP32/bf16 elasticity operator inside a multigrid preconditioner on about 50 million unknowns.
        dict(name="sshex8_elasticity_fp32_L8_32", kind="sshex8_elasticity", level=8, nx=33, ny=31, nz=32, warp=1,
             coeff=1, fp32=1),
        # A whole solve to 1e-10 in FP64: CG with a graph-replayed multigrid cycle on 2.1 million unknowns.
        dict(name="solve_laplacian_fp64_L8_16", kind="solve", problem="laplacian", level=8, n=16, coeff=0, mixed=0),
        # A whole mixed-precision solve: FP32 cycle in FP64 flexible CG, elasticity, 0.8 million unknowns.
        dict(name="solve_elasticity_mixed_L8_8", kind="solve", problem="elasticity", level=8, n=8, coeff=1, mixed=1),
        # Inference of the learned smoother: the scalar network over every macro element of a 32^3 mesh.
        dict(name="cnn_inference_bf16_L8", kind="cnn_forward", level=8, elements=32768, channels=1, bf16=1),
        # One training step's loss and gradients on a minibatch of macro elements.
        dict(name="cnn_training_L8_32", kind="cnn_train", level=8, elements=32, channels=1),
    ]


def draw(rng):
    """One more case of the ranges above."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def box(lo, hi):
        n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        return {k: max(1, min(int(hi * 1.1), int(round(n * rng.uniform(0.8, 1.25))))) for k in ("nx", "ny", "nz")}

    kind = rng.choice(["tet4_laplacian", "hex8_laplacian", "hex8_elasticity", "sshex8_laplacian", "sshex8_elasticity",
                       "solve", "cnn_forward", "cnn_train"])
    warp, coeff, fp32, scatter = rng.randint(0, 1), rng.randint(0, 1), rng.randint(0, 1), int(rng.random() < 0.3)
    if kind == "tet4_laplacian":
        return dict(kind=kind, **box(8, 90), warp=warp, scatter=scatter)
    if kind == "hex8_laplacian":
        return dict(kind=kind, **box(8, 128), warp=warp, coeff=coeff, scatter=scatter)
    if kind == "hex8_elasticity":
        return dict(kind=kind, **box(8, 128), warp=warp, coeff=coeff, scatter=scatter, fp32=fp32)
    if kind in ("sshex8_laplacian", "sshex8_elasticity"):
        level = rng.choice([2, 3, 4, 5, 6, 8, 8, 12, 16])
        return dict(kind=kind, level=level, **box(2, 192 // level), warp=warp, coeff=coeff, fp32=fp32)
    if kind == "solve":
        problem = rng.choice(["laplacian", "elasticity"])
        n = rng.choice([4, 6, 8, 12, 16] if problem == "laplacian" else [4, 6, 8])
        return dict(kind=kind, problem=problem, level=rng.choice([2, 4, 8]), n=n, coeff=coeff, mixed=rng.randint(0, 1))
    channels = rng.choice([1, 3])
    if kind == "cnn_forward":
        bf16 = int(channels == 1 and rng.random() < 0.7)
        return dict(kind=kind, level=rng.randint(2, 8), elements=log_int(32, 32768 if bf16 else 2048),
                    channels=channels, bf16=bf16)
    return dict(kind=kind, level=rng.randint(2, 8), elements=log_int(8, 256), channels=channels)


# ------------------------------------------------------------------ inputs
def _rng(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 1000003 + salt) & 0x7fffffffffff)
    return g


def _uniform(n, seed, salt, lo=-1.0, hi=1.0, dtype=torch.float64):
    t = torch.rand(n, generator=_rng(seed, salt), device=DEV, dtype=dtype)
    return t.mul_(hi - lo).add_(lo)


def _coefficients(case, n, seed):
    if not case.get("coeff"):
        return None
    return (10.0 ** _uniform(n, seed, 2)).float()


def _scatter(case, nodes, elements, seed):
    """A renumbering in no useful order: (new id of each node, old element of each new one)."""
    if not case.get("scatter"):
        return None, None
    p = torch.randperm(nodes, generator=_rng(seed, 3), device=DEV)
    q = torch.randperm(elements, generator=_rng(seed, 4), device=DEV)
    return p, q


def _warped(points, warp):
    """A smooth invertible map of the unit cube ([3][N], float64)."""
    if not warp:
        return points
    x, y, z = points
    s = torch.sin(math.pi * x) * torch.sin(math.pi * y) * torch.sin(math.pi * z)
    return torch.stack([x + 0.15 * y + 0.06 * s, y - 0.1 * z + 0.05 * x * x, 1.1 * z + 0.08 * torch.sin(2 * x + y)])


def _box(nx, ny, nz, tet=False):
    """Corners [8 or 4][E] and unit-cube points [3][N] (float32 words) in the framework's box numbering:
    node (x, y, z) is y (nx+1)(nz+1) + x (nz+1) + z, elements run x fastest, z slowest."""
    ld0, ld1 = nz + 1, (nz + 1) * (nx + 1)
    zi, yi, xi = torch.meshgrid(torch.arange(nz, device=DEV), torch.arange(ny, device=DEV),
                                torch.arange(nx, device=DEV), indexing="ij")
    base = (xi * ld0 + yi * ld1 + zi).reshape(-1)
    hexa = torch.stack([base + cx * ld0 + cy * ld1 + cz for cx, cy, cz in CORNERS])
    if tet:
        hexa = torch.stack([torch.stack([hexa[v] for v in t]) for t in TETS], 2).reshape(4, -1)
    ax = [torch.linspace(0, 1, n + 1, device=DEV, dtype=torch.float64).float() for n in (nx, ny, nz)]
    py, px, pz = torch.meshgrid(ax[1], ax[0], ax[2], indexing="ij")
    return hexa, torch.stack([px.reshape(-1), py.reshape(-1), pz.reshape(-1)])


def _jacobians(corners, points):
    """Centre Jacobians [E][3][3] (row: coordinate, column: reference direction) of the elements."""
    p = points.double()
    if corners.shape[0] == 4:
        return torch.stack([torch.stack([p[d][corners[k]] - p[d][corners[0]] for k in (1, 2, 3)], -1)
                            for d in range(3)], 1)
    J = torch.zeros(corners.shape[1], 3, 3, dtype=torch.float64, device=DEV)
    for v, bits in enumerate(CORNERS):
        for d in range(3):
            for a in range(3):
                J[:, d, a] += (0.25 if bits[a] else -0.25) * p[d][corners[v]]
    return J


def _adjugate(J):
    """adj(J) [E][3][3] and det(J) [E]."""
    c = [[None] * 3 for _ in range(3)]
    for i in range(3):
        for j in range(3):
            a, b = [k for k in range(3) if k != j], [k for k in range(3) if k != i]
            m = J[:, a[0], b[0]] * J[:, a[1], b[1]] - J[:, a[0], b[1]] * J[:, a[1], b[0]]
            c[i][j] = m if (i + j) % 2 == 0 else -m
    A = torch.stack([torch.stack(r, -1) for r in c], 1)
    return A, (J[:, 0, :] * A[:, :, 0]).sum(-1)


def _fff_words(corners, points):
    """J^-1 J^-T det as float32 words [E][6] (tet4: over the reference tet's volume)."""
    A, det = _adjugate(_jacobians(corners, points))
    scale = 1.0 / 6.0 if corners.shape[0] == 4 else 1.0
    rows = [(A[:, a] * A[:, b]).sum(-1) / det * scale for a in range(3) for b in range(a, 3)]
    return torch.stack(rows, -1).float()


def _adjugate_words(corners, points):
    A, det = _adjugate(_jacobians(corners, points))
    return A.reshape(-1, 9).float(), det.float()


def _host(t):
    return None if t is None else t.cpu().numpy()


def _geometry(case, tet=False):
    corners, points = _box(case["nx"], case["ny"], case["nz"], tet)
    return corners, _warped(points.double(), case["warp"]).float()


# ------------------------------------------------------------------ prepare
def prepare(case, seed):
    return {"tet4_laplacian": _prepare_unstructured, "hex8_laplacian": _prepare_unstructured,
            "hex8_elasticity": _prepare_unstructured, "sshex8_laplacian": _prepare_sshex8,
            "sshex8_elasticity": _prepare_sshex8, "solve": _prepare_solve, "cnn_forward": _prepare_cnn,
            "cnn_train": _prepare_cnn}[case["kind"]](case, seed)


def _apply_state(case, op, seed):
    dtype = torch.float32 if case.get("fp32") else torch.float64
    x = _uniform(op.cols, seed, 1, dtype=dtype)
    return dict(case=case, op=op, x=x, y=torch.empty_like(x))


def _unstructured_mesh(case, seed):
    corners, points = _geometry(case, case["kind"] == "tet4_laplacian")
    p, q = _scatter(case, points.shape[1], corners.shape[1], seed)
    if p is not None:
        corners = p[corners][:, q]
        moved = torch.empty_like(points)
        moved[:, p] = points
        points = moved
    return corners, points


def _prepare_unstructured(case, seed):
    corners, points = _unstructured_mesh(case, seed)
    mesh = S.Mesh(S.TET4 if case["kind"] == "tet4_laplacian" else S.HEX8, 1, _host(corners.int()), points.shape[1])
    coeff = _host(_coefficients(case, corners.shape[1], seed))
    if case["kind"] == "hex8_elasticity":
        adj, det = _adjugate_words(corners, points)
        op = S.linear_elasticity(mesh, _host(adj), _host(det), MU, LAM, coeff,
                                 real_type=S.FLOAT32 if case["fp32"] else S.FLOAT64)
    else:
        op = S.laplacian(mesh, _host(_fff_words(corners, points)), coeff)
    return _apply_state(case, op, seed)


def _prepare_sshex8(case, seed):
    corners, points = _geometry(case)
    mesh, _ = S.sshex8_refine_device(case["level"], _host(corners.int()), nnodes=points.shape[1])
    rt = S.FLOAT32 if case["fp32"] else S.FLOAT64
    coeff = _host(_coefficients(case, corners.shape[1], seed))
    if case["kind"] == "sshex8_elasticity":
        adj, det = _adjugate_words(corners, points)
        op = S.linear_elasticity(mesh, _host(adj), _host(det), MU, LAM, coeff, real_type=rt)
    else:
        op = S.laplacian(mesh, _host(_fff_words(corners, points)), coeff, real_type=rt)
    return _apply_state(case, op, seed)


def _solve_rhs(case, seed, nodes, bc):
    """Zero on the constrained nodes; else uniform in [0, 1] (Laplacian) or a body force (elasticity)."""
    if case["problem"] == "laplacian":
        b = _uniform(nodes, seed, 1, 0.0, 1.0)
        b[bc] = 0
        return b
    b = _uniform(3 * nodes, seed, 1, -0.1, 0.1).view(nodes, 3)
    b[:, 2] -= 1
    b[bc] = 0
    return b.reshape(-1)


def _prepare_solve(case, seed):
    n, level = case["n"], case["level"]
    elements, points = S.box_mesh(n + 1, n + 1, n + 1)
    mesh, fine = S.sshex8_refine_device(level, elements, points)
    p = fine.numpy().reshape(3, mesh.nnodes)
    coeff = _host(_coefficients(case, n ** 3, seed))
    config = dict(coeff=coeff, smoother="cheb3_jacobi" if case["coeff"] else "cheb3", coarse="dense",
                  macro_box=(n, 1.0), lanczos_steps=60)
    if case["problem"] == "laplacian":
        bc = np.where((p.min(0) < 1e-6) | (p.max(0) > 1 - 1e-6))[0].astype(np.int32)
        geometry = S.fff(S.HEX8, 1, elements, points)
    else:
        bc = np.where(p[2] < 1e-6)[0].astype(np.int32)
        geometry = S.adjugate_det(S.HEX8, 1, elements, points)
        config.update(mu=MU, lam=LAM)
    h64 = gmg.SSGMG(mesh, case["problem"], geometry, bc, **config) if not case["mixed"] else None
    if case["mixed"]:
        h32 = gmg.SSGMG(mesh, case["problem"], geometry, bc, real_type=S.FLOAT32, **config)
        if case["problem"] == "laplacian":
            op = S.laplacian(mesh, geometry, coeff)
        else:
            op = S.linear_elasticity(mesh, *geometry, MU, LAM, coeff)
        A = S.constrained(op, bc, 1 if case["problem"] == "laplacian" else 3)
        solver = S.cg(A, h32.preconditioner(graph=True), flexible=True, rtol=1e-10, max_it=500)
    else:
        solver = S.cg(h64.fine.A, h64.preconditioner(graph=True), rtol=1e-10, max_it=500, stop_on_residual=True)
    b = _solve_rhs(case, seed, mesh.nnodes, torch.from_numpy(bc).to(DEV).long())
    return dict(case=case, op=solver, x=b, y=torch.empty_like(b), keep=mesh)


def _weights(case, seed):
    """He-normal weights of the 4-layer network of 16 channels, [layer][out][in][27]."""
    c = case["channels"]
    out = [torch.randn(co * ci * 27, generator=_rng(seed, 10 + i), device=DEV, dtype=torch.float64)
           * math.sqrt(2.0 / (27 * ci)) for i, (ci, co) in enumerate([(c, 16), (16, 16), (16, 16), (16, c)])]
    return torch.cat(out).float()


def _cnn_arrays(case, seed):
    n = case["elements"] * case["channels"] * (case["level"] + 1) ** 3
    return (_uniform(n, seed, 20, dtype=torch.float32),
            _uniform(n, seed, 21, dtype=torch.float32) if case["kind"] == "cnn_train" else None)


def _prepare_cnn(case, seed):
    z, t = _cnn_arrays(case, seed)
    cnn = S.CNN(16, 4, weights=_host(_weights(case, seed)), channels=case["channels"])
    return dict(case=case, cnn=cnn, z=z, t=t, out=torch.empty_like(z))


# ------------------------------------------------------------------ run
def run(state):
    case = state["case"]
    if case["kind"] == "cnn_forward":
        return state["cnn"].forward(case["level"], state["z"], state["out"], mode=case["bf16"])
    if case["kind"] == "cnn_train":
        loss, grad = state["cnn"].loss_grad(case["level"], state["z"], state["t"])
        return [loss, grad]
    # y += A x into a zeroed y, or a solve from a zero initial guess
    return state["op"].apply(state["x"], state["y"].zero_())


# ------------------------------------------------------------------ work
def work(case):
    kind = case["kind"]
    if kind in ("cnn_forward", "cnn_train"):
        nodes = case["elements"] * (case["level"] + 1) ** 3
        c = case["channels"]
        macs = 27 * (2 * 16 * c + 2 * 2 * 16 * 16) * nodes  # the hidden layers for both signs of the odd network
        if kind == "cnn_forward":
            return {"bytes": 8 * c * nodes, "flops": 2 * macs}
        return {"bytes": 8 * c * nodes + 8 * 27 * (32 * c + 512), "flops": 6 * macs}
    if kind == "solve":
        L, E = case["level"], case["n"] ** 3
        N, bs = (case["n"] * L + 1) ** 3, 1 if case["problem"] == "laplacian" else 3
        # about 10 iterations, each an FP64 product and a cycle with 5 fine products and updates
        real = 4 if case["mixed"] else 8
        product = 4 * (L + 1) ** 3 * E
        per_it = 6 * product + bs * N * (2 * 8 + 6 * 8) + 5 * bs * N * 6 * real * 8 // 7
        return {"bytes": 10 * per_it, "flops": 10 * 6 * 2 * (27 if bs == 1 else 243) * N}
    E = case["nx"] * case["ny"] * case["nz"]
    if kind.startswith("sshex8"):
        L = case["level"]
        N = (case["nx"] * L + 1) * (case["ny"] * L + 1) * (case["nz"] * L + 1)
        ids, words, flops = (L + 1) ** 3, 6 if kind == "sshex8_laplacian" else 10, 0
        flops = 2 * (27 if kind == "sshex8_laplacian" else 243) * N
    else:
        N = (case["nx"] + 1) * (case["ny"] + 1) * (case["nz"] + 1)
        E = 6 * E if kind == "tet4_laplacian" else E
        ids = 4 if kind == "tet4_laplacian" else 8
        words = 10 if kind == "hex8_elasticity" else 6
        flops = E * {"tet4_laplacian": 30, "hex8_laplacian": 128, "hex8_elasticity": 1000}[kind]
    bs = 3 if kind.endswith("elasticity") else 1
    real, word = (4, 2) if case.get("fp32") else (8, 4)
    return {"bytes": 2 * real * bs * N + 4 * ids * E + word * words * E + (4 * E if case.get("coeff") else 0),
            "flops": flops}


# ------------------------------------------------------------------ exact
def _reference_integrals():
    """I[a][b][i][j] = integral over the unit cube of d_a phi_i d_b phi_j."""
    g = [0.5 - 0.5 / math.sqrt(3), 0.5 + 0.5 / math.sqrt(3)]
    out = torch.zeros(3, 3, 8, 8, dtype=torch.float64)
    for q in [(a, b, c) for a in g for b in g for c in g]:
        grad = torch.zeros(8, 3, dtype=torch.float64)
        for i, bits in enumerate(CORNERS):
            f = [q[d] if bits[d] else 1 - q[d] for d in range(3)]
            for d in range(3):
                w = 1.0 if bits[d] else -1.0
                for e in range(3):
                    w *= f[e] if e != d else 1.0
                grad[i, d] = w
        out += 0.125 * torch.einsum("ia,jb->abij", grad, grad)
    return out.to(DEV)


def _element_matrices(kind, words, coeff):
    """[E][k][k] element matrices in 64 bits from the float32 geometry words; vector dofs run corner
    by corner, component fastest."""
    scale = 1.0 if coeff is None else coeff.double()[:, None, None]
    if kind == "tet4_laplacian":
        f = words.double()
        G = f[:, [0, 1, 2, 1, 3, 4, 2, 4, 5]].reshape(-1, 3, 3)
        grad = torch.tensor([[-1, -1, -1], [1, 0, 0], [0, 1, 0], [0, 0, 1]], dtype=torch.float64, device=DEV)
        return torch.matmul(torch.matmul(grad, G), grad.t().contiguous()) * scale
    I = _reference_integrals()
    if kind.endswith("laplacian"):
        G = words.double()[:, [0, 1, 2, 1, 3, 4, 2, 4, 5]]
        return torch.matmul(G, I.reshape(9, 64)).reshape(-1, 8, 8) * scale
    adj, det = words[0].double().reshape(-1, 3, 3), words[1].double()
    P = adj / det[:, None, None]  # P[e][a][k] = d(reference a) / d(physical k)
    M = torch.zeros(adj.shape[0], 3, 3, 64, dtype=torch.float64, device=DEV)
    for k in range(3):
        for l in range(3):
            for a in range(3):
                for b in range(3):
                    M[:, k, l] += (P[:, a, k] * P[:, b, l])[:, None] * I[a, b].reshape(1, 64)
    M = M.reshape(-1, 3, 3, 8, 8)
    trace = MU * (M[:, 0, 0] + M[:, 1, 1] + M[:, 2, 2])
    K = torch.empty(adj.shape[0], 8, 3, 8, 3, dtype=torch.float64, device=DEV)
    for c in range(3):
        for d in range(3):
            K[:, :, c, :, d] = LAM * M[:, c, d] + MU * M[:, d, c] + (trace if c == d else 0)
    return K.reshape(-1, 24, 24) * det[:, None, None] * scale


def _sshex8_ids(nx, ny, nz, level):
    """Node ids [E][(L+1)^3] of the hierarchical numbering: macro corners keep their box ids, the other
    nodes are numbered at their first encounter over (level 1 < ... < L, element, z, y, x)."""
    L = level
    ar = lambda n: torch.arange(n, device=DEV)
    zi, yi, xi = (t.reshape(-1, 1) for t in torch.meshgrid(ar(nz), ar(ny), ar(nx), indexing="ij"))
    lz, ly, lx = (t.reshape(1, -1) for t in torch.meshgrid(ar(L + 1), ar(L + 1), ar(L + 1), indexing="ij"))
    mx, my = nx * L + 1, ny * L + 1
    grid = ((zi * L + lz) * my + (yi * L + ly)) * mx + (xi * L + lx)  # lattice point of each local node
    number = torch.full((mx * my * (nz * L + 1),), -1, dtype=torch.int64, device=DEV)
    ld0, ld1 = nz + 1, (nz + 1) * (nx + 1)
    for cx, cy, cz in CORNERS:
        number[grid[:, (cz * L * (L + 1) + cy * L) * (L + 1) + cx * L]] = \
            ((xi + cx) * ld0 + (yi + cy) * ld1 + (zi + cz)).reshape(-1)
    count = (nx + 1) * (ny + 1) * (nz + 1)
    chain = [L]
    while chain[-1] % 2 == 0 and (chain[-1] // 2) % 2 == 0:
        chain.append(chain[-1] // 2)
    for l in reversed([c for c in chain if c > 1]):
        s = L // l
        local = ((lx % s == 0) & (ly % s == 0) & (lz % s == 0)).reshape(-1).nonzero().reshape(-1)
        order = grid[:, local].reshape(-1)
        order = order[number[order] < 0]
        first = torch.full_like(number, order.numel())
        first.scatter_reduce_(0, order, torch.arange(order.numel(), device=DEV), "amin")
        at = (first < order.numel()).nonzero().reshape(-1)
        rank = torch.argsort(first[at])
        number[at[rank]] = count + torch.arange(at.numel(), device=DEV)
        count += at.numel()
    return number[grid], number.numel()


def _micro_corners(L):
    """Local node [L^3][8] of every micro element's corners."""
    ar = torch.arange(L, device=DEV)
    z, y, x = (t.reshape(-1) for t in torch.meshgrid(ar, ar, ar, indexing="ij"))
    return torch.stack([((z + cz) * (L + 1) + y + cy) * (L + 1) + x + cx for cx, cy, cz in CORNERS], -1)


def _product(K, groups, x, bs):
    """A x for element matrices K [E][k][k] and groups(e0, e1) -> node ids [e][m][corners]."""
    y = torch.zeros_like(x).view(-1, bs)
    E, k = K.shape[0], K.shape[1]
    m = groups(0, 1).shape[1]
    step = max(1, (1 << 26) // (m * k))
    Kt = K.transpose(1, 2)
    for e in range(0, E, step):
        ids = groups(e, min(E, e + step))
        u = x.view(-1, bs)[ids].reshape(ids.shape[0], m, k)
        v = torch.matmul(u, Kt[e:e + step].contiguous()) if m > 1 else \
            torch.matmul(K[e:e + step], u.transpose(1, 2).contiguous())
        y.index_add_(0, ids.reshape(-1), v.reshape(-1, bs))
    return y.reshape(-1)


def _exact_product(case, seed):
    kind = case["kind"]
    bs = 3 if kind.endswith("elasticity") else 1
    coeff = None
    if kind.startswith("sshex8"):
        corners, points = _geometry(case)
        ids, N = _sshex8_ids(case["nx"], case["ny"], case["nz"], case["level"])
        micro = _micro_corners(case["level"])
        groups = lambda a, b: ids[a:b][:, micro]
        # a micro element's share of the macro element's words: FFF and (adjugate, det) scale by 1/L
        scale = 1.0 / case["level"]
    else:
        corners, points = _unstructured_mesh(case, seed)
        N, scale = points.shape[1], 1.0
        groups = lambda a, b: corners[:, a:b].t().reshape(b - a, 1, -1)
    coeff = _coefficients(case, corners.shape[1], seed)
    dtype = torch.float32 if case.get("fp32") else torch.float64
    x = _uniform(bs * N, seed, 1, dtype=dtype).double()
    y = torch.zeros_like(x)
    step = 1 << 18
    for e in range(0, corners.shape[1], step):
        part = corners[:, e:e + step]
        words = _adjugate_words(part, points) if bs == 3 else _fff_words(part, points)
        K = _element_matrices(kind, words, None if coeff is None else coeff[e:e + step]) * scale
        y += _product(K, lambda a, b: groups(e + a, e + b), x, bs)
    return y


def _exact_solve(case, seed):
    n, L, bs = case["n"], case["level"], 1 if case["problem"] == "laplacian" else 3
    corners, points = _box(n, n, n)
    words = _adjugate_words(corners, points) if bs == 3 else _fff_words(corners, points)
    K = _element_matrices(case["problem"], words, _coefficients(case, n ** 3, seed)) / L
    ids, N = _sshex8_ids(n, n, n, L)
    lz, ly, lx = torch.meshgrid(*[torch.arange(L + 1, device=DEV)] * 3, indexing="ij")
    e = torch.arange(n ** 3, device=DEV)
    at = lambda i, l: (i[:, None] * L + l.reshape(1, -1))
    gx, gy, gz = at(e % n, lx), at(e // n % n, ly), at(e // (n * n), lz)
    fixed = gz == 0
    if bs == 1:
        for g in (gx, gy, gz):
            fixed = fixed | (g == 0) | (g == n * L)
    free = torch.ones(N, dtype=torch.float64, device=DEV)
    free[ids[fixed]] = 0
    bc = (free == 0).nonzero().reshape(-1)
    free = free.repeat_interleave(bs)
    b = _solve_rhs(case, seed, N, bc)
    micro = _micro_corners(L)
    A = lambda v: free * _product(K, lambda i, j: ids[i:j][:, micro], free * v, bs) + (1 - free) * v
    d = torch.zeros(N, bs, dtype=torch.float64, device=DEV)
    diag = torch.diagonal(K, dim1=1, dim2=2)[:, None, :].expand(-1, L ** 3, -1).reshape(-1, bs)
    d.index_add_(0, ids[:, micro].reshape(-1), diag)
    d = free * d.reshape(-1) + (1 - free)
    # Jacobi-preconditioned CG to a relative residual of 1e-13
    x, r = torch.zeros_like(b), b.clone()
    z = r / d
    p, rz, stop = z.clone(), torch.dot(r, z), 1e-13 * float(torch.linalg.norm(b))
    for it in range(4000):
        q = A(p)
        alpha = rz / torch.dot(p, q)
        x += alpha * p
        r -= alpha * q
        if it % 10 == 9 and float(torch.linalg.norm(r)) < stop:
            break
        z = r / d
        rz, old = torch.dot(r, z), rz
        p = z + (rz / old) * p
    return x


def _network(z, weights, c, L):
    """g(z) on [E][c][(L+1)^3] in 64 bits."""
    a = z.reshape(-1, c, L + 1, L + 1, L + 1)
    for i, (ci, co) in enumerate([(c, 16), (16, 16), (16, 16), (16, c)]):
        a = torch.nn.functional.pad(torch.relu(a) if i else a, (1,) * 6)
        n = L + 1
        cols = torch.stack([a[:, :, k // 9:k // 9 + n, k // 3 % 3:k // 3 % 3 + n, k % 3:k % 3 + n]
                            for k in range(27)], 2).reshape(a.shape[0], ci * 27, n ** 3)
        a = torch.matmul(weights[i].reshape(co, ci * 27), cols).reshape(-1, co, n, n, n)
    return a.reshape(z.shape)


def _exact_cnn(case, seed):
    c, L = case["channels"], case["level"]
    w = _weights(case, seed).double()
    sizes = [16 * c * 27, 16 * 16 * 27, 16 * 16 * 27, 16 * c * 27]
    z, t = _cnn_arrays(case, seed)
    shape = (case["elements"], c * (L + 1) ** 3)
    z = z.double().reshape(shape)
    step = max(1, (1 << 27) // (16 * 27 * (L + 1) ** 3))
    if case["kind"] == "cnn_forward":
        ws = torch.split(w, sizes)
        out = [_network(p, ws, c, L) - _network(-p, ws, c, L) for p in torch.split(z, step)]
        return torch.cat(out).reshape(-1)
    w.requires_grad_(True)
    t = t.double().reshape(shape)
    norm, total = float((t * t).sum()), 0.0
    for p, q in zip(torch.split(z, step), torch.split(t, step)):
        ws = torch.split(w, sizes)
        loss = ((_network(p, ws, c, L) - _network(-p, ws, c, L) - q) ** 2).sum() / norm
        loss.backward()
        total += float(loss.detach())
    return [total, w.grad.cpu().numpy()]


def exact(case, seed):
    if case["kind"].startswith("cnn"):
        return _exact_cnn(case, seed)
    if case["kind"] == "solve":
        return _exact_solve(case, seed)
    return _exact_product(case, seed)
