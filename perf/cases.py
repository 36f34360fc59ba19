"""Performance cases of the operator library: what a user's program has it do, through the public entry points.

The paths are those of a finite-element solve with this library and of a program that uses its element routines alone:
operator applications inside a Krylov loop (jv, linear), nonlinear residuals (residual), the set-up and first
Krylov vector of a Newton step (newton), the multigrid preconditioner (vcycle), whole linear solves (solve), batched
element applications (efs), the geometry of a rule (physical), gathers and scatters (transfer) and the batched
mixed-order operator (batch).  Sizes are those of the benchmark's workloads (64^3 elements at degree 6, 48^3 at degree
5, 32^3 at degree 6, the 32^3 mixed-order batch with its small Poisson problems), of the tests' small meshes, and odd
boxes between them.

exact() recomputes every output in 64 bits with plain torch, from the same inputs and without the library.
"""
import math

import numpy as np
import torch

DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64 = torch.float64
FORCED = dict(exact=0, a=1.0, b=1.0, c=1.0)  # manufactured solution cos(a x) exp(b y) sin(c z)
CHUNK_POINTS = 4_000_000                     # quadrature points per chunk of the 64-bit evaluation


def listed():
    nl = dict(p=1.5, eps2=0.005, lam=0.0)
    return [
        # the smallest call: a test-sized mesh, where launches and the check's wait are everything
        dict(name="jv_f64_4c_p3", op="jv", m0=4, m1=4, m2=4, degree=3, fp32=False, **nl),
        # the benchmark's headline: Jacobian action inside a Krylov loop of a large nonlinear problem
        dict(name="jv_f64_64c_p6", op="jv", m0=64, m1=64, m2=64, degree=6, fp32=False, **nl),
        # single precision inner iterations, high order, a box with no round size, with the Bratu term
        dict(name="jv_f32_odd_p8", op="jv", m0=23, m1=19, m2=29, degree=8, fp32=True, p=1.5, eps2=0.005, lam=0.5),
        # linear diffusion with a variable coefficient at low order (many small elements)
        dict(name="linear_f64_odd_p3", op="linear", m0=61, m1=53, m2=67, degree=3, fp32=False),
        # the residual of a Newton line search with a manufactured forcing
        dict(name="residual_32c_p6", op="residual", m0=32, m1=32, m2=32, degree=6, forced=True, **nl),
        # a Newton step up to its first Krylov vector: residual, Q1 matrix, hierarchy, V-cycle, Jacobian action
        dict(name="newton_32c_p6", op="newton", m0=32, m1=32, m2=32, degree=6, corrected=True, forced=True, **nl),
        # the preconditioner of the mixed-precision solve, once per iteration
        dict(name="vcycle_f32_48c_p5", op="vcycle", m0=48, m1=48, m2=48, degree=5, fp32=True, corrected=False,
             smooth=2),
        # a whole variable-coefficient solve to 1e-10: FP64 CG with the preconditioner in FP32
        dict(name="solve_32c_p5", op="solve", m0=32, m1=32, m2=32, degree=5, mixed=2, corrected=True),
        # element routines alone: gradients at the quadrature points of many elements of one order
        dict(name="efs_grad_p6", op="efs", P=7, Q=7, D=1, nelem=8192, mode="grad", noalloc=False),
        # their transpose for a three-component field, more points than nodes, a call that may not allocate
        dict(name="efs_gradt_p3_d3", op="efs", P=4, Q=5, D=3, nelem=1500, mode="grad_t", noalloc=True),
        # many small problems of different order in one launch
        dict(name="batch_f32_16c_64", op="batch", mesh=16, problems=64, fp32=True),
        # a program with its own element loop: expanded vectors gathered and scattered
        dict(name="transfer_32c_p4", op="transfer", m0=32, m1=32, m2=32, degree=4),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _box(rng, nodes, degree):
    """A box of about `nodes` lattice nodes at a degree, its sides within a factor of two of each other."""
    side = max(2.0, nodes ** (1 / 3) / degree)
    return {f"m{d}": max(2, round(side * _log(rng, 0.71, 1.4))) for d in range(3)}


def draw(rng):
    op = rng.choice(["jv", "jv", "linear", "residual", "newton", "vcycle", "solve", "efs", "efs", "physical", "batch",
                     "transfer"])
    deg = rng.randint(2, 10)
    if op in ("jv", "linear"):
        c = dict(op=op, degree=deg, fp32=rng.random() < 0.4, **_box(rng, _log(rng, 2e3, 2e7), deg))
        return c if op == "linear" else {**c, "p": rng.choice([1.5, 1.5, 1.6, 1.75]), "eps2": 0.005,
                                         "lam": rng.choice([0.0, 0.0, 0.5])}
    if op == "residual":
        return dict(op=op, degree=deg, forced=rng.random() < 0.5, p=1.5, eps2=0.005, lam=rng.choice([0.0, 0.5]),
                    **_box(rng, _log(rng, 2e3, 1e7), deg))
    if op == "newton":
        return dict(op=op, degree=deg, corrected=rng.random() < 0.6, forced=False, p=1.5, eps2=0.005, lam=0.0,
                    **_box(rng, _log(rng, 1e4, 5e6), deg))
    if op == "vcycle":
        return dict(op=op, degree=deg, fp32=rng.random() < 0.6, corrected=rng.random() < 0.5, smooth=rng.choice([1, 2]),
                    **_box(rng, _log(rng, 1e4, 1e7), deg))
    if op == "solve":
        deg = rng.randint(2, 6)
        corrected = rng.random() < 0.6
        return dict(op=op, degree=deg, mixed=rng.choice([0, 1, 2]), corrected=corrected,
                    **_box(rng, _log(rng, 1e4, 2e6), deg))
    if op == "efs":
        P = rng.randint(2, 9)
        Q = P + rng.choice([0, 0, 0, 1, 2])
        D = rng.choice([1, 1, 2, 3])
        points = _log(rng, 2e3, 3e6)
        return dict(op=op, P=P, Q=Q, D=D, nelem=max(1, round(points / (Q ** 3 * D))),
                    mode=rng.choice(["interp", "interp_t", "grad", "grad_t"]), noalloc=rng.random() < 0.5)
    if op == "physical":
        Q = rng.randint(2, 9)
        return dict(op=op, Q=Q, nelem=max(1, round(_log(rng, 2e3, 3e6) / Q ** 3)))
    if op == "batch":
        return dict(op=op, mesh=rng.randint(2, 16), problems=rng.randint(1, 48), fp32=rng.random() < 0.6)
    return dict(op=op, degree=deg, **_box(rng, _log(rng, 2e3, 5e6), deg))


# ------------------------------------------------------------------------------------------------ inputs
def _gen(seed, device=DEV):
    return torch.Generator(device=device).manual_seed(int(seed))


def _uniform(seed, shape, lo=-1.0, hi=1.0, dtype=F64):
    return torch.empty(shape, dtype=dtype, device=DEV).uniform_(lo, hi, generator=_gen(seed))


def _vertices(M, seed):
    """Vertices [(M0+1)(M1+1)(M2+1)][3] of a block on the unit cube, interior ones moved by up to a tenth of h."""
    ax = [torch.linspace(0, 1, m + 1, dtype=F64) for m in M]
    X = torch.stack(torch.meshgrid(*ax, indexing="ij"), dim=-1)
    h = torch.tensor([1.0 / m for m in M], dtype=F64)
    X[1:-1, 1:-1, 1:-1] += (torch.rand((M[0] - 1, M[1] - 1, M[2] - 1, 3), dtype=F64, generator=_gen(seed, "cpu")) - 0.5) * 0.2 * h
    return X


def _coefficient(X, seed):
    """Log-normal coefficient at the vertices: unit variance, correlation length 0.1, by random Fourier features."""
    g = _gen(seed, "cpu")
    w = (torch.randn((256, 3), dtype=F64, generator=g) / 0.1).to(DEV)
    phi = (2 * math.pi * torch.rand(256, dtype=F64, generator=g)).to(DEV)
    f = torch.cos(X.reshape(-1, 3).to(DEV) @ w.T + phi).sum(dim=1) * math.sqrt(2 / 256)
    return torch.exp(f).cpu()


def _gll(n):
    """Gauss-Lobatto-Legendre nodes."""
    if n == 2:
        return np.array([-1.0, 1.0])
    P = np.polynomial.legendre.Legendre.basis(n - 1)
    d1, d2 = P.deriv(), P.deriv(2)
    z = np.sort(np.real(d1.roots()))
    for _ in range(3):
        z = z - d1(z) / d2(z)
    z = 0.5 * (z - z[::-1])
    return np.concatenate([[-1.0], z, [1.0]])


def _lattice_axes(M, p):
    z = (_gll(p + 1) + 1) / 2
    return [np.append(np.concatenate([(e + z[:-1]) / m for e in range(m)]), 1.0) for m in M]


def _state(M, p, seed):
    """Smooth state on the node lattice: eight random-phase sine modes of amplitude 0.1 (wave numbers 1 to 4)."""
    rng = np.random.RandomState(int(seed) % (1 << 31))
    ax = [torch.from_numpy(a).to(DEV) for a in _lattice_axes(M, p)]
    u = torch.zeros([len(a) for a in ax], dtype=F64, device=DEV)
    for _ in range(8):
        k, phi = rng.randint(1, 5, 3), rng.uniform(0, 2 * math.pi)
        s = [torch.sin(2 * math.pi * kd * a) for kd, a in zip(k, ax)]
        c = [torch.cos(2 * math.pi * kd * a) for kd, a in zip(k, ax)]
        xy_s = s[0][:, None] * c[1] + c[0][:, None] * s[1]  # sin(x + y), cos(x + y)
        xy_c = c[0][:, None] * c[1] - s[0][:, None] * s[1]
        z_s, z_c = s[2] * math.cos(phi) + c[2] * math.sin(phi), c[2] * math.cos(phi) - s[2] * math.sin(phi)
        u.addcmul_(xy_s[:, :, None], z_c, value=0.1).addcmul_(xy_c[:, :, None], z_s, value=0.1)
    return u


def _mesh_of(case):
    return (case["m0"], case["m1"], case["m2"])


def _owned_shape(M, p):
    return tuple(m * p - 1 for m in M)


def _inner(u):
    return u[1:-1, 1:-1, 1:-1]


def _mesh_inputs(case, seed):
    """Vertices, coefficient, state and direction of a block-space case."""
    M, p, op = _mesh_of(case), case["degree"], case["op"]
    X = _vertices(M, seed)
    linear = op in ("linear", "vcycle", "solve")
    k = _coefficient(X, seed + 1) if linear else None
    u = None if linear or op == "transfer" else _state(M, p, seed + 2)
    x = _uniform(seed + 3, _owned_shape(M, p))
    return X, k, u, x


def _spaces(case, X, k, u):
    import dohp_amd.capi as C
    fs = C.FS(_mesh_of(case), case["degree"], X.reshape(-1, 3).numpy())
    if u is not None:
        edge = torch.ones(u.shape, dtype=torch.bool, device=DEV)
        _inner(edge).fill_(False)
        fs.dirichlet_commit(u[edge].cpu().numpy())
    prm = dict(FORCED) if case.get("forced") else {}
    return fs, C.Ellip(fs, p=case.get("p", 2.0), eps=math.sqrt(case.get("eps2", 1.0)), lam=case.get("lam", 0.0),
                       kvert=None if k is None else k.numpy(), **prm)


def _degrees(case):
    """Element degrees of the mixed-order mesh and (elements per side, degree) of its small problems."""
    rng = np.random.RandomState(7)  # the layout is the plan's: the same for every seed
    deg = rng.randint(2, 11, case["mesh"] ** 3).astype(np.int32)
    return deg, [(int(rng.randint(4, 17)), int(rng.randint(2, 9))) for _ in range(case["problems"])]


def _element_corners(X):
    return torch.stack([X[a:X.shape[0] - 1 + a, b:X.shape[1] - 1 + b, c:X.shape[2] - 1 + c]
                        for a in (0, 1) for b in (0, 1) for c in (0, 1)], dim=3).reshape(-1, 8, 3)


def _batch_meshes(case, seed):
    deg, probs = _degrees(case)
    return deg, _element_corners(_vertices((case["mesh"],) * 3, seed)), \
        [(m, d, _vertices((m,) * 3, seed + 10 + i)) for i, (m, d) in enumerate(probs)]


def _efs_inputs(case, seed):
    P, Q, D, E, mode = case["P"], case["Q"], case["D"], case["nelem"], case["mode"]
    shape = {"interp": (E, P, P, P, D), "grad": (E, P, P, P, D), "interp_t": (E, Q, Q, Q, D),
             "grad_t": (E, Q, Q, Q, D, 3)}[mode]
    out = {"interp": (E, Q, Q, Q, D), "grad": (E, Q, Q, Q, D, 3), "interp_t": (E, P, P, P, D),
           "grad_t": (E, P, P, P, D)}[mode]
    jinv = None
    if mode.startswith("grad"):
        jinv = _uniform(seed + 1, (E, Q, Q, Q, 3, 3), -0.2, 0.2) + 2 * torch.eye(3, dtype=F64, device=DEV)
    return _uniform(seed, shape), jinv, out


def _jacobians(case, seed):
    Q = case["Q"]
    return _uniform(seed, (case["nelem"], Q, Q, Q, 3, 3), -0.05, 0.05) + 0.3 * torch.eye(3, dtype=F64, device=DEV)


def prepare(case, seed):
    import dohp_amd.capi as C
    op = case["op"]
    s = dict(case=case)
    if op == "efs":
        x, jinv, out = _efs_inputs(case, seed)
        rc = np.polynomial.legendre.leggauss(case["Q"])[0]
        mode = {"interp": C.APPLY_INTERP, "interp_t": C.APPLY_INTERP_TRANSPOSE, "grad": C.APPLY_GRAD,
                "grad_t": C.APPLY_GRAD_TRANSPOSE}[case["mode"]]
        return dict(s, x=x, jinv=jinv, y=torch.zeros(out, dtype=F64, device=DEV), rc=rc, mode=mode,
                    apply=C.efs_apply_hex_batched_noalloc if case["noalloc"] else C.efs_apply_hex_batched)
    if op == "physical":
        jac = _jacobians(case, seed)
        return dict(s, jac=jac, w=np.polynomial.legendre.leggauss(case["Q"])[1], jinv=torch.zeros_like(jac),
                    jw=torch.zeros(jac.shape[:4], dtype=F64, device=DEV), apply=C.rule_compute_physical_batched)
    if op == "batch":
        deg, ev, probs = _batch_meshes(case, seed)
        b = C.Batch()
        for m, d, X in probs:
            b.add_space(C.FS((m, m, m), d, X.reshape(-1, 3).numpy()))
        b.add_elements(deg, ev.numpy())
        x = _uniform(seed + 3, (b.size,), dtype=torch.float32 if case["fp32"] else F64)
        s.update(b=b, x=x, y=torch.zeros_like(x))
        run(s)  # the tiles are timed by the first application
        return s
    X, k, u, x = _mesh_inputs(case, seed)
    fs, A = _spaces(case, X, k, u)
    s.update(fs=fs, A=A, x=x.reshape(-1))
    if op == "transfer":
        s.update(e=torch.zeros(fs.nexpanded, dtype=F64, device=DEV), g=torch.zeros_like(s["x"]))
        return s
    if u is not None:
        s.update(u=_inner(u).reshape(-1), f=torch.zeros_like(s["x"]))
        A.function(s["u"], s["f"])
    if op in ("jv", "linear"):
        if case["fp32"]:
            s["x"] = s["x"].float()
        s["y"] = torch.zeros_like(s["x"])
        run(s)  # the launch shapes are timed and the linearization is formed by the first application
    elif op == "vcycle":
        A.set_q1_mode(int(case["corrected"]))
        s["q1"] = A.assemble_q1()
        s["mg"] = C.MG(s["q1"], smooth_degree=case["smooth"])
        if case["fp32"]:
            s["x"] = s["x"].float()
        s["z"] = torch.zeros_like(s["x"])
    elif op == "newton":
        A.set_q1_mode(int(case["corrected"]))
        s["q1"] = A.assemble_q1(s["u"])
        s["mg"] = C.MG(s["q1"])
        s.update(z=torch.zeros_like(s["x"]), y=torch.zeros_like(s["x"]))
        A.mat_mult(s["f"], s["y"])
    elif op == "solve":
        A.set_q1_mode(int(case["corrected"]))
        s["q1"] = A.assemble_q1()
        s["b"] = torch.zeros_like(s["x"])
        A.mat_mult(s["x"], s["b"])
        s["z"] = torch.zeros_like(s["x"])
    return s


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "jv" or op == "linear":
        (s["A"].mat_mult_f32 if case["fp32"] else s["A"].mat_mult)(s["x"], s["y"])
        return s["y"]
    if op == "residual":
        s["A"].function(s["u"], s["f"])
        return s["f"]
    if op == "newton":
        s["A"].function(s["u"], s["f"])
        s["A"].assemble_q1(s["u"], mat=s["q1"])
        s["mg"].refresh(s["q1"])
        s["mg"].apply(s["f"], s["z"])
        s["A"].mat_mult(s["z"], s["y"])
        return dict(f=s["f"], z=s["z"], y=s["y"])
    if op == "vcycle":
        (s["mg"].apply_f32 if case["fp32"] else s["mg"].apply)(s["x"], s["z"])
        return s["z"]
    if op == "solve":
        s["z"].zero_()
        s["A"].solve(s["q1"], s["b"], s["z"], mixed=case["mixed"], rtol=1e-10)
        return s["z"]
    if op == "efs":
        s["apply"](case["P"], s["rc"], case["nelem"], s["jinv"], case["D"], s["x"], s["y"], s["mode"])
        return s["y"]
    if op == "physical":
        s["apply"](s["w"], case["nelem"], s["jac"], s["jinv"], s["jw"])
        return dict(jinv=s["jinv"], jw=s["jw"])
    if op == "batch":
        (s["b"].mult_f32 if case["fp32"] else s["b"].mult)(s["x"], s["y"])
        return s["y"]
    s["fs"].global_to_expanded(s["x"], s["e"])
    s["fs"].expanded_to_global(s["e"], s["g"])
    return dict(e=s["e"], g=s["g"])


# -------------------------------------------------------------------------------------------------- work
def _gradient_flops(P, Q):
    return 3 * 2 * (Q * P ** 3 + Q ** 2 * P ** 2 + Q ** 3 * P)


def _apply_flops(n, kind):
    """One element's apply: gradient and its transpose (and the state's), geometry and pointwise step."""
    return (3 if kind == "residual" else 2) * _gradient_flops(n, n) + 150 * n ** 3


def work(case):
    op = case["op"]
    if op == "efs":
        P3, Q3, D, E = case["P"] ** 3, case["Q"] ** 3, case["D"], case["nelem"]
        grad = case["mode"].startswith("grad")
        return dict(bytes=8.0 * E * (P3 * D + Q3 * (3 * D + 9 if grad else D)),
                    flops=float(E * D * (_gradient_flops(case["P"], case["Q"]) + 18 * Q3 if grad else
                                         _gradient_flops(case["P"], case["Q"]) / 3)))
    if op == "physical":
        n = case["nelem"] * case["Q"] ** 3
        return dict(bytes=8.0 * 19 * n, flops=50.0 * n)
    if op == "batch":
        deg, probs = _degrees(case)
        s = 4 if case["fp32"] else 8
        by = sum(2 * s * (d + 1) ** 3 + 192 for d in deg.tolist())
        fl = sum(_apply_flops(d + 1, "linear") for d in deg.tolist())
        for m, d in probs:
            by += 2 * s * (m * d - 1) ** 3 + 24 * (m + 1) ** 3
            fl += m ** 3 * _apply_flops(d + 1, "linear")
        return dict(bytes=float(by), flops=float(fl))
    M, p = _mesh_of(case), case["degree"]
    n, E = math.prod(m * p - 1 for m in M), math.prod(M)
    lat, vert = math.prod(m * p + 1 for m in M), 24 * math.prod(m + 1 for m in M)
    s = 4 if case.get("fp32") else 8
    one = _apply_flops(p + 1, "linear") * E
    if op == "jv":  # x, the state and the vertices read, y written
        return dict(bytes=float(2 * s * n + s * lat + vert), flops=float(one))
    if op == "linear":
        return dict(bytes=float(2 * s * n + vert * 4 / 3), flops=float(one))
    if op == "residual":
        return dict(bytes=float(8 * (n + lat) + 8 * n * case["forced"] + vert), flops=float(1.5 * one))
    if op == "transfer":
        return dict(bytes=8.0 * (2 * n + 2 * E * (p + 1) ** 3), flops=float(E * (p + 1) ** 3))
    # a V-cycle: the symmetric stencil (14 values a node) once, the vectors, 27-point products on levels of 1/8 each
    deg = case.get("smooth", 2)
    vc = dict(bytes=(16 * s + 0.0) * n * 8 / 7, flops=54.0 * 2 * deg * n * 8 / 7)
    if op == "vcycle":
        return vc
    if op == "newton":
        cells = math.prod(m * p for m in M)
        return dict(bytes=vc["bytes"] + 8.0 * (n * 14 + 5 * n + 2 * lat) + vert,
                    flops=vc["flops"] + 2.5 * one + cells * 8 * 400.0)
    its = 30  # a solve: at least some thirty applications of the operator and the preconditioner
    return dict(bytes=its * (4.0 * 16 * n + 8.0 * 6 * n), flops=its * (54.0 * 2 * n * 8 / 7 + one))


# ------------------------------------------------------------------------------- the same in plain 64 bits
def _lagrange(z, x):
    """Values and derivatives at x of the Lagrange basis through z: two [len(x)][len(z)] matrices."""
    n = len(z)
    B, Dm = np.ones((len(x), n)), np.zeros((len(x), n))
    for j in range(n):
        for m in range(n):
            if m == j:
                continue
            B[:, j] *= (x - z[m]) / (z[j] - z[m])
            t = np.full(len(x), 1 / (z[j] - z[m]))
            for q in range(n):
                if q != j and q != m:
                    t *= (x - z[q]) / (z[j] - z[q])
            Dm[:, j] += t
    return torch.from_numpy(B).to(DEV), torch.from_numpy(Dm).to(DEV)


def _along(A, x, d):
    return torch.movedim(torch.tensordot(A, x, dims=([1], [d])), 0, d)


def _tensor(A0, A1, A2, x):
    return _along(A2, _along(A1, _along(A0, x, 1), 2), 3)


def _grad(B, D, x):
    return torch.stack([_tensor(D, B, B, x), _tensor(B, D, B, x), _tensor(B, B, D, x)], dim=-1)


def _grad_t(B, D, f):
    Bt, Dt = B.T.contiguous(), D.T.contiguous()
    return _tensor(Dt, Bt, Bt, f[..., 0]) + _tensor(Bt, Dt, Bt, f[..., 1]) + _tensor(Bt, Bt, Dt, f[..., 2])


def _corner_values(V, z):
    """Trilinear interpolation of corner data V [E][8][c] at the tensor points of z: values and reference gradient."""
    B, D = _lagrange(np.array([-1.0, 1.0]), z)
    v = V.reshape(len(V), 2, 2, 2, -1)
    return _tensor(B, B, B, v), torch.stack([_tensor(D, B, B, v), _tensor(B, D, B, v), _tensor(B, B, D, v)], dim=-1)


def _inverse(J):
    """Inverse and determinant of J [..., x, ref]."""
    c = torch.stack([torch.linalg.cross(J[..., 1], J[..., 2]), torch.linalg.cross(J[..., 2], J[..., 0]),
                     torch.linalg.cross(J[..., 0], J[..., 1])], dim=-2)
    det = (c[..., 0, :] * J[..., 0]).sum(-1)
    return c / det[..., None, None], det


def _forcing(case, X):
    """-div(eta grad u) of the manufactured solution at the points X."""
    a, b, c = FORCED["a"], FORCED["b"], FORCED["c"]
    cx, sx, ey = torch.cos(a * X[..., 0]), torch.sin(a * X[..., 0]), torch.exp(b * X[..., 1])
    cz, sz = torch.cos(c * X[..., 2]), torch.sin(c * X[..., 2])
    du = torch.stack([-a * sx * ey * sz, b * cx * ey * sz, c * cx * ey * cz], dim=-1)
    xy, xz, yz = -a * b * sx * ey * sz, -a * c * sx * ey * cz, b * c * cx * ey * cz
    diag = [-a * a * cx * ey * sz, b * b * cx * ey * sz, -c * c * cx * ey * sz]
    H = torch.stack([torch.stack([diag[0], xy, xz], -1), torch.stack([xy, diag[1], yz], -1),
                     torch.stack([xz, yz, diag[2]], -1)], -2)
    g = case["eps2"] + 0.5 * (du * du).sum(-1)
    quad = (du * (H * du[..., None, :]).sum(-1)).sum(-1)
    return -g ** ((case["p"] - 2) / 2) * sum(diag) - (case["p"] - 2) / 2 * g ** ((case["p"] - 4) / 2) * quad


def _element_apply(n, V, k, ue, xe, case):
    """Contributions [E][n][n][n] of elements: the residual at ue (xe None) or the Jacobian action on xe."""
    z, w = np.polynomial.legendre.leggauss(n)
    B, D = _lagrange(_gll(n), z)
    pos, J = _corner_values(V, z)
    Ji, det = _inverse(J)
    w = torch.from_numpy(w).to(DEV)
    jw = det * w[:, None, None] * w[:, None] * w
    kq = 1.0 if k is None else _corner_values(k[..., None], z)[0][..., 0]
    p, lam = case.get("p", 2.0), case.get("lam", 0.0)
    phys = lambda e: (_grad(B, D, e)[..., None] * Ji).sum(-2)  # noqa: E731
    eta, v = 1.0, None
    if ue is not None:
        gu = phys(ue)
        gam = case["eps2"] + 0.5 * (gu * gu).sum(-1)
        eta = gam ** ((p - 2) / 2)
        if lam:
            v = -jw * lam * torch.exp(_tensor(B, B, B, ue))
    if xe is None:
        F = (jw * eta * kq)[..., None] * gu
        if case.get("forced"):
            v = -jw * _forcing(case, pos) + (0 if v is None else v)
    else:
        gx = phys(xe)
        F = (jw * eta * kq)[..., None] * gx if ue is not None or k is not None else jw[..., None] * gx
        if ue is not None:
            F = F + (jw * kq * (p - 2) / 2 * eta / gam * (gu * gx).sum(-1))[..., None] * gu
            if v is not None:
                v = v * _tensor(B, B, B, xe)
    y = _grad_t(B, D, (Ji * F[..., None, :]).sum(-1))
    return y if v is None else y + _tensor(B.T.contiguous(), B.T.contiguous(), B.T.contiguous(), v)


def _slabs(M, n):
    """Runs of element layers along the first direction holding about CHUNK_POINTS points each."""
    step = max(1, CHUNK_POINTS // (M[1] * M[2] * n ** 3))
    return [(a, min(M[0], a + step)) for a in range(0, M[0], step)]


def _gather(lat, a0, a1, M, p):
    """Element nodes [E][n][n][n] of the element layers a0..a1 of a lattice array."""
    n = p + 1
    v = lat[a0 * p:a1 * p + 1].unfold(0, n, p).unfold(1, n, p).unfold(2, n, p)
    return v.reshape(-1, n, n, n)


def _scatter_add(lat, y, a0, a1, M, p):
    n = p + 1
    y = y.reshape(a1 - a0, M[1], M[2], n, n, n)
    for a in range(n):
        for b in range(n):
            for c in range(n):
                lat[a0 * p + a:(a1 - 1) * p + a + 1:p, b:(M[1] - 1) * p + b + 1:p,
                    c:(M[2] - 1) * p + c + 1:p] += y[..., a, b, c]


def _exact_apply(case, X, k, u, x):
    """Residual (x None) or operator application on the owned nodes of a block space; x zero on the boundary."""
    M, p = _mesh_of(case), case["degree"]
    out = torch.zeros([m * p + 1 for m in M], dtype=F64, device=DEV)
    xl = None
    if x is not None:
        xl = torch.zeros_like(out)
        _inner(xl).copy_(x.reshape(_owned_shape(M, p)))
    V = X.to(DEV)
    kk = None if k is None else k.reshape(V.shape[:3]).to(DEV)
    for a0, a1 in _slabs(M, p + 1):
        ev = _element_corners(V[a0:a1 + 1])
        ke = None if kk is None else _element_corners(kk[a0:a1 + 1, ..., None].expand(-1, -1, -1, 3))[..., 0]
        y = _element_apply(p + 1, ev, ke, None if u is None else _gather(u, a0, a1, M, p),
                           None if xl is None else _gather(xl, a0, a1, M, p), case)
        _scatter_add(out, y, a0, a1, M, p)
    return _inner(out).reshape(-1)


def _q1_stencil(case, X, k, u):
    """27-point stencil [3][3][3][box] of the embedded-Q1 matrix over the owned nodes."""
    M, p = _mesh_of(case), case["degree"]
    n, gll = p + 1, _gll(p + 1)
    h = np.diff(gll)
    s = np.array([-1.0, 1.0]) / math.sqrt(3.0)
    z = (0.5 * (gll[:-1] + gll[1:])[:, None] + 0.5 * h[:, None] * s).reshape(-1)
    w = torch.from_numpy(np.repeat(h / 2, 2)).to(DEV)
    B, D = _lagrange(gll, z)
    hat = torch.tensor([[(1 - t) / 2, (1 + t) / 2] for t in s], dtype=F64, device=DEV)  # [point][node]
    st = torch.zeros([3, 3, 3] + [m * p + 1 for m in M], dtype=F64, device=DEV)
    V = X.to(DEV)
    kk = None if k is None else k.reshape(V.shape[:3]).to(DEV)
    pp, lam = case.get("p", 2.0), case.get("lam", 0.0)
    corr = case["corrected"]

    def cells(f):  # element-ordered points [E][2p][2p][2p] -> [E][p][p][p][8]
        f = f.reshape(len(f), p, 2, p, 2, p, 2, *f.shape[4:])
        return f.permute(0, 1, 3, 5, 2, 4, 6, *range(7, f.dim())).reshape(len(f), p, p, p, 8, *f.shape[7:])

    scale = torch.from_numpy(1 / h if corr else np.ones(p)).to(DEV)
    for a0, a1 in _slabs(M, 4 * p):
        ev = _element_corners(V[a0:a1 + 1])
        Ji, det = _inverse(_corner_values(ev, z)[1])
        W = det * w[:, None, None] * w[:, None] * w
        kq = None
        if kk is not None:
            ke = _element_corners(kk[a0:a1 + 1, ..., None].expand(-1, -1, -1, 3))[..., 0]
            kq = _corner_values(ke[..., None], z)[0][..., 0]
        eta, r1, Du, lex = W if kq is None else W * kq, None, None, None
        if u is not None:
            ue = _gather(u, a0, a1, M, p)
            Du = (_grad(B, D, ue)[..., None] * Ji).sum(-2)
            g = case["eps2"] + 0.5 * (Du * Du).sum(-1)
            r1 = cells(eta * (pp - 2) / 2 * g ** ((pp - 4) / 2))
            eta = eta * g ** ((pp - 2) / 2)
            Du = cells(Du)
            if lam:
                lex = cells(-W * lam * torch.exp(_tensor(B, B, B, ue)))
        eta = cells(eta)
        # the reference's arithmetic reads the inverse Jacobians in element order, the corrected one at each point
        Jc = cells(Ji) if corr else Ji.reshape(len(Ji), p, p, p, 8, 3, 3)
        for q in range(8):
            f = [hat[(q >> 2) & 1], hat[(q >> 1) & 1], hat[q & 1]]
            Dq, Iq = [], []
            for r in range(8):
                a, b, c = r >> 2, (r >> 1) & 1, r & 1
                sg = [1.0 if t else -1.0 for t in (a, b, c)]
                d0 = sg[0] * f[1][b] * f[2][c] * scale[:, None, None, None]
                d1 = sg[1] * f[0][a] * f[2][c] * scale[:, None, None]
                d2 = sg[2] * f[0][a] * f[1][b] * scale[:, None]
                J = Jc[..., q, :, :]
                Dq.append(d0 * J[..., 0, :] + d1 * J[..., 1, :] + d2 * J[..., 2, :])
                Iq.append(f[0][a] * f[1][b] * f[2][c])
            sd = [None if Du is None else (Du[..., q, :] * t).sum(-1) for t in Dq]
            for r in range(8):
                for c in range(8):
                    K = eta[..., q] * (Dq[r] * Dq[c]).sum(-1)
                    if r1 is not None:
                        K = K + r1[..., q] * sd[r] * sd[c]
                    if lex is not None:
                        K = K + lex[..., q] * Iq[r] * Iq[c]
                    K = K.reshape(a1 - a0, M[1], M[2], p, p, p).permute(0, 3, 1, 4, 2, 5)
                    K = K.reshape((a1 - a0) * p, M[1] * p, M[2] * p)
                    o = [((c >> t) & 1) - ((r >> t) & 1) + 1 for t in (2, 1, 0)]
                    i = [(r >> t) & 1 for t in (2, 1, 0)]
                    st[o[0], o[1], o[2], a0 * p + i[0]:a1 * p + i[0], i[1]:i[1] + M[1] * p,
                       i[2]:i[2] + M[2] * p] += K
    st = st[:, :, :, 1:-1, 1:-1, 1:-1].contiguous()
    for d in range(3):  # entries toward boundary nodes are dropped
        st.select(d, 0).select(2 + d, 0).zero_()
        st.select(d, 2).select(2 + d, -1).zero_()
    return st


def _product(st, x):
    xp = torch.nn.functional.pad(x, (1, 1, 1, 1, 1, 1))
    y = torch.zeros_like(x)
    for i in range(3):
        for j in range(3):
            for k in range(3):
                y.addcmul_(st[i, j, k], xp[i:i + x.shape[0], j:j + x.shape[1], k:k + x.shape[2]])
    return y


def _prolong(v, shape):
    for d in range(3):
        v = torch.movedim(v, d, 0)
        n = shape[d]
        f = torch.zeros((n,) + v.shape[1:], dtype=F64, device=DEV)
        f[1::2] = v[:len(f[1::2])]
        f[0::2] += 0.5 * torch.cat([v, torch.zeros_like(v[:1])])[:len(f[0::2])]
        f[2::2] += 0.5 * v[:len(f[2::2])]
        v = torch.movedim(f, 0, d)
    return v


def _restrict(r, shape):
    for d in range(3):
        r = torch.movedim(r, d, 0)
        n = shape[d]
        r = torch.cat([r, torch.zeros_like(r[:1])])
        r = r[1:2 * n:2] + 0.5 * (r[0:2 * n:2] + r[2:2 * n + 1:2])
        r = torch.movedim(r, 0, d)
    return r


def _galerkin(st, shape):
    """Coarse 27-point stencil of P^T A P, by products with the 27 colours of coarse nodes."""
    out = torch.zeros([3, 3, 3] + list(shape), dtype=F64, device=DEV)
    ix = [torch.arange(s, device=DEV) for s in shape]
    for c0 in range(min(3, shape[0])):
        for c1 in range(min(3, shape[1])):
            for c2 in range(min(3, shape[2])):
                v = torch.zeros(list(shape), dtype=F64, device=DEV)
                v[c0::3, c1::3, c2::3] = 1
                w = _restrict(_product(st, _prolong(v, st.shape[3:])), shape)
                m = [(c - i + 1) % 3 for c, i in zip((c0, c1, c2), ix)]  # offset slot of this colour at each row
                for i in range(3):
                    for j in range(3):
                        for k in range(3):
                            on = ((m[0] == i)[:, None, None] & (m[1] == j)[:, None]) & (m[2] == k)
                            out[i, j, k] += w * on
    for d in range(3):
        out.select(d, 0).select(2 + d, 0).zero_()
        out.select(d, 2).select(2 + d, -1).zero_()
    return out


def _power_start(n):
    with np.errstate(over="ignore"):
        z = np.arange(n, dtype=np.uint64) + np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    return torch.from_numpy((z >> np.uint64(11)).astype(np.float64) / 9007199254740992.0 + 0.25).to(DEV)


def _levels(st):
    L = []
    while True:
        box = tuple(st.shape[3:])
        dinv = 1 / st[1, 1, 1]
        coarse = tuple(b // 2 for b in box)
        if math.prod(box) <= 512 or min(coarse) < 1:
            L.append((st, dinv, None))
            return L
        v = _power_start(math.prod(box)).reshape(box)
        v /= torch.linalg.vector_norm(v)
        for _ in range(15):
            v = dinv * _product(st, v)
            lmax = float(torch.linalg.vector_norm(v))
            v /= lmax
        L.append((st, dinv, lmax))
        st = _galerkin(st, coarse)


def _smooth(lv, degree, b, x):
    st, dinv, lmax = lv
    lo, hi = 0.1 * lmax, 1.1 * lmax
    theta, delta = 0.5 * (hi + lo), 0.5 * (hi - lo)
    sigma = theta / delta
    rho = 1 / sigma
    d = dinv * (b if x is None else b - _product(st, x)) / theta
    x = d if x is None else x + d
    for _ in range(1, degree):
        new = 1 / (2 * sigma - rho)
        d = new * rho * d + 2 * new / delta * dinv * (b - _product(st, x))
        x = x + d
        rho = new
    return x


def _vcycle(L, l, degree, b):
    st = L[l][0]
    if l + 1 == len(L):
        n = b.numel()
        I = torch.eye(n, dtype=F64, device=DEV).reshape(n, *b.shape)
        A = torch.stack([_product(st, e).reshape(-1) for e in I], dim=1)
        return torch.linalg.solve(A.cpu(), b.reshape(-1).cpu()).to(DEV).reshape(b.shape)
    x = _smooth(L[l], degree, b, None)
    e = _vcycle(L, l + 1, degree, _restrict(b - _product(st, x), L[l + 1][0].shape[3:]))
    return _smooth(L[l], degree, b, x + _prolong(e, b.shape))


def exact(case, seed):
    op = case["op"]
    if op == "efs":
        x, jinv, _ = _efs_inputs(case, seed)
        B, D = _lagrange(_gll(case["P"]), np.polynomial.legendre.leggauss(case["Q"])[0])
        if case["mode"] == "interp":
            return _tensor(B, B, B, x)
        if case["mode"] == "interp_t":
            return _tensor(*(B.T.contiguous(),) * 3, x)
        if case["mode"] == "grad":  # sum over reference directions of d x / d X_m times dX_m / dx_e
            return (_grad(B, D, x)[..., None] * jinv[:, :, :, :, None]).sum(-2)
        return _grad_t(B, D, (jinv[:, :, :, :, None] * x[..., None, :]).sum(-1))
    if op == "physical":
        jinv, det = _inverse(_jacobians(case, seed))
        w = torch.from_numpy(np.polynomial.legendre.leggauss(case["Q"])[1]).to(DEV)
        return dict(jinv=jinv, jw=det * w[:, None, None] * w[:, None] * w)
    if op == "batch":
        deg, ev, probs = _batch_meshes(case, seed)
        sizes = [(m * d - 1) ** 3 for m, d, _ in probs]
        dof = [(d + 1) ** 3 for d in deg.tolist()]
        x = _uniform(seed + 3, (sum(sizes) + sum(dof),), dtype=torch.float32 if case["fp32"] else F64).double()
        y, off = torch.zeros_like(x), 0
        for (m, d, X), n in zip(probs, sizes):
            c = dict(m0=m, m1=m, m2=m, degree=d)
            y[off:off + n] = _exact_apply(c, X, None, None, x[off:off + n])
            off += n
        at = off + np.concatenate([[0], np.cumsum(dof)[:-1]])
        for d in range(2, 11):
            e = np.nonzero(deg == d)[0]
            if len(e):
                i = torch.from_numpy(at[e][:, None] + np.arange((d + 1) ** 3)).to(DEV)
                xe = x[i].reshape(-1, d + 1, d + 1, d + 1)
                y[i] = _element_apply(d + 1, ev[torch.from_numpy(e)].to(DEV), None, None, xe, {}).reshape(i.shape)
        return y
    X, k, u, x = _mesh_inputs(case, seed)
    if op == "solve":  # the right-hand side is the operator's at x
        return x.reshape(-1)
    if op == "transfer":
        M, p = _mesh_of(case), case["degree"]
        xl = torch.nn.functional.pad(x, (1, 1, 1, 1, 1, 1))
        e = _gather(xl, 0, M[0], M, p)
        g = torch.zeros_like(xl)
        _scatter_add(g, e, 0, M[0], M, p)
        return dict(e=e.reshape(-1), g=_inner(g).reshape(-1))
    if op == "residual":
        return _exact_apply(case, X, k, u, None)
    if op in ("jv", "linear"):
        return _exact_apply(case, X, k, u, x.float().double() if case["fp32"] else x)
    L = _levels(_q1_stencil(case, X, k, u))
    if op == "vcycle":
        return _vcycle(L, 0, case["smooth"], x.float().double() if case["fp32"] else x).reshape(-1)
    f = _exact_apply(case, X, k, u, None)
    z = _vcycle(L, 0, 2, f.reshape(x.shape)).reshape(-1)
    return dict(f=f, z=z, y=_exact_apply(case, X, k, u, z))
