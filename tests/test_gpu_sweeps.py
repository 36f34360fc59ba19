"""The multigrid's sweeps (products with the half stencil from a staged tile, fused smoothing steps, power iterations of
all levels together) against plain torch in FP64 on the levels' own 27-point stencils: boxes on both sides of the rule
that picks the tile, odd and even sides, every smoothing degree's buffer order, all three coefficient precisions."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

# (elements, degree): owned boxes of 95 x 191 x 131 and 97 x 89 x 127 rows (64 x 8 x 2 tiles on the finest level,
# 64 x 4 x 1 below), and of 13 x 25 x 63 and 19 x 9 x 9 rows (small tiles only)
BOXES = [((24, 48, 33), 4, 7), ((24, 22, 32), 4, 6), ((3, 6, 16), 4, 6), ((4, 2, 2), 5, 7)]


@pytest.fixture(scope="module")
def C():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    import dohp_amd.capi as capi
    return capi


def product(st, x):
    xp = F.pad(x, (1, 1, 1, 1, 1, 1))
    y = torch.zeros_like(x)
    for s in range(27):
        i, j, k = s // 9, s // 3 % 3, s % 3
        y += st[s] * xp[i:i + x.shape[0], j:j + x.shape[1], k:k + x.shape[2]]
    return y


def interp(nf, nc):
    P = torch.zeros(nf, nc, dtype=torch.float64, device="cuda")
    for c in range(nc):
        P[2 * c + 1, c] = 1
        for f in (2 * c, 2 * c + 2):
            if f < nf:
                P[f, c] = 0.5
    return P


def smooth(st, lmax, degree, b, x):
    lo, hi = 0.1 * lmax, 1.1 * lmax
    theta, delta = 0.5 * (hi + lo), 0.5 * (hi - lo)
    rho, d = delta / theta, 0
    for k in range(degree):
        r = b if x is None else b - product(st, x)
        if k == 0:
            d = r / st[13] / theta
        else:
            new = 1 / (2 * theta / delta - rho)
            d = new * rho * d + 2 * new / delta * r / st[13]
            rho = new
        x = d if x is None else x + d
    return x


def vcycle(L, l, degree, b):
    st, lmax = L[l]
    if l + 1 == len(L):
        n = b.numel()
        eye = torch.eye(n, dtype=torch.float64, device="cuda").reshape(n, *b.shape)
        A = torch.stack([product(st, e).reshape(-1) for e in eye], dim=1)
        return torch.as_tensor(np.linalg.solve(A.cpu().numpy(), b.reshape(-1).cpu().numpy()), device="cuda").reshape(b.shape)
    Ps = [interp(f, c) for f, c in zip(b.shape, L[l + 1][0].shape[1:])]
    x = smooth(st, lmax, degree, b, None)
    r = b - product(st, x)
    for d in range(3):
        r = torch.movedim(torch.tensordot(Ps[d].T.contiguous(), r, dims=([1], [d])), 0, d)
    e = vcycle(L, l + 1, degree, r.contiguous())
    for d in range(3):
        e = torch.movedim(torch.tensordot(Ps[d], e, dims=([1], [d])), 0, d)
    return smooth(st, lmax, degree, b, x + e)


def lmax_of(st):
    n = st[0].numel()
    with np.errstate(over="ignore"):
        z = np.arange(n, dtype=np.uint64) + np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    v = torch.as_tensor((z >> np.uint64(11)).astype(np.float64) / 2.0 ** 53 + 0.25, device="cuda").reshape(st[0].shape)
    v = v / torch.linalg.vector_norm(v)
    for _ in range(15):
        v = product(st, v) / st[13]
        nw = float(torch.linalg.vector_norm(v))
        v = v / nw
    return nw


def setup(C, M, p, mask, degree):
    from dohp_amd.mesh import block_vertices, splitmix64_uniform
    V = block_vertices(M, box=(0, 1, 0, 1, 0, 1), perturb=0.1, seed=2)
    op = C.Ellip(C.FS(M, p, V, dirichlet_mask=mask), p=2.0, kvert=0.5 + splitmix64_uniform(4, len(V)))
    op.set_q1_mode(1)
    q1 = op.assemble_q1()
    mg = C.MG(q1, smooth_degree=degree)
    L = []
    for l in range(mg.nlevels):
        box, st = mg.level(l)
        L.append(torch.as_tensor(st, device="cuda").reshape(27, *box))
    return op, q1, mg, [(st, lmax_of(st) if l + 1 < len(L) else None) for l, st in enumerate(L)]


# FP64: about 30 roundings of 1.1e-16 per row and sweep, a dozen sweeps on each of up to five levels: 1e-12 leaves two
# digits.  FP32: the same with 6e-8: 5e-5.  FP16 off-diagonals: each is off by up to 2^-11 of itself while the row sums
# are kept: 5e-4 a sweep, smoothed down by the V-cycle; 2e-3.
@pytest.mark.parametrize("degree", [1, 2, 3])
@pytest.mark.parametrize("M,p,mask", BOXES)
def test_vcycle_matches_plain_fp64(C, M, p, mask, degree):
    print(f"V-cycle M={M} p={p} mask={mask} degree={degree}", flush=True)
    op, q1, mg, L = setup(C, M, p, mask, degree)
    assert abs(mg.lmax - L[0][1]) <= 1e-12 * L[0][1]
    g = torch.Generator(device="cuda").manual_seed(5)
    r = torch.rand(q1.nrows, dtype=torch.float64, device="cuda", generator=g) * 2 - 1
    ref = vcycle(L, 0, degree, r.reshape(L[0][0].shape[1:])).reshape(-1)
    z = torch.full_like(r, float("nan"))
    mg.apply(r, z)
    assert float(torch.linalg.norm(z - ref)) <= 1e-12 * float(torch.linalg.norm(ref))
    r32, z32 = r.float(), torch.full_like(r, float("nan"), dtype=torch.float32)
    ref = vcycle(L, 0, degree, r32.double().reshape(L[0][0].shape[1:])).reshape(-1)
    for fp16, tol in ((False, 5e-5), (True, 2e-3)):
        mg.set_coefficients(fp16)
        for _ in range(4):  # eager, captured, replayed
            z32.fill_(float("nan"))
            mg.apply_f32(r32, z32)
            torch.cuda.synchronize()
            assert float(torch.linalg.norm(z32.double() - ref)) <= tol * float(torch.linalg.norm(ref)), fp16
    assert torch.equal(r32, r.float())


# One level: the V-cycle is the explicit inverse.  Sizes on both sides of the elimination's 32-row blocks and the largest
# default coarsest level; well-conditioned Q1 matrices: 512 roundings of 1.1e-16 times a condition number below 1e3.
@pytest.mark.parametrize("M", [(2, 2, 2), (2, 2, 32), (3, 5, 5), (4, 12, 2), (5, 5, 5), (6, 14, 2), (9, 9, 9)])
def test_direct_coarse_solve(C, M):
    n = (M[0] - 1) * (M[1] - 1) * (M[2] - 1)
    print(f"coarse inverse n={n}", flush=True)
    op, q1, mg, L = setup(C, M, 1, 7, 2)
    assert mg.nlevels == 1 and mg.ncoarse == n == q1.nrows
    A = q1.to_scipy().toarray()
    r = torch.as_tensor(np.sin(1.0 + np.arange(n)), device="cuda")
    ref = np.linalg.solve(A, r.cpu().numpy())
    z, z32 = torch.zeros_like(r), torch.zeros(n, dtype=torch.float32, device="cuda")
    mg.apply(r, z)
    mg.apply_f32(r.float(), z32)
    assert np.linalg.norm(z.cpu().numpy() - ref) <= 1e-11 * np.linalg.norm(ref)
    assert np.linalg.norm(z32.cpu().numpy() - ref) <= 1e-4 * np.linalg.norm(ref)
